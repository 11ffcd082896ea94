"""hi/lo layers whose Q epilogue runs on a copy of Q in front of the attention
kernel (hilo_prepare_q in dr_api.cpp): head dims up to 128 and padded head
dims with bias, QK-norm or RoPE, and a partial rotary at every head dim, in
front of the 16-row and of the 32-row kernel.  Batch slots of different
lengths, one of scattered rows, in rows of a fused projection: the attention
output of every slot against the oracle at scale 1.0 (max-abs 1e-2, mean-abs
1e-3, as the other hi/lo tests).  Needs an MI355X.
"""
from __future__ import annotations

import pytest

from test_gpu_hilo32 import run_slots
from test_gpu_parity import dev, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# (h, hkv, hd, n_total, slots' active positions, window, prefix, rotary dims, epilogue, rows per wave)
CASES = {
    "hd64_bias": (4, 2, 64, 130, [range(100, 130), [3, 64, 99]], None, None, 0, "b", 16),
    "hd128_full_rotary": (8, 2, 128, 300, [range(260, 300), range(0, 300, 7)], 90, None, 128, "nb", 16),
    "hd128_partial_rotary": (4, 4, 128, 97, [[96], range(33, 97)], None, 60, 64, "n", 16),
    "hd96_padded": (6, 2, 96, 200, [range(150, 200), [0, 31, 32, 199]], None, None, 32, "nb", 16),
    "hd192_padded_norm": (4, 2, 192, 150, [range(100, 150), range(7, 9)], 64, None, 192, "n", 16),
    "hd256_partial_short": (4, 2, 256, 100, [range(80, 100), [5, 50]], None, None, 64, "nb", 16),
    "hd256_partial_long": (8, 8, 256, 1200, [range(1071, 1200), range(0, 1200, 100)], None, None, 64, "n", 32),
    "hd512_partial_short": (4, 1, 512, 90, [range(60, 90), [89]], None, 75, 128, "n", 16),
    "hd512_partial_long": (4, 2, 512, 4200, [range(4160, 4200), [1, 4199]], None, None, 256, "nb", 32),
}


@pytest.mark.parametrize("name", list(CASES))
def test_hilo_q_copy_vs_oracle(dev, name):
    h, hkv, hd, n_t, slots, window, prefix, rot, epi, rows = CASES[name]
    info = run_slots(dev, h, hkv, hd, n_t, [list(a) for a in slots], window, prefix, rot, epi, sum(map(ord, name)))
    assert info["rows_per_wave"] == rows
