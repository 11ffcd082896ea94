"""dr_qmatmul at the sizes where its two families of kernels can go wrong: the
slice kernels (an eighth of the blocks per wave) with fewer blocks than waves,
one block, ragged weight rows, 32 / 33 / 64 / 65 / 129 activation rows and
weights at addresses of either 2-byte parity, and the kernels that walk all
blocks, at the first size past the slices' limit of 256 workgroups -- against
the oracle with the bound of the other dr_qmatmul tests (exact integers, f32
combine: helpers.kquant_bound, legacy_bound).  Needs an MI355X.
"""
from __future__ import annotations

import numpy as np
import pytest

import dr_attn as dr
import oracle as orc
from helpers import kquant_acts, kquant_bound, kquant_weights, legacy_bound, legacy_weights

from test_gpu_parity import dev, say, torch  # noqa: F401
from test_gpu_qmatmul import _check

pytestmark = pytest.mark.gpu

TYPES = [orc.WTYPE_Q4K, orc.WTYPE_Q6K, orc.WTYPE_Q4_0, orc.WTYPE_Q5_0, orc.WTYPE_Q8_0]


@pytest.mark.parametrize("wtype", TYPES)
@pytest.mark.parametrize("rows,blocks,n,skew", [
    (1, 1, 1, 0), (31, 3, 32, 2), (33, 8, 33, 0), (65, 9, 64, 2), (40, 17, 65, 0), (70, 40, 129, 2),
    (32 * 256 + 1, 2, 64, 0),  # 257 workgroups: the walking kernels
    (32 * 64 + 1, 5, 257, 0),
])
def test_qmatmul_slices_vs_oracle(dev, wtype, rows, blocks, n, skew):
    legacy = wtype in orc.LEGACY_BYTES
    rng = np.random.default_rng(rows + 31 * blocks + 7 * n + wtype)
    cols = blocks * (32 if legacy else 256)
    w = (legacy_weights if legacy else kquant_weights)(rng, wtype, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32) if legacy else kquant_acts(rng, n, cols)
    res = rng.standard_normal((n, rows)).astype(np.float32)
    want = orc.qmatmul(wtype, w, rows, cols, x, n, res).reshape(n, rows)
    tol = (legacy_bound if legacy else kquant_bound)(orc, wtype, w, rows, cols, x, n, res)
    skew = 0 if wtype == orc.WTYPE_Q4K else skew  # (Q4_K blocks start 16-byte aligned)
    buf = dev.put(np.concatenate([np.zeros(skew, np.uint8), w.view(np.uint8).reshape(-1)]))
    out = dev.put(res.reshape(-1))
    dr.qmatmul(dev.ctx, wtype, buf.data_ptr() + skew, rows, cols, dev.put(x), n, out, out)
    _check(dev.get(out).reshape(n, rows), want, tol, f"wtype {wtype} {rows} x {cols}, {n} rows, skew {skew}")


def test_q6k_rows_past_32_bit_offsets(dev):
    """Q6_K over 2^26 columns and 33 activation rows: two tiles of Q8_K
    activations are 2^32 bytes, past the slices' 32-bit offsets.  All but a few
    blocks of the activations are zero and add nothing, so the oracle runs on
    those blocks alone."""
    t, rows, n, nb = dev.t, 2, 33, 1 << 18
    at = [0, 1, 4095, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, nb - 2, nb - 1]
    rng = np.random.default_rng(26)
    cols = 256 * len(at)
    w, x = kquant_weights(rng, orc.WTYPE_Q6K, rows, cols), kquant_acts(rng, n, cols)
    res = rng.standard_normal((n, rows)).astype(np.float32)
    want = orc.qmatmul(orc.WTYPE_Q6K, w, rows, cols, x, n, res).reshape(n, rows)
    tol = kquant_bound(orc, orc.WTYPE_Q6K, w, rows, cols, x, n, res)
    ctx = dr.Context(0)  # (its workspace of 10 GB goes with it)
    ctx.set_stream(dev.stream.cuda_stream)
    with t.cuda.stream(dev.stream):
        wd = t.zeros((rows, nb, 210), dtype=t.uint8, device="cuda")
        xd = t.zeros((n, nb, 256), dtype=t.float32, device="cuda")
        wd[:, at] = t.from_numpy(w.reshape(rows, len(at), 210)).cuda()
        xd[:, at] = t.from_numpy(x.reshape(n, len(at), 256)).cuda()
    out = dev.put(res.reshape(-1))
    dr.qmatmul(ctx, orc.WTYPE_Q6K, wd, rows, nb * 256, xd, n, out, out)
    got = dev.get(out).reshape(n, rows)
    ctx.close()
    del wd, xd
    t.cuda.empty_cache()
    _check(got, want, tol, f"Q6_K {rows} x {nb * 256}, {n} rows")
