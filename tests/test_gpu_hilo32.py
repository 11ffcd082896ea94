"""The 32-row hi/lo kernel (attn_hilo32.hip, head dims 256 and 512) where its
tiles and ranges can go wrong: row counts around a wave (32) and a workgroup
(128 rows at head dim 256, 64 at 512), one key tile, ragged key counts, causal
prefixes whose rows end inside, at the edge of and before a tile, windows of
one key, key splits with fewer tiles than splits, active rows that are not
contiguous, and the Q epilogue (bias, QK-norm, full RoPE) applied as Q is
loaded -- against the oracle of attention() (attention.rs:101-186) over the
oracle's epilogue, at kq_scale 1.0 with the bar of the other hi/lo tests
(max-abs 1e-2, mean-abs 1e-3).  Needs an MI355X.
"""
from __future__ import annotations

import numpy as np
import pytest

import dr_attn as dr
import oracle as orc
from helpers import RowsSpec, Shape

from test_gpu_parity import _epilogue_oracle, check, dev, oracle_run, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# (h, hkv, hd, n_total, active positions, window, prefix, n_split)
CASES = {
    "hd256_one_row": (2, 2, 256, 1, [0], None, None, 1),
    "hd256_wave_edge": (2, 1, 256, 65, range(49, 65), None, None, 1),  # 32 packed rows
    "hd256_workgroup_plus_one": (3, 3, 256, 129, range(129), None, 100, 1),
    "hd256_causal_all": (4, 2, 256, 200, range(200), None, 200, 1),
    "hd256_causal_window": (4, 2, 256, 333, range(333), 64, 301, 1),
    "hd256_window_one_key": (2, 2, 256, 97, range(97), 1, None, 1),
    "hd256_splits_over_tiles": (4, 4, 256, 70, range(40, 70), None, None, 5),
    "hd256_split_causal": (4, 2, 256, 257, range(257), None, 250, 3),
    "hd256_scattered": (4, 2, 256, 300, [0, 1, 5, 31, 32, 33, 64, 100, 163, 164, 255, 256, 298, 299], 120, 200, 1),
    "hd512_one_row": (2, 1, 512, 3, [2], None, None, 1),
    "hd512_workgroup_plus_one": (2, 2, 512, 65, range(65), None, 33, 1),
    "hd512_causal_window": (8, 2, 512, 170, range(170), 48, 150, 1),
    "hd512_split_scattered": (4, 2, 512, 260, [3, 31, 32, 95, 96, 97, 200, 259], None, 97, 4),
}


@pytest.mark.parametrize("name", list(CASES))
def test_hilo32_vs_oracle(dev, name):
    h, hkv, hd, n_t, active, window, prefix, n_split = CASES[name]
    active = list(active)
    rng = np.random.default_rng(sum(map(ord, name)))
    eps, kvs, put = 1e-6, hkv * hd, dev.put
    qn, kn = (rng.uniform(0.5, 1.5, hd).astype(np.float32) for _ in range(2))
    bq, bk, bv = ((0.1 * rng.standard_normal(m * hd)).astype(np.float32) for m in (h, hkv, hkv))
    table = orc.rope_table(n_t, hd, 10000.0)
    rope = dr.Rope(dev.ctx, n_t, hd, 10000.0)
    cache = dr.StepCache(dev.ctx, n_t, [hkv], [hd], precision=[dr.PRECISION_HILO])
    K, V = (rng.standard_normal(n_t * kvs).astype(np.float32) for _ in range(2))
    Q = rng.standard_normal(len(active) * h * hd).astype(np.float32)
    cache.store(0, dr.Pass(dev.ctx, range(n_t)), put(K), put(V))  # rows that are not active keep these
    rows = np.concatenate([np.arange(p * kvs, (p + 1) * kvs) for p in active])
    out = dev.empty(len(active) * h * hd)
    dev.ctx.set_split(n_split)
    try:
        cache.step_epi(0, [(put(Q), out, dr.Pass(dev.ctx, active), put(K[rows]), put(V[rows]))], h,
                       sliding_window=window, causal_prefix=prefix, scale=1.0, bq=put(bq), bk=put(bk), bv=put(bv),
                       q_norm_w=put(qn), k_norm_w=put(kn), v_norm=True, eps=eps, rope=rope)
        info = dev.ctx.last_launch()
    finally:
        dev.ctx.set_split(0)
    say(f"{name}: launch {info}")
    assert info["kernel"] == dr.KERNEL_HILO and info["rows_per_wave"] == 32 and info["n_split"] == n_split
    q, k, v = _epilogue_oracle(Q.copy(), K[rows].copy(), V[rows].copy(), active, h, hkv, hd, bq, bk, bv, qn, kn,
                               True, eps, table, hd)
    K[rows], V[rows] = k, v
    s = Shape(len(active), n_t, h, hkv, hd, sliding_window=window, causal_prefix=prefix, scale=1.0)
    want = oracle_run(s, RowsSpec(active), RowsSpec(list(range(n_t))), q, K, V)
    check(dev.get(out), want, name)
