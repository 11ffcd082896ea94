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
from helpers import RowsSpec, Shape, brute_force

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


# ---- which of the two hi/lo kernels a call takes, and batch slots of different lengths


def run_slots(dev, h, hkv, hd, n_t, actives, window, prefix, rot, epi, seed):
    """One step of a batch of slots (their active positions) on a hi/lo layer
    at scale 1.0, Q, K and V in rows of a fused projection; epi: letters b
    (biases), n (QK-norm), rot dims of rotary (0: none).  Checks every slot
    against the oracle and returns the launch."""
    rng = np.random.default_rng(seed)
    eps, put, qs, kvs = 1e-6, dev.put, h * hd, hkv * hd
    fused = qs + 2 * kvs
    kw, qn, kn, bq, bk, bv, table = {}, None, None, None, None, None, None
    if "n" in epi:
        qn, kn = (rng.uniform(0.5, 1.5, hd).astype(np.float32) for _ in range(2))
        kw.update(q_norm_w=put(qn), k_norm_w=put(kn))
    if "b" in epi:
        bq, bk, bv = ((0.1 * rng.standard_normal(m)).astype(np.float32) for m in (qs, kvs, kvs))
        kw.update(bq=put(bq), bk=put(bk), bv=put(bv))
    if rot:
        table = orc.rope_table(n_t, rot, 10000.0)
        kw.update(rope=dr.Rope(dev.ctx, n_t, rot, 10000.0))
    cache = dr.StepCache(dev.ctx, n_t, [hkv], [hd], n_batch=len(actives), precision=[dr.PRECISION_HILO])
    items, wants, keep = [], [], []
    for b, active in enumerate(actives):
        n = len(active)
        K, V = ((rng.standard_normal((n_t, kvs))).astype(np.float32) for _ in range(2))
        R = rng.standard_normal((n, fused)).astype(np.float32)
        if "n" not in epi:  # (scores of unit rows at scale 1.0 would be near one-hot: keep them spread)
            R[:, :qs] *= 0.25
        cache.store(0, dr.Pass(dev.ctx, range(n_t)), put(K), put(V), batch=b)
        rows, out = put(R), dev.empty(n * qs)
        base = rows.data_ptr()
        items.append((base, out, dr.Pass(dev.ctx, active), base + 4 * qs, base + 4 * (qs + kvs)))
        keep.append((R, rows, out))
        q, k, v = _epilogue_oracle(R[:, :qs].reshape(-1).copy(), R[:, qs:qs + kvs].reshape(-1).copy(),
                                   R[:, qs + kvs:].reshape(-1).copy(), active, h, hkv, hd, bq, bk, bv, qn, kn, False,
                                   eps, table, rot)
        K[active], V[active] = k.reshape(n, kvs), v.reshape(n, kvs)
        s = Shape(n, n_t, h, hkv, hd, sliding_window=window, causal_prefix=prefix, scale=1.0)
        wants.append(oracle_run(s, RowsSpec(active), RowsSpec(list(range(n_t))), q, K.reshape(-1), V.reshape(-1)))
    cache.step_rows(0, items, h, fused, fused, sliding_window=window, causal_prefix=prefix, scale=1.0, eps=eps, **kw)
    info = dev.ctx.last_launch()
    say(f"{h}/{hkv} x {hd}, {[len(a) for a in actives]} of {n_t}: launch {info}")
    assert info["kernel"] == dr.KERNEL_HILO
    for b, (R, rows, out) in enumerate(keep):
        check(dev.get(out), wants[b], f"slot {b}")
        assert np.array_equal(dev.get(rows), R)  # the caller's rows are only read
    return info


# (h, hkv, hd, n_total, slots' active positions, window, prefix, rotary dims, epilogue, rows per wave)
PLANS = {
    "hd256_short_plain": (4, 2, 256, 100, [range(80, 100)], None, None, 0, "", 16),
    "hd256_short_norm": (16, 8, 256, 320, [range(64, 320)], 1024, None, 0, "n", 16),  # 2 tiles per workgroup
    "hd256_few_rows": (8, 8, 256, 1321, [range(1319, 1321)] * 3 + [range(1321 - 17, 1321)], None, None, 0, "n", 16),
    "hd256_long_slots": (8, 8, 256, 1200, [range(1071, 1200), range(1130, 1200)], None, None, 0, "n", 32),
    "hd256_long_plain": (8, 8, 256, 1200, [range(1198, 1200), range(1071, 1200)], None, 1100, 0, "", 32),
    "hd256_short_rotary": (4, 2, 256, 100, [range(80, 100), range(99, 100)], None, None, 256, "n", 32),
    "hd256_short_bias": (4, 2, 256, 100, [range(70, 100, 3), range(33, 100)], 50, None, 0, "b", 32),
    "hd512_short_norm": (8, 2, 512, 90, [range(60, 90), range(89, 90)], None, None, 0, "n", 16),
    "hd512_long_slots": (4, 2, 512, 4200, [range(4160, 4200), range(4195, 4200)], None, None, 0, "n", 32),
    "hd512_short_rotary": (8, 2, 512, 90, [range(60, 90), range(89, 90)], None, 75, 512, "nb", 32),
}


@pytest.mark.parametrize("name", list(PLANS))
def test_hilo_kernel_choice(dev, name):
    h, hkv, hd, n_t, slots, window, prefix, rot, epi, rows = PLANS[name]
    info = run_slots(dev, h, hkv, hd, n_t, [list(a) for a in slots], window, prefix, rot, epi, sum(map(ord, name)))
    assert info["rows_per_wave"] == rows


def test_hilo_forced_splits_fit_the_fixed_scratch(dev):
    """32 forced key splits of 150 rows of 8 heads of 256: the 16-row kernel's
    partials (192 rows each, 51 MB) fit the 64 MB of
    dr_attention_cached_noalloc, the 128-row groups of the 32-row kernel (256
    rows each, 67.6 million bytes) would not."""
    h, hd, n_t, n = 8, 256, 5100, 150
    rng = np.random.default_rng(65)
    K, V = ((rng.standard_normal(n_t * h * hd)).astype(np.float32) for _ in range(2))
    Q = (0.25 * rng.standard_normal(n * h * hd)).astype(np.float32)
    cache = dr.StepCache(dev.ctx, n_t, [h], [hd], precision=[dr.PRECISION_HILO])
    cache.store(0, dr.Pass(dev.ctx, range(n_t)), dev.put(K), dev.put(V))
    active, out = list(range(n_t - n, n_t)), dev.empty(n * h * hd)
    dev.ctx.set_split(32)
    try:
        cache.attention(0, [(dev.put(Q), out, dr.Pass(dev.ctx, active))], h, scale=1.0, noalloc=True)
        info = dev.ctx.last_launch()
    finally:
        dev.ctx.set_split(0)
    assert info["n_split"] == 32 and info["rows_per_wave"] == 16
    s = Shape(n, n_t, h, h, hd, scale=1.0)
    check(dev.get(out), oracle_run(s, RowsSpec(active), RowsSpec(list(range(n_t))), Q, K, V), "32 forced splits")


def test_hilo32_error_against_64_bits(dev):
    """Near one-hot rows at scale 1.0, 64 rows over one range of 32 key tiles:
    a row's largest weight is exactly 1 in bf16 (the running maximum is its
    score), so only the others' rounding reaches the output: 2.5e-4 here,
    4.3e-4 when the maximum moves only past a threshold of 8.  Bound between
    them, at their geometric mean."""
    h, hd, n_t, n = 4, 256, 1024, 64
    rng = np.random.default_rng(256)
    K, V = (rng.standard_normal(n_t * h * hd).astype(np.float32) for _ in range(2))
    Q = rng.standard_normal(n * h * hd).astype(np.float32)
    active = list(range(n_t - n, n_t))
    cache = dr.StepCache(dev.ctx, n_t, [h], [hd], precision=[dr.PRECISION_HILO])
    cache.store(0, dr.Pass(dev.ctx, range(n_t)), dev.put(K), dev.put(V))
    rows = slice((n_t - n) * h * hd, None)
    out = dev.empty(n * h * hd)
    dev.ctx.set_split(1)
    try:  # (a bias, of zeros: the 32-row kernel)
        cache.step_epi(0, [(dev.put(Q), out, dr.Pass(dev.ctx, active), dev.put(K[rows].copy()), dev.put(V[rows].copy()))],
                       h, scale=1.0, bq=dev.put(np.zeros(h * hd, np.float32)))
        info = dev.ctx.last_launch()
    finally:
        dev.ctx.set_split(0)
    assert info["rows_per_wave"] == 32 and info["n_split"] == 1
    want = brute_force(Q, K, V, Shape(n, n_t, h, h, hd, scale=1.0), RowsSpec(active), RowsSpec(list(range(n_t))))
    err = np.linalg.norm(dev.get(out).reshape(want.shape) - want) / np.linalg.norm(want)
    say(f"relative error {err:.3e}")
    assert err < 3.3e-4
