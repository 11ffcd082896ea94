"""The store of contiguous rows that need not fill whole 32-key tiles, and of
rows at a sorted position list (kv_store_run_kernel): runs that begin and end
inside a tile or inside a row group of 4, one-row runs, lists with gaps of
every size, every built head dim, bf16 and hi/lo layers, with and without the
epilogue (bias, K norm, V norm, full and partial RoPE).
StepCache::store (cache.rs:62-71) over forward.rs:291-310: gathered rows equal
bf16 (hi/lo layers: hi + lo halves) of the oracle's rows bit for bit, and every
other position keeps its value.  Needs an MI355X.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

import dr_attn as dr
import oracle as orc

from test_gpu_parity import dev, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _stored(x: np.ndarray, t, hilo: bool) -> np.ndarray:
    x = t.from_numpy(x.reshape(-1).copy())
    hi = x.to(t.bfloat16).to(t.float32)
    return (hi + (x - hi).to(t.bfloat16).to(t.float32) if hilo else hi).numpy()


@pytest.mark.parametrize("hilo", [False, True])
@pytest.mark.parametrize("hd,hkv,p0,n,epi,rot", [
    (64, 3, 5, 1, False, 0), (64, 2, 31, 2, True, 64), (64, 2, 30, 70, True, 24), (128, 4, 2041, 77, True, 128),
    (128, 2, 33, 30, True, 64), (128, 3, 0, 33, False, 0), (256, 2, 61, 6, True, 256), (256, 8, 100, 129, False, 0),
    (256, 2, 3, 64, True, 64), (512, 2, 7, 60, True, 512), (512, 1, 32, 32, False, 0), (512, 2, 63, 2, True, 0),
])
def test_store_run_vs_oracle(dev, hd, hkv, p0, n, epi, rot, hilo):
    _store_and_check(dev, hd, hkv, list(range(p0, p0 + n)), epi, rot, hilo)


@pytest.mark.parametrize("hilo", [False, True])
@pytest.mark.parametrize("hd,hkv,n,epi,rot", [
    (64, 3, 2, False, 0), (64, 2, 33, True, 24), (128, 4, 145, True, 128), (128, 2, 31, False, 0), (256, 2, 70, True, 256),
    (256, 3, 32, True, 64), (512, 2, 37, True, 512), (512, 1, 65, False, 0),
])
def test_store_list_vs_oracle(dev, hd, hkv, n, epi, rot, hilo):
    rng = np.random.default_rng(hd + 5 * n + rot)
    _store_and_check(dev, hd, hkv, sorted(rng.choice(3 * n + 40, n, replace=False).tolist()), epi, rot, hilo)


@pytest.mark.parametrize("hd,hkv,p0,n,ops,rot,hilo", [
    # whole tiles of bf16 layers with an epilogue, both sides of the rule between the tile and the run kernel
    (64, 2, 32, 64, "n", 0, False), (64, 2, 0, 96, "b", 24, False), (64, 3, 32, 32, "b", 64, False),
    (64, 8, 0, 32 * 17, "", 64, False), (64, 8, 64, 32 * 33, "nv", 64, False), (128, 2, 64, 64, "bn", 64, False),
    (128, 8, 32, 32 * 16, "b", 0, False), (128, 8, 0, 32 * 17, "b", 0, False), (128, 8, 0, 32 * 17, "n", 128, False),
    (128, 16, 0, 32 * 32, "b", 128, False), (128, 16, 0, 32 * 64, "n", 128, False), (128, 4, 0, 96, "v", 0, False),
    (256, 2, 32, 64, "n", 256, False), (256, 8, 0, 32 * 17, "b", 0, False), (256, 8, 0, 32 * 17, "", 64, False),
    (256, 2, 32, 64, "nv", 64, False),
    # hi/lo tiles and head dim 512, both sides of the rule between the general and the run kernel
    (64, 8, 0, 32 * 41, "", 0, True), (128, 8, 0, 32 * 17, "", 0, True), (256, 8, 0, 32 * 16, "", 0, True),
    (256, 8, 0, 32 * 17, "", 0, True), (512, 2, 0, 64, "n", 0, True), (512, 2, 0, 96, "n", 0, True),
    (512, 2, 32, 64, "b", 0, True), (512, 2, 64, 32 * 33, "", 0, False), (256, 2, 5, 20, "", 0, True),
])
def test_store_whole_tiles_vs_oracle(dev, hd, hkv, p0, n, ops, rot, hilo):
    _store_and_check(dev, hd, hkv, list(range(p0, p0 + n)), bool(ops or rot), rot, hilo, ops)


@pytest.mark.parametrize("hd,hkv,n,hilo", [
    (64, 8, 32 * 81, False), (64, 8, 32 * 41, True), (128, 8, 32 * 17, False), (128, 8, 32 * 17, True),
    (256, 2, 31, False), (256, 8, 32 * 40, True), (256, 8, 32 * 41, True), (512, 2, 70, True), (512, 4, 32 * 49, False),
])
def test_store_plain_lists_both_sides(dev, hd, hkv, n, hilo):
    rng = np.random.default_rng(hd + n)
    _store_and_check(dev, hd, hkv, sorted(rng.choice(2 * n + 40, n, replace=False).tolist()), False, 0, hilo)


def _store_and_check(dev, hd, hkv, positions, epi, rot, hilo, ops="bnv"):
    n = len(positions)
    rng = np.random.default_rng(hd + positions[0] + 3 * n + rot)
    n_t, kvs, eps, put = positions[-1] + 36, hkv * hd, 1e-6, dev.put
    cache = dr.StepCache(dev.ctx, n_t, [hkv], [hd], precision=[dr.PRECISION_HILO if hilo else dr.PRECISION_BF16])
    K0, V0 = (rng.standard_normal((n_t, kvs)).astype(np.float32) for _ in range(2))
    cache.store(0, dr.Pass(dev.ctx, range(n_t)), put(K0), put(V0))
    K, V = (rng.standard_normal((n, kvs)).astype(np.float32) for _ in range(2))
    wk, wv, p = K.reshape(-1).copy(), V.reshape(-1).copy(), dr.Pass(dev.ctx, positions)
    if epi:
        bk, bv = ((0.1 * rng.standard_normal(kvs)).astype(np.float32) for _ in range(2))
        kn = rng.uniform(0.5, 1.5, hd).astype(np.float32)
        kw = dict(bk=put(bk), bv=put(bv)) if "b" in ops else {}
        if "n" in ops:
            kw.update(k_norm_w=put(kn))
        q = np.zeros(n * kvs, np.float32)
        cache.step_epi(0, [(put(q), dev.empty(n * kvs), p, put(K), put(V))], hkv, scale=1 / math.sqrt(hd), v_norm="v" in ops,
                       eps=eps, rope=dr.Rope(dev.ctx, n_t, rot, 10000.0) if rot else None, **kw)
        if "b" in ops:
            orc.add_bias(wk, bk, n)
            orc.add_bias(wv, bv, n)
        for o in range(0, wk.size, hd):
            if "n" in ops:
                seg = wk[o:o + hd].copy()
                orc.rms_norm_inplace(seg, kn, eps)
                wk[o:o + hd] = seg
            if "v" in ops:
                seg = wv[o:o + hd].copy()
                orc.rms_norm_noscale(seg, eps)
                wv[o:o + hd] = seg
        if rot:
            orc.rotate_rows(wk, orc.rope_table(n_t, rot, 10000.0), positions, hkv, hd, rot)
    else:
        cache.store(0, p, put(K), put(V))
    K0[positions], V0[positions] = wk.reshape(n, kvs), wv.reshape(n, kvs)
    ok, ov = dev.empty(n_t * kvs), dev.empty(n_t * kvs)
    cache.gather(0, list(range(n_t)), ok, ov)
    assert np.array_equal(dev.get(ok), _stored(K0, dev.t, hilo))
    assert np.array_equal(dev.get(ov), _stored(V0, dev.t, hilo))
