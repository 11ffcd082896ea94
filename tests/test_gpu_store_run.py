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


def _store_and_check(dev, hd, hkv, positions, epi, rot, hilo):
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
        q = np.zeros(n * kvs, np.float32)
        cache.step_epi(0, [(put(q), dev.empty(n * kvs), p, put(K), put(V))], hkv, scale=1 / math.sqrt(hd), bk=put(bk),
                       bv=put(bv), k_norm_w=put(kn), v_norm=True, eps=eps,
                       rope=dr.Rope(dev.ctx, n_t, rot, 10000.0) if rot else None)
        orc.add_bias(wk, bk, n)
        orc.add_bias(wv, bv, n)
        for o in range(0, wk.size, hd):
            seg = wk[o:o + hd].copy()
            orc.rms_norm_inplace(seg, kn, eps)
            wk[o:o + hd] = seg
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
