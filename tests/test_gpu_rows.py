"""The attention kernel for many query rows (attn_rows.hip, head dims 64 and
128; the planner takes it when 64-row workgroups outnumber the CUs) where its
tiles and ranges can go wrong: one key tile, tile counts that leave a key
group without a tile in the last step (1, 2, 3, 5), ragged rows and keys,
grouped heads whose row blocks span two heads, causal prefixes, windows of one
key, scattered active rows, batch slots and the folded Q epilogue -- against
the oracle of attention() (attention.rs:101-186) on the operands as the kernel
rounds them (max-abs 1e-2, mean-abs 1e-3).  Needs an MI355X.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

import dr_attn as dr
import oracle as orc
from helpers import RowsSpec, Shape, bf16_round

from test_gpu_parity import _epilogue_oracle, check, dev, oracle_run, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# (h, hkv, hd, n_total, active positions, window, prefix, batch, epilogue)
CASES = {
    "one_tile": (257, 257, 64, 31, range(31), None, None, 1, False),
    "two_tiles": (130, 130, 128, 64, range(64), None, None, 2, False),
    "three_tiles_causal": (90, 90, 64, 65, range(65), None, 65, 2, True),
    "five_tiles_gqa": (84, 12, 128, 150, range(150), None, None, 2, True),
    "causal_prefix_window": (48, 48, 64, 333, range(333), 70, 300, 1, True),
    "window_one_key": (100, 50, 128, 97, range(97), 1, None, 2, False),
    "window_gqa_span": (70, 10, 64, 290, range(290), 33, None, 2, True),
    "scattered": (64, 32, 128, 400, sorted({*range(0, 400, 7), *range(100, 233), 399}), 150, 120, 2, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_rows_kernel_vs_oracle(dev, name):
    h, hkv, hd, n_t, active, window, prefix, batch, epi = CASES[name]
    active = list(active)
    rng = np.random.default_rng(sum(map(ord, name)))
    n, kvs, eps, put, scale = len(active), hkv * hd, 1e-6, dev.put, 1 / math.sqrt(hd)
    cache = dr.StepCache(dev.ctx, n_t, [hkv], [hd], n_batch=batch)
    p, rows = dr.Pass(dev.ctx, active), np.concatenate([np.arange(i * kvs, (i + 1) * kvs) for i in active])
    table = orc.rope_table(n_t, hd, 10000.0)
    kw = {}
    if epi:
        qn, kn = (rng.uniform(0.5, 1.5, hd).astype(np.float32) for _ in range(2))
        bq, bk, bv = ((0.1 * rng.standard_normal(m * hd)).astype(np.float32) for m in (h, hkv, hkv))
        kw = dict(bq=put(bq), bk=put(bk), bv=put(bv), q_norm_w=put(qn), k_norm_w=put(kn), eps=eps,
                  rope=dr.Rope(dev.ctx, n_t, hd, 10000.0))
    items, wants = [], []
    for b in range(batch):
        K, V = (rng.standard_normal(n_t * kvs).astype(np.float32) for _ in range(2))
        Q = rng.standard_normal(n * h * hd).astype(np.float32)
        cache.store(0, dr.Pass(dev.ctx, range(n_t)), put(K), put(V), batch=b)
        items.append((put(Q), dev.empty(n * h * hd), p, put(K[rows]), put(V[rows])))
        if epi:
            q, K[rows], V[rows] = _epilogue_oracle(Q.copy(), K[rows].copy(), V[rows].copy(), active, h, hkv, hd, bq, bk,
                                                   bv, qn, kn, False, eps, table, hd)
        else:
            q = Q
        s = Shape(n, n_t, h, hkv, hd, sliding_window=window, causal_prefix=prefix, scale=scale)
        c = np.float32(scale * 1.4426950408889634)  # the kernel rounds q * scale * log2 e to bf16
        wants.append(oracle_run(s, RowsSpec(active), RowsSpec(list(range(n_t))), bf16_round(q * c) / c, bf16_round(K),
                                bf16_round(V)))
    cache.step_epi(0, items, h, sliding_window=window, causal_prefix=prefix, scale=scale, **kw)
    info = dev.ctx.last_launch()
    say(f"{name}: launch {info}")
    assert (info["kernel"], info["waves_per_wg"], info["row_blocks"], info["key_groups"]) == (dr.KERNEL_STAGED, 4, 2, 2)
    for b in range(batch):
        check(dev.get(items[b][1]), wants[b], f"{name} slot {b}")


@pytest.mark.parametrize("h,hkv,hd,n_t,slots,window,prefix", [
    (48, 48, 64, 333, (range(333), range(301, 333), [7, 64, 65, 332]), None, 300),
    (84, 12, 128, 150, (range(100, 150), range(150), [0, 149]), 40, None),
])
def test_rows_kernel_slots_of_different_lengths(dev, h, hkv, hd, n_t, slots, window, prefix):
    """Batch slots of different lengths (the shorter ones' workgroups past
    their rows leave at once) in rows of a fused QKV projection, with the
    whole Q epilogue."""
    rng = np.random.default_rng(h + hd)
    qs, kvs, eps, put, scale = h * hd, hkv * hd, 1e-6, dev.put, 1 / math.sqrt(hd)
    fused = qs + 2 * kvs
    qn, kn = (rng.uniform(0.5, 1.5, hd).astype(np.float32) for _ in range(2))
    bq, bk, bv = ((0.1 * rng.standard_normal(m)).astype(np.float32) for m in (qs, kvs, kvs))
    table = orc.rope_table(n_t, hd, 10000.0)
    cache = dr.StepCache(dev.ctx, n_t, [hkv], [hd], n_batch=len(slots))
    items, wants, keep = [], [], []
    for b, active in enumerate(map(list, slots)):
        n = len(active)
        K, V = (rng.standard_normal((n_t, kvs)).astype(np.float32) for _ in range(2))
        R = rng.standard_normal((n, fused)).astype(np.float32)
        cache.store(0, dr.Pass(dev.ctx, range(n_t)), put(K), put(V), batch=b)
        rows, out = put(R), dev.empty(n * qs)
        base = rows.data_ptr()
        items.append((base, out, dr.Pass(dev.ctx, active), base + 4 * qs, base + 4 * (qs + kvs)))
        keep.append((rows, out))
        q, k, v = _epilogue_oracle(R[:, :qs].reshape(-1).copy(), R[:, qs:qs + kvs].reshape(-1).copy(),
                                   R[:, qs + kvs:].reshape(-1).copy(), active, h, hkv, hd, bq, bk, bv, qn, kn, False,
                                   eps, table, hd)
        K[active], V[active] = k.reshape(n, kvs), v.reshape(n, kvs)
        s = Shape(n, n_t, h, hkv, hd, sliding_window=window, causal_prefix=prefix, scale=scale)
        c = np.float32(scale * 1.4426950408889634)
        wants.append(oracle_run(s, RowsSpec(active), RowsSpec(list(range(n_t))), bf16_round(q * c) / c,
                                bf16_round(K.reshape(-1)), bf16_round(V.reshape(-1))))
    cache.step_rows(0, items, h, fused, fused, sliding_window=window, causal_prefix=prefix, scale=scale, bq=put(bq),
                    bk=put(bk), bv=put(bv), q_norm_w=put(qn), k_norm_w=put(kn), eps=eps,
                    rope=dr.Rope(dev.ctx, n_t, hd, 10000.0))
    info = dev.ctx.last_launch()
    assert (info["kernel"], info["waves_per_wg"], info["row_blocks"], info["key_groups"]) == (dr.KERNEL_STAGED, 4, 2, 2)
    for b, (_, out) in enumerate(keep):
        check(dev.get(out), wants[b], f"slot {b}")
