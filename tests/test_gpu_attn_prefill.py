"""GPU envelope: tiled prefill attention over the KV ring.

Reference: the GPU engine's --flash-prefill tier (attention_flash,
src/gpu/gpu_engine.cpp:3292-3372; k_flash_softmax 1481-1545; k_flash_finish
1547-1560). Like that tier this is a tile-wise summation schedule with bf16
probabilities in the p.v product, gated on an envelope, not bits. The oracle is
exact f64 attention over the same bf16 q, K, V (scaling taken as the f32 value
the kernel uses). Each weight enters the p.v product as bf16(e), within 2^-8
of e relative (bf16 carries 8 significant bits; round to nearest), while the
normalizer sums e itself, so per output
|o - o64| <= (2^-8 + 2e-5) * sum_j p_j |v_j|; the 2e-5 covers the f32 scores,
exp2 and the per-tile rescales.
"""
import math

import numpy as np
import pytest

import oracle as O
from util import BF16, to_dev

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -8 + 2e-5


def prefill_case(prims, T, nq, nkv, D, slots, pos0, window=0, seed=101, scaling=None, heads=None, rows=None):
    """keys 0..pos0+T-1 live in the ring (key j in slot j % slots); check the
    given heads and query rows (all by default) against f64 attention"""
    q = O.normal(seed, (T, nq, D), 0.0, 1.0, BF16)
    kc = O.normal(seed + 1, (slots, nkv, D), 0.0, 1.0, BF16)
    vc = O.normal(seed + 2, (slots, nkv, D), 0.0, 1.0, BF16)
    scaling = 1.0 / math.sqrt(D) if scaling is None else scaling
    out = prims.attn_prefill(to_dev(q, BF16), to_dev(kc, BF16), to_dev(vc, BF16), pos0, scaling, window)
    out = out.cpu().numpy().astype(np.float64)
    qf, K, Vv = O.to_f64(q, BF16), O.to_f64(kc, BF16), O.to_f64(vc, BF16)
    s32 = float(np.float32(scaling))
    hpg = nq // nkv
    heads = range(nq) if heads is None else heads
    rows = range(T) if rows is None else rows
    worst = 0.0
    for h in heads:
        g = h // hpg
        for t in rows:
            p_ = pos0 + t
            lo = max(0, p_ - window + 1) if window > 0 else 0
            sl = np.arange(lo, p_ + 1) % slots
            Kg, Vg = K[sl, g, :], Vv[sl, g, :]
            s = (Kg @ qf[t, h]) * s32
            p = np.exp(s - s.max())
            p /= p.sum()
            ref = p @ Vg
            bound = p @ np.abs(Vg)
            err = np.abs(out[t, h] - ref)
            assert np.all(err <= TOL * bound), (h, t, float((err / bound).max()))
            worst = max(worst, float((err / bound).max()))
    return worst


@pytest.mark.parametrize("nq,nkv,D", ((40, 8, 128), (8, 8, 64), (16, 2, 128), (7, 7, 64)))
def test_shapes(prims, nq, nkv, D):
    prefill_case(prims, 100, nq, nkv, D, 128, 0)


@pytest.mark.parametrize("hpg", (1, 2, 3, 4, 5, 6, 8))
@pytest.mark.parametrize("D", (64, 128))
def test_group_sizes(prims, hpg, D):
    """query-head counts per KV head: pairs of a wave mix rows and heads"""
    prefill_case(prims, 70, 2 * hpg, 2, D, 80, 0, seed=110 + hpg)


@pytest.mark.parametrize("hpg", (9, 10, 16))
def test_large_groups(prims, hpg):
    """groups past 8 heads (a window's key steps start by groups of 3 x 3, 2 x 5, 2 x 8)"""
    prefill_case(prims, 70, 2 * hpg, 2, 128, 80, 0, seed=160 + hpg)


def test_real_model_heads(prims):
    """32 query / 2 kv heads, head_dim 128, a chunk after a 200-token prefix"""
    prefill_case(prims, 130, 32, 2, 128, 400, 200, seed=170)


def test_chunked_prefill(prims):
    """a second chunk: rows at positions 50..126 see the first chunk's keys too"""
    prefill_case(prims, 77, 40, 8, 128, 160, 50, seed=120)


def test_window_and_ring(prims):
    """sliding window of 64 keys over a 128-slot ring that has wrapped"""
    prefill_case(prims, 60, 40, 8, 128, 128, 200, window=64, seed=121)
    prefill_case(prims, 96, 16, 2, 64, 200, 0, window=33, seed=122)


def test_window_ring_many_steps(prims):
    """a 256-key window over a 600-slot ring, positions 1000..1299: nine 64-key
    steps per tile, the ring wrapping (slot 0 again at key 1200) inside the
    chunk, so steps staged two ahead straddle the wrap"""
    prefill_case(prims, 300, 8, 2, 128, 600, 1000, window=256, seed=123)
    prefill_case(prims, 300, 10, 2, 64, 600, 1000, window=200, seed=124)


def test_short_and_ragged(prims):
    """one row, and row counts about a wave's 32 pairs and a tile's 128"""
    for T in (1, 15, 17, 31, 32, 33):
        prefill_case(prims, T, 8, 2, 128, 64, 0, seed=130 + T)


def test_peaked_scores(prims):
    """scaling 1: the running maxima move late and the lazy rescale runs"""
    prefill_case(prims, 300, 8, 2, 128, 512, 0, scaling=1.0, seed=140)


@pytest.mark.parametrize("scaling", (0.35, 0.6))
def test_reference_kept_below_threshold(prims, scaling):
    """a row's reference maximum moves only when a new maximum passes it by more
    than 8 in log2 units; at these scalings the maxima of later steps often pass
    the first one by a few units without moving it, so weights between 1 and 2^8
    reach the sums and the p.v product"""
    prefill_case(prims, 257, 8, 2, 128, 512, 0, scaling=scaling, seed=141)


@pytest.mark.parametrize("scaling", (-1.0 / math.sqrt(128), -1.0, 0.0, 1e-30))
def test_scaling_signs(prims, scaling):
    """the kernel multiplies by |scaling| inside the exponent: a negative
    scaling (q enters negated, so the weights favour the least similar keys),
    zero (every attended key weighs the same) and a tiny one"""
    prefill_case(prims, 90, 8, 2, 128, 128, 20, scaling=scaling, seed=145)


def test_config3_prefill_sampled(prims):
    """config 3's prompt: 4096 tokens, 40 q / 8 kv heads, causal; a sample of
    heads and rows against f64 (the full f64 check is minutes of numpy)"""
    rows = list(range(0, 40)) + list(range(2040, 2056)) + list(range(4060, 4096))
    prefill_case(prims, 4096, 40, 8, 128, 4096, 0, seed=150, heads=(0, 4, 5, 23, 39), rows=rows)


def test_errors(prims):
    import torch
    q = torch.zeros((4, 6, 128), dtype=torch.bfloat16, device="cuda:0")
    kc = torch.zeros((16, 4, 128), dtype=torch.bfloat16, device="cuda:0")
    with pytest.raises(Exception, match="multiple"):
        prims.attn_prefill(q, kc, kc, 0, 0.1)
    q = torch.zeros((20, 8, 128), dtype=torch.bfloat16, device="cuda:0")
    with pytest.raises(Exception, match="cache ring"):
        prims.attn_prefill(q, kc, kc, 0, 0.1)


@pytest.mark.parametrize("T,nq,nkv,D,pos0,window", (
    (1, 40, 8, 128, 4000, 0),       # one row: eleven live pairs short of one wave, many parts
    (2, 7, 7, 64, 9000, 0),         # more parts than one wave merges
    (51, 40, 8, 128, 2111, 0),      # 255 pairs: a tile one pair short of full
    (52, 40, 8, 128, 2112, 0),      # 260 pairs: a second tile of four
    (33, 32, 2, 128, 5000, 0),      # two tiles of 16 heads a row, the last with one wave live
    (129, 16, 2, 64, 1000, 700),    # window starts inside, before and past the parts
    (300, 2, 2, 128, 5000, 2000),   # 256 rows a tile: parts whose keys lie before the last rows' windows
    (400, 8, 1, 128, 0, 0),         # causal from key 0: tiles of different length, empty parts
))
def test_key_split(prims, T, nq, nkv, D, pos0, window):
    """few pair tiles over many keys: the tiles' keys split into parts that a
    second kernel merges; edges of pair tiles, parts and windows, on a ring
    that has wrapped when a window allows it"""
    slots = T + window + 40 if window else pos0 + T
    rows = sorted({0, 1, T // 2, T - 2, T - 1} & set(range(T)))
    prefill_case(prims, T, nq, nkv, D, slots, pos0, window=window, seed=180 + T, heads=(0, nq // 2, nq - 1), rows=rows)


def test_key_split_without_workspace(prims):
    """a context whose workspace holds no partials runs the tiles unsplit: the
    same envelope, and both close to each other"""
    import mgprims
    import torch
    small = mgprims.Prims(0, workspace_bytes=4096)
    q = to_dev(O.normal(190, (20, 40, 128), 0.0, 1.0, BF16), BF16)
    k = to_dev(O.normal(191, (3000, 8, 128), 0.0, 1.0, BF16), BF16)
    v = to_dev(O.normal(192, (3000, 8, 128), 0.0, 1.0, BF16), BF16)
    a = small.attn_prefill(q, k, v, 2980, 0.088)
    b = prims.attn_prefill(q, k, v, 2980, 0.088)
    small.close()
    # both are within 2^-8 sum p |v| of the same value, and sum p |v| is below 1
    assert float((a - b).abs().max()) <= 2 * TOL
    prefill_case(prims, 20, 40, 8, 128, 3000, 2980, seed=190)
    assert torch.isfinite(a).all()


@pytest.mark.parametrize("T,nq,nkv,D,pos0,window", (
    (57, 32, 2, 128, 986, 1024),
    (129, 40, 8, 128, 938, 1024),
    (1606, 1, 1, 128, 0, 542),
    (130, 8, 1, 64, 950, 1030),
))
def test_key_split_window_fills(prims, T, nq, nkv, D, pos0, window):
    """a window that fills inside the call: the middle tiles attend more keys
    than the first and the (partial) last one; every row of some heads"""
    prefill_case(prims, T, nq, nkv, D, pos0 + T, pos0, window=window, seed=200 + T, heads=sorted({0, nq // 2, nq - 1}))


@pytest.mark.parametrize("T,nq,nkv,D,pos0,window", (
    (100, 32, 2, 128, 9000, 0),
    (64, 8, 8, 64, 3000, 0),
    (129, 40, 8, 128, 938, 1024),
    (57, 32, 2, 128, 986, 1024),    # tiles of 16 or 8 rows in groups of 32
    (300, 2, 2, 128, 5000, 2000),   # 256 rows a tile: rows whose keys start four steps in
))
def test_key_split_rounds_the_same_weights(prims, T, nq, nkv, D, pos0, window):
    """Split or not, a pair's weights start from one reference, so bf16 rounds the
    same numbers and a row's output does not depend on how its call is cut: only
    f32 sums differ, a chain of some 600 additions of 2^-25 rms each (1.5e-6 by a
    random walk, gated at 2e-5). Weights rounded against another reference are 2e-3
    apart. (No reference moves here: scores of std 1 stay within 8 of the first
    step's maximum.)"""
    import mgprims
    import torch
    small = mgprims.Prims(0, workspace_bytes=4096)
    q = to_dev(O.normal(210, (T, nq, D), 0.0, 1.0, BF16), BF16)
    k = to_dev(O.normal(211, (pos0 + T, nkv, D), 0.0, 1.0, BF16), BF16)
    v = to_dev(O.normal(212, (pos0 + T, nkv, D), 0.0, 1.0, BF16), BF16)
    a = small.attn_prefill(q, k, v, pos0, 1.0 / math.sqrt(D), window)
    b = prims.attn_prefill(q, k, v, pos0, 1.0 / math.sqrt(D), window)
    again = prims.attn_prefill(q, k, v, pos0, 1.0 / math.sqrt(D), window)
    small.close()
    assert torch.equal(b, again)
    assert float((a - b).norm() / a.norm()) < 2e-5
