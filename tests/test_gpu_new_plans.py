"""Cut prefill units and launches of prefill units beside decode work-groups,
over pool layouts, blocks of 32 tokens, calls without causal masking and values
that are not finite, and with both kinds of work-group in turns: against the
fp64 oracle, with the plan looked at."""
import math

import numpy as np
import pytest
import torch

from oracle import paged_ref
from parity import check_attention, custom
from test_gpu_nonfinite import INF, NAN, reference
from test_gpu_parity import announce, assert_attention, f32, hip_step, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

SHAPES = [(32, 8, 128, torch.bfloat16), (12, 12, 64, torch.float16), (24, 8, 128, torch.bfloat16), (12, 4, 96, torch.float16)]
# cut units beside decode rows, one of them cut; a chunk that ends inside a block
ROWS = [(40, 2500, 2460), (1, 900, 899), (1, 3000, 2999), (3, 35, 32), (1, 17, 16)]


def plan(meta):
    """(decode, prefill, merge, prefix) units of the call's launch list."""
    (_, n_dec, n_pre, n_mrg, _, n_pfx), = meta["_schedules"].values()
    return n_dec, n_pre, n_mrg, n_pfx


def assert_mixed(meta):
    """Decode work-groups of 4 waves and prefill units in one launch."""
    n_dec, n_pre, _, n_pfx = plan(meta)
    assert n_dec % 8 == 4 and n_pre > n_pfx


@pytest.mark.parametrize("hq,hkv,d,dtype", SHAPES)
@pytest.mark.parametrize("layout", ["kv-interleaved", "head-major", "token-major"])
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("decode", [True, False])
def test_layouts_and_block_sizes(cuda, sea, wl, hq, hkv, d, dtype, layout, bs, decode):  # noqa: F811
    w = custom(wl, [x for x in ROWS if decode or x[0] > 1], hq, hkv, d, dtype, bs=bs)
    T = wl.make_tensors(w, cuda, layout=layout)
    ref_o, ref_l = oracle_step(w, T)
    announce(f"cut units Hq={hq} Hkv={hkv} D={d} {dtype} {layout} blocks of {bs}, decode rows {decode}")
    meta = wl.metadata_tensors(w, cuda)
    o, l = hip_step(sea, wl, w, T, meta=meta)
    assert_attention(w, o, l, ref_o, ref_l)
    assert plan(meta)[2] > 0  # merge units
    if decode:
        assert_mixed(meta)


@pytest.mark.parametrize("hq,hkv,d,dtype", SHAPES + [(16, 4, 256, torch.bfloat16)])
@pytest.mark.parametrize("decode", [True, False])
def test_without_causal_masking(cuda, sea, wl, hq, hkv, d, dtype, decode):  # noqa: F811
    w = custom(wl, [x for x in ROWS if decode or x[0] > 1] + [(40, 1500, 1000)], hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    kc, vc = cache.blocks(0)
    q_lens, k_lens, q_starts, offs, bt = w.arrays()
    scale = 1.0 / math.sqrt(d)
    ref_o, ref_l = paged_ref.paged_attention(f32(T.q), f32(kc), f32(vc), q_lens, k_lens, q_starts, offs, bt, hq, hkv,
                                             scale, is_causal=False)
    announce(f"no causal masking Hq={hq} Hkv={hkv} D={d} {dtype}, decode rows {decode}")
    meta = wl.metadata_tensors(w, cuda)
    o, l = sea.paged_flash_attention(T.q, kc, vc, meta, hq, hkv, scale, is_causal=False)
    check_attention(f32(o), l.cpu().numpy(), ref_o, ref_l, dtype)
    assert plan(meta)[2] > 0
    if decode and d <= 128:
        assert_mixed(meta)


@pytest.mark.parametrize("hq,hkv,d,dtype", [(32, 8, 128, torch.bfloat16), (12, 12, 64, torch.float16),
                                            (16, 4, 256, torch.bfloat16)])
@pytest.mark.parametrize("rows", [ROWS[:1], ROWS])
def test_infinite_values_beside_a_cut(cuda, sea, wl, hq, hkv, d, dtype, rows):  # noqa: F811
    """Keys that all of a row's queries see, in the first and in a later part."""
    w = custom(wl, rows, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    for key, h, dim, x in ((5, 0, 3, INF), (700, 0, 4, -INF), (1900, 1, 5, NAN), (2459, 1, 6, INF)):
        T.kv_cache[0, 1, int(w.rows[0].block_table[key // 16]), key % 16, h, dim] = x
    kc, vc = cache.blocks(0)
    ref = reference(w, T, True)
    announce(f"infinite values beside a cut Hq={hq} Hkv={hkv} D={d} {dtype}, {len(rows)} rows")
    meta = wl.metadata_tensors(w, cuda)
    o, _ = sea.paged_flash_attention(T.q, kc, vc, meta, hq, hkv, 1.0 / math.sqrt(d))
    o = f32(o).astype(np.float64)
    assert plan(meta)[2] > 0
    assert np.array_equal(np.isnan(o), np.isnan(ref))
    assert np.array_equal(np.where(np.isinf(o), o, 0), np.where(np.isinf(ref), ref, 0))
    fin = np.isfinite(ref)
    check_attention(np.where(fin, o, 0), None, np.where(fin, ref, 0), None, dtype)


@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (32, 8, 128, torch.bfloat16), (16, 1, 128, torch.float16), (16, 2, 64, torch.bfloat16), (12, 12, 64, torch.float16),
    (24, 8, 128, torch.bfloat16), (12, 4, 96, torch.float16),
])
@pytest.mark.parametrize("units,groups,prior", [(256, 256, 0), (300, 256, 16), (700, 256, 0), (1100, 512, 500)])
def test_both_kinds_in_turns(cuda, sea, wl, hq, hkv, d, dtype, units, groups, prior):  # noqa: F811
    """At least `units` prefill units and `groups` decode work-groups: whole
    turns of 256, and what is left of either."""
    g = hq // hkv
    qpw = 4 * ({64: 64, 96: 32, 128: 32}[d] // g)
    rows = [(qpw, qpw + prior + i % 3, prior + i % 3) for i in range(-(-units // hkv))]
    rows += [(1, 250 + 5 * (i % 13), 249 + 5 * (i % 13)) for i in range(-(-3 * groups // (2 * hkv)))]
    w = custom(wl, rows, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    announce(f"turns of {units} units and {groups} work-groups Hq={hq} Hkv={hkv} D={d} {dtype}")
    meta = wl.metadata_tensors(w, cuda)
    o, l = hip_step(sea, wl, w, T, meta=meta)
    assert_attention(w, o, l, ref_o, ref_l)
    assert_mixed(meta)
    n_dec, n_pre, _, n_pfx = plan(meta)
    assert n_pre - n_pfx >= units and n_dec // 4 >= groups
