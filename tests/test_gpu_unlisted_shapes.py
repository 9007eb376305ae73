"""Shapes whose kernels split the probabilities in two -- query groups of 1 to
16 heads that are not a power of two, and head_dim 96 -- from launch lists and
from the padded grid, against the fp64 oracle."""
import math

import pytest
import torch

from parity import custom
from test_gpu_parity import announce, assert_attention, hip_step, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

# Prefill rows around a work-group's queries (8 * (32 // G) at D = 128) and
# 16- and 32-key edges, decode rows around one slice, one wave's slices and
# one partition (128 to 1024 keys), a row without queries.
ROWS = [(1, 17, 16), (20, 50, 30), (1, 1, 0), (0, 16, 16), (3, 3, 0), (1, 1024, 1023), (41, 41, 0), (1, 1025, 1024),
        (9, 300, 291), (2, 33, 31), (1, 2100, 2099), (130, 257, 127), (1, 128, 127), (1, 129, 128)]


@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (24, 8, 128, torch.bfloat16), (24, 8, 64, torch.float16), (12, 4, 96, torch.float16), (4, 4, 96, torch.bfloat16),
    (32, 2, 96, torch.bfloat16), (10, 2, 256, torch.bfloat16), (30, 2, 128, torch.float16), (9, 1, 64, torch.bfloat16),
    (12, 2, 96, torch.bfloat16), (22, 2, 256, torch.float16), (7, 1, 128, torch.bfloat16), (13, 1, 96, torch.bfloat16),
])
@pytest.mark.parametrize("layout", ["kv-interleaved", "token-major"])
def test_grid_shapes(cuda, sea, wl, hq, hkv, d, dtype, layout):  # noqa: F811
    w = custom(wl, ROWS, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda, layout=layout)
    ref_o, ref_l = oracle_step(w, T)
    listed = wl.metadata_tensors(w, cuda)
    grid = {k: v for k, v in listed.items() if not k.startswith("host_")}
    for pt, meta in ((p, m) for p in (None, 32, 512) for m in (listed, grid)):
        announce(f"shape Hq={hq} Hkv={hkv} D={d} {dtype} {layout} partition {pt}, {'list' if meta is listed else 'grid'}")
        o, l = hip_step(sea, wl, w, T, partition_tokens=pt, meta=meta)
        if meta is listed and pt is None:
            assert all(plan[1] > 0 and plan[2] > 0 for plan in meta["_schedules"].values())
        assert_attention(w, o, l, ref_o, ref_l, rows=[i for i, x in enumerate(w.rows) if x.q_len > 0])


def test_grid_without_workspace(cuda, sea, wl):  # noqa: F811
    """A caller that brings no workspace gets every row in one partition."""
    hq, hkv, d, dtype = 24, 8, 128, torch.bfloat16
    w = custom(wl, ROWS, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    announce("grid shape without a workspace")
    _lib, m = sea._lib, wl.metadata_tensors(w, cuda)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    kc, vc = cache.blocks(0)
    o = torch.empty_like(T.q)
    l = torch.empty(T.q.shape[:2], dtype=torch.float32, device=cuda)
    arr = _lib.i64_array
    need = _lib.load().kvhot_paged_attention_workspace_bytes(
        len(w.rows), T.q.shape[0], m["max_q_len"], m["max_k_len"], hq, hkv, d, 16, 0, _lib.dtype_code(dtype))
    assert need > 0
    _lib.check(_lib.load().kvhot_paged_attention(
        T.q.data_ptr(), arr(T.q.stride()), kc.data_ptr(), arr(kc.stride()), vc.data_ptr(), arr(vc.stride()),
        o.data_ptr(), arr(o.stride()), l.data_ptr(), arr(l.stride()), m["block_table"].data_ptr(),
        m["block_table_row_stride"], m["q_lens"].data_ptr(), m["k_lens"].data_ptr(), m["q_starts"].data_ptr(),
        m["q_pos_offsets"].data_ptr(), len(w.rows), T.q.shape[0], m["max_q_len"], m["max_k_len"], hq, hkv, d, 16,
        kc.shape[0], 1.0 / math.sqrt(d), 1, _lib.dtype_code(dtype), 0, None, 0, 0, 0, 0, 0, None, 0,
        _lib.stream_handle(cuda)), "kvhot_paged_attention")
    torch.cuda.synchronize()
    assert_attention(w, o, l, ref_o, ref_l, rows=[i for i, x in enumerate(w.rows) if x.q_len > 0])
