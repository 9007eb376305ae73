"""A launch list runs as it was planned whatever partition_tokens the call is
passed (with a schedule it does not apply), through both C entry points,
against the fp64 oracle.  (After test_zz_no_alloc.py, whose first test makes
the process's first no-alloc call.)"""
import math

import pytest
import torch

from conftest import sea_module
from parity import custom
from test_gpu_parity import announce, assert_attention, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

# Segments shared by all the waves of a work-group, several to a work-group, and cut ones, beside a chunk.
ROWS = [(1, 300, 299), (20, 50, 30), (1, 600, 599), (1, 3000, 2999), (1, 17, 16)]


@pytest.mark.parametrize("hq,hkv,d,dtype", [(32, 8, 128, torch.bfloat16), (12, 12, 64, torch.float16),
                                            (8, 1, 128, torch.bfloat16), (16, 4, 256, torch.bfloat16), (24, 8, 128, torch.bfloat16)])
@pytest.mark.parametrize("planned,passed", [(512, 0), (0, 512), (64, 0), (0, 64), (64, 512)])
@pytest.mark.parametrize("rows", [ROWS, ROWS[:2]])
def test_list_of_another_partition_size(cuda, sea, wl, hq, hkv, d, dtype, planned, passed, rows):  # noqa: F811
    _lib, pak = sea_module("_lib"), sea_module("paged_attention_kernel")
    lib, arr = _lib.load(), _lib.i64_array
    w = custom(wl, rows, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    kc, vc = cache.blocks(0)
    m = wl.metadata_tensors(w, cuda)
    code = _lib.dtype_code(dtype)
    plan = pak._schedule(m, cuda, hq, hkv, d, 16, planned, True, code)
    if plan is None:  # no lists of fixed partitions: the planner returned no units
        plan = (torch.zeros(8, dtype=torch.int32, device=cuda), 0, 0, 0, 0, 0)
    sched, n_dec, n_pre, n_mrg, need, n_pfx = plan
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=cuda)
    for noalloc in (False, True):
        announce(f"list planned with {planned}, called with {passed}: Hq={hq} Hkv={hkv} D={d} {len(rows)} rows, "
                 f"{'no-alloc' if noalloc else 'workspace'}")
        o = torch.full_like(T.q, float("nan"))
        l = torch.full(T.q.shape[:2], float("nan"), device=cuda)
        args = (T.q.data_ptr(), arr(T.q.stride()), kc.data_ptr(), arr(kc.stride()), vc.data_ptr(), arr(vc.stride()),
                o.data_ptr(), arr(o.stride()), l.data_ptr(), arr(l.stride()), m["block_table"].data_ptr(),
                m["block_table_row_stride"], m["q_lens"].data_ptr(), m["k_lens"].data_ptr(), m["q_starts"].data_ptr(),
                m["q_pos_offsets"].data_ptr(), len(w.rows), T.q.shape[0], m["max_q_len"], m["max_k_len"], hq, hkv, d, 16,
                kc.shape[0], 1.0 / math.sqrt(d), 1, code, passed, sched.data_ptr(), n_dec, n_pre, n_mrg, n_pfx, need)
        if noalloc:
            status = lib.kvhot_paged_attention_noalloc(*args, _lib.stream_handle(cuda))
        else:
            status = lib.kvhot_paged_attention(*args, ws.data_ptr(), need, _lib.stream_handle(cuda))
        _lib.check(status, "attention")
        torch.cuda.synchronize()
        assert_attention(w, o, l, ref_o, ref_l)
