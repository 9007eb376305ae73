"""Calls of the no-alloc entry point that stay off its scratch array, and so
may overlap on several streams: fp32, query groups that are not a power of
two, head_dim 96, and lists without decode rows.  On the CPU: none of them
asks for the array or is held to its size.  On a GPU: their results against the fp64 oracle.
(After test_zz_no_alloc.py, whose first test makes the process's first no-alloc
call.)"""
import math

import pytest
import torch

from conftest import sea_module
from parity import custom
from test_abi import FAKE, _i64, lib, no_gpu  # noqa: F401  (lib: fixture)
from test_gpu_parity import announce, assert_attention, oracle_step, wl  # noqa: F401  (wl: fixture)


@no_gpu
@pytest.mark.parametrize("hq,d,dtype,units", [
    (32, 128, 2, (0, 16, 8, 0)),                                            # no decode rows
    (32, 128, 0, None), (24, 128, 2, (16, 0, 8, 0)), (32, 96, 1, (16, 8, 8, 8)), (24, 64, 1, None),
])
@pytest.mark.parametrize("nbytes", [1 << 20, (64 << 20) + 1])
def test_the_scratch_is_not_asked_for(lib, hq, d, dtype, units, nbytes):  # noqa: F811
    f = FAKE
    q3, c4, l2 = _i64(hq * d, d, 1), _i64(16 * 8 * d, 8 * d, d, 1), _i64(hq, 1)
    args = [f, q3, f, c4, f, c4, f, q3, f, l2, f, 4096, f, f, f, f,
            64, 64, 1, 65536, hq, 8, d, 16, 1 << 20, 0.1, 1, dtype, 0, f if units else None, *(units or (0, 0, 0, 0)),
            nbytes if units else 0, None]
    # No device here: the call fails where it launches, not where it asks for the scratch's address.
    assert lib.kvhot_paged_attention_noalloc(*args) > 0
    assert lib.kvhot_last_error().startswith(b"paged_attention: ")


PREFILL = [(40, 2500, 2460), (3, 1500, 1497), (130, 700, 570)]
MIXED = PREFILL[:2] + [(1, 300, 299), (1, 3000, 2999), (1, 17, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,dtype,spec,scheduled", [
    (32, 8, 128, torch.bfloat16, PREFILL, True), (12, 12, 64, torch.float16, PREFILL, True),
    (16, 4, 256, torch.bfloat16, PREFILL, True), (24, 8, 128, torch.bfloat16, PREFILL, True),
    (24, 8, 128, torch.bfloat16, MIXED, True), (24, 8, 64, torch.bfloat16, MIXED, False),
    (12, 4, 96, torch.float16, MIXED, True), (12, 4, 96, torch.bfloat16, MIXED, False),
    (8, 2, 64, torch.float32, MIXED, False), (32, 8, 128, torch.float32, MIXED, False),
])
def test_whole_rows(cuda, sea, wl, hq, hkv, d, dtype, spec, scheduled):  # noqa: F811
    _lib, pak = sea_module("_lib"), sea_module("paged_attention_kernel")
    arr, code = _lib.i64_array, _lib.dtype_code(dtype)
    w = custom(wl, spec, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    kc, vc = cache.blocks(0)
    m = wl.metadata_tensors(w, cuda)
    plan = (None, 0, 0, 0, 0, 0)
    if scheduled:
        plan = pak._schedule(m, cuda, hq, hkv, d, 16, 0, True, code)
        assert plan[3] > 0 and plan[4] > 0  # merge units and partials
    sched, n_dec, n_pre, n_mrg, need, n_pfx = plan
    announce(f"no-alloc, off the scratch: Hq={hq} Hkv={hkv} D={d} {dtype} {len(spec)} rows, scheduled={scheduled}")
    o = torch.full_like(T.q, float("nan"))
    l = torch.full(T.q.shape[:2], float("nan"), device=cuda)
    _lib.check(_lib.load().kvhot_paged_attention_noalloc(
        T.q.data_ptr(), arr(T.q.stride()), kc.data_ptr(), arr(kc.stride()), vc.data_ptr(), arr(vc.stride()),
        o.data_ptr(), arr(o.stride()), l.data_ptr(), arr(l.stride()), m["block_table"].data_ptr(),
        m["block_table_row_stride"], m["q_lens"].data_ptr(), m["k_lens"].data_ptr(), m["q_starts"].data_ptr(),
        m["q_pos_offsets"].data_ptr(), len(w.rows), T.q.shape[0], m["max_q_len"], m["max_k_len"], hq, hkv, d, 16,
        kc.shape[0], 1.0 / math.sqrt(d), 1, code, 0, sched.data_ptr() if scheduled else None, n_dec, n_pre, n_mrg,
        n_pfx, need, _lib.stream_handle(cuda)), "kvhot_paged_attention_noalloc")
    torch.cuda.synchronize()
    assert_attention(w, o, l, ref_o, ref_l)
