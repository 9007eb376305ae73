"""Prefill units and decode work-groups of one launch, against the fp64 oracle:
up to a turn of 256 of either and more, the smallest of both.  (Whole turns at
every shape: test_gpu_new_plans.py.)"""
import math

import pytest
import torch

from parity import custom
from test_gpu_parity import announce, assert_attention, hip_step, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

SPECS = {
    # about a turn of both kinds where there are 8 kv heads, less or more elsewhere
    "turns": [(1, 90 + 61 * (i % 17), 89 + 61 * (i % 17)) for i in range(40)] + [(300, 400, 100), (513, 513, 0), (270, 300, 30)],
    # slices, ranges and blocks around their edges; a decode row without a key
    "edges": [(1, 1, 0), (1, 16, 15), (2, 2, 0), (1, 17, 16), (0, 5, 5), (1, 129, 128), (33, 65, 32), (1, 1030, 1029),
              (1, 0, -1)],
    "smallest": [(1, 1, 0), (2, 2, 0)],
    # one long row, cut over many work-groups and merged, beside cut prefill units
    "long": [(1, 5000, 4999), (40, 2500, 2460)],
}


@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (32, 8, 128, torch.bfloat16), (16, 1, 128, torch.float16), (8, 8, 128, torch.bfloat16), (16, 2, 64, torch.bfloat16),
    (12, 12, 64, torch.float16), (24, 8, 128, torch.bfloat16), (12, 4, 96, torch.float16), (10, 2, 64, torch.bfloat16),
])
@pytest.mark.parametrize("spec", list(SPECS))
def test_mixed_launch(cuda, sea, wl, hq, hkv, d, dtype, spec):  # noqa: F811
    w = custom(wl, SPECS[spec], hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    rows = [i for i, x in enumerate(w.rows) if x.q_len > 0]
    announce(f"mixed launch {spec} Hq={hq} Hkv={hkv} D={d} {dtype}")
    meta = wl.metadata_tensors(w, cuda)
    o, l = hip_step(sea, wl, w, T, meta=meta)
    assert_attention(w, o, l, ref_o, ref_l, rows=rows)
    (_, n_dec, n_pre, _, _, n_pfx), = meta["_schedules"].values()
    assert n_dec % 8 == 4 and n_pre > n_pfx  # a list for one launch of both kinds
    kc, vc = sea._PagedKVCache(T.kv_cache).blocks(0)
    scale = 1.0 / math.sqrt(d)
    for kw in (dict(deterministic=True), dict(verify_block_table=True), dict(partition_tokens=64)):
        outs = [sea.paged_flash_attention(T.q, kc, vc, meta, hq, hkv, scale, **kw) for _ in range(2)]
        torch.cuda.synchronize()
        assert_attention(w, *outs[0], ref_o, ref_l, rows=rows)
        if "deterministic" in kw:
            starts = w.arrays()[2]
            for i in rows:
                sl = slice(int(starts[i]), int(starts[i]) + w.rows[i].q_len)
                assert torch.equal(outs[0][0][sl], outs[1][0][sl]) and torch.equal(outs[0][1][sl], outs[1][1][sl])
