"""Pools whose tokens lie further apart than their blocks ([block_size,
num_blocks, Hkv, D] in memory), against the fp64 oracle: the kernels that
address a block by one descriptor of its stride do not take them."""
import math

import pytest
import torch

from parity import custom
from test_gpu_parity import announce, assert_attention, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

ROWS = [(1, 17, 16), (20, 50, 30), (1, 300, 299), (3, 3, 0)]


@pytest.mark.parametrize("hq,hkv,d,dtype", [(8, 2, 64, torch.float32), (24, 8, 128, torch.bfloat16),
                                            (12, 4, 96, torch.float16), (32, 8, 128, torch.bfloat16)])
@pytest.mark.parametrize("outer", ["token, block, head", "token, head, block", "head, block, token"])
def test_token_strides_above_the_block_stride(cuda, sea, wl, hq, hkv, d, dtype, outer):  # noqa: F811
    w = custom(wl, ROWS, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    order = [("block", "token", "head").index(x) for x in outer.split(", ")] + [3]
    back = [order.index(i) for i in range(4)]
    kc, vc = (x.permute(order).contiguous().permute(back) for x in cache.blocks(0))
    announce(f"pool in {outer} order, Hq={hq} Hkv={hkv} D={d} {dtype}")
    for _ in range(2):
        o, l = sea.paged_flash_attention(T.q, kc, vc, wl.metadata_tensors(w, cuda), hq, hkv, 1.0 / math.sqrt(d))
        torch.cuda.synchronize()
        assert_attention(w, o, l, ref_o, ref_l)
