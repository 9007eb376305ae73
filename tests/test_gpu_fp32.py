"""fp32 attention on the fp32 MFMA kernels (every head_dim they take, query
groups of 1 to 16 heads) against the fp64 oracle, within the fp32 bounds of
tests/parity.py (1e-5)."""
import pytest
import torch

from parity import custom
from test_gpu_parity import announce, assert_attention, hip_step, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

# Decode rows around one slice, a wave's slices and a partition; prefill rows
# around a work-group's 16 / G queries, one slice for each of 4 waves (64
# keys) and two (128).
ROWS = [(1, 17, 16), (20, 50, 30), (1, 1, 0), (0, 16, 16), (2, 2, 0), (1, 512, 511), (41, 41, 0), (1, 1025, 1024),
        (9, 300, 291), (16, 64, 48), (17, 65, 48), (1, 2100, 2099), (130, 257, 127), (1, 128, 127), (5, 133, 128)]


@pytest.mark.parametrize("hq,hkv,d", [
    (12, 12, 64), (8, 2, 64), (16, 1, 64), (12, 4, 96), (32, 2, 96), (4, 4, 96), (32, 8, 128), (7, 1, 128),
    (24, 8, 128), (32, 2, 128), (16, 4, 256), (2, 2, 256), (32, 2, 256), (33, 3, 256),
])
@pytest.mark.parametrize("layout", ["kv-interleaved", "token-major"])
def test_fp32_shapes(cuda, sea, wl, hq, hkv, d, layout):  # noqa: F811
    w = custom(wl, ROWS, hq, hkv, d, torch.float32)
    T = wl.make_tensors(w, cuda, layout=layout)
    ref_o, ref_l = oracle_step(w, T)
    for pt in (None, 64):
        announce(f"fp32 Hq={hq} Hkv={hkv} D={d} {layout} partition {pt}")
        o, l = hip_step(sea, wl, w, T, partition_tokens=pt)
        assert_attention(w, o, l, ref_o, ref_l, rows=[i for i, x in enumerate(w.rows) if x.q_len > 0])


def test_fp32_keys_past_the_end_are_not_read(cuda, sea, wl):  # noqa: F811
    """NaN in the cache's unused token slots does not reach an output."""
    w = custom(wl, [(1, 17, 16), (5, 40, 35), (1, 130, 129), (33, 70, 37)], 8, 2, 64, torch.float32)
    T = wl.make_tensors(w, cuda)
    ref_o, ref_l = oracle_step(w, T)
    used = torch.zeros(w.num_blocks, 16, dtype=torch.bool, device=cuda)
    for x in w.rows:
        for j in range(x.k_len):
            used[int(x.block_table[j // 16]), j % 16] = True
    T.kv_cache[0].masked_fill_(~used[None, :, :, None, None], float("nan"))
    announce("fp32 NaN past the keys")
    o, l = hip_step(sea, wl, w, T)
    assert_attention(w, o, l, ref_o, ref_l)
