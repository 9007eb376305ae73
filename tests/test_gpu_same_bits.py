"""fp32 calls, and 16-bit calls whose query groups are not a power of two or
whose head_dim is 96, give the same bits on every call without
deterministic=True: decode rows of one and of several work-groups, beside
prefill rows, behind a shared prefix, from launch lists and from the grid."""
import pytest
import torch

from parity import custom, shared_custom
from test_gpu_parity import announce, hip_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

DECODE = [(1, 90 + 137 * i, 89 + 137 * i) for i in range(16)]


@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (12, 12, 64, torch.float32), (32, 8, 128, torch.float32), (12, 4, 96, torch.float32), (16, 4, 256, torch.float32),
    (24, 8, 128, torch.bfloat16), (12, 4, 96, torch.float16), (10, 2, 64, torch.bfloat16), (6, 2, 256, torch.bfloat16),
])
def test_every_call_gives_the_same_bits(cuda, sea, wl, hq, hkv, d, dtype):  # noqa: F811
    for name, w in (
            ("decode", custom(wl, DECODE, hq, hkv, d, dtype)),
            ("one long row", custom(wl, [(1, 9000, 8999)], hq, hkv, d, dtype)),
            ("mixed", custom(wl, DECODE + [(40, 700, 660), (3, 3, 0)], hq, hkv, d, dtype)),
            ("shared prefix", shared_custom(wl, [(1, 700 + i, 699 + i) for i in range(9)], [(0, 9, 40)], hq, hkv, d, dtype))):
        T = wl.make_tensors(w, cuda)
        listed = wl.metadata_tensors(w, cuda)
        for meta in (listed, {k: v for k, v in listed.items() if not k.startswith("host_")}):
            announce(f"same bits: {name} Hq={hq} Hkv={hkv} D={d} {dtype} {'list' if meta is listed else 'grid'}")
            o, l = hip_step(sea, wl, w, T, meta=meta)
            for _ in range(6):
                o2, l2 = hip_step(sea, wl, w, T, meta=meta)
                assert torch.equal(o, o2) and torch.equal(l, l2)
