"""Infinite and NaN keys and values, fp32 and split-probability shapes: they
reach the queries that see them and no other, as key-by-key attention in fp64
has it.  Decode rows (one key with probability 1 among them), prefill rows with
the value between their own queries, prefill units cut by keys, a shared
prefix; from launch lists and from the grid, causal and not."""
import math

import numpy as np
import pytest
import torch

from parity import REL_L2, custom, shared_custom
from test_gpu_parity import announce, f32, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")
# rows, shared blocks, and (row, key, K or V, kv head, head_dim, value)
CASES = {
    "decode": ([(1, 1, 0), (1, 300, 299), (1, 300, 299), (1, 40, 39)], [],
               [(0, 0, "v", 0, 3, INF), (1, 5, "v", 1, 0, -INF), (1, 290, "v", 0, 9, INF), (2, 17, "v", 0, 1, NAN),
                (3, 33, "k", 1, 2, NAN)]),
    "prefill": ([(40, 100, 60), (33, 33, 0), (70, 70, 0), (40, 100, 60)], [],
                [(0, 80, "v", 0, 3, INF), (0, 3, "v", 1, 4, -INF), (1, 32, "v", 1, 5, NAN), (2, 40, "k", 0, 6, NAN),
                 (3, 99, "v", 0, 7, INF)]),
    "mixed": ([(1, 500, 499), (40, 100, 60), (2, 2, 0)], [],
              [(0, 77, "v", 1, 3, INF), (1, 80, "v", 0, 3, -INF), (2, 1, "v", 0, 3, NAN)]),
    "cut": ([(40, 2500, 2460)], [], [(0, 100, "v", 0, 3, INF), (0, 2475, "v", 1, 4, NAN), (0, 2490, "v", 0, 5, -INF)]),
    "prefix": ([(1, 700 + i, 699 + i) for i in range(6)], [(0, 6, 40)],
               [(0, 100, "v", 0, 3, INF), (0, 690, "v", 1, 4, NAN), (3, 650, "v", 1, 5, -INF)]),
}


def reference(w, T, causal):
    """fp64 attention of every query over the keys it sees, and no others."""
    q_lens, k_lens, q_starts, offs, bt = w.arrays()
    q, g, d = f32(T.q).astype(np.float64), w.num_q_heads // w.num_kv_heads, w.head_dim
    kc, vc = f32(T.kv_cache[0, 0]).astype(np.float64), f32(T.kv_cache[0, 1]).astype(np.float64)
    out = np.zeros(q.shape)
    with np.errstate(all="ignore"):
        for r in range(len(w.rows)):
            for i in range(q_lens[r]):
                m = min(k_lens[r], offs[r] + i + 1) if causal else k_lens[r]
                j = np.arange(m)
                k, v = kc[bt[r, j // 16], j % 16], vc[bt[r, j // 16], j % 16]  # [m, Hkv, D]
                s = np.einsum("hgd,mhd->hgm", q[q_starts[r] + i].reshape(-1, g, d), k) / math.sqrt(d)
                p = np.exp(s - s.max(-1, keepdims=True))
                p /= p.sum(-1, keepdims=True)
                out[q_starts[r] + i] = (p[..., None] * v.transpose(1, 0, 2)[:, None]).sum(2).reshape(-1, d)
    return out


@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (8, 2, 64, torch.float32), (4, 2, 128, torch.float32), (8, 2, 96, torch.float32), (4, 2, 256, torch.float32),
    (6, 2, 128, torch.bfloat16), (12, 2, 64, torch.float16), (8, 2, 96, torch.bfloat16), (10, 2, 256, torch.float16),
])
@pytest.mark.parametrize("name", list(CASES))
def test_reaches_the_queries_that_see_it(cuda, sea, wl, hq, hkv, d, dtype, name):  # noqa: F811
    spec, share, bad = CASES[name]
    w = shared_custom(wl, spec, share, hq, hkv, d, dtype) if share else custom(wl, spec, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    for r, key, kv, h, dim, x in bad:
        T.kv_cache[0, "kv".index(kv), int(w.rows[r].block_table[key // 16]), key % 16, h, dim] = x
    kc, vc = cache.blocks(0)
    listed = wl.metadata_tensors(w, cuda)
    for causal in (True, False):
        ref = reference(w, T, causal)
        for meta in (listed, {k: v for k, v in listed.items() if not k.startswith("host_")}):
            announce(f"non-finite {name} Hq={hq} Hkv={hkv} D={d} {dtype} causal={causal} {'list' if meta is listed else 'grid'}")
            o, _ = sea.paged_flash_attention(T.q, kc, vc, meta, hq, hkv, 1.0 / math.sqrt(d), is_causal=causal)
            o = f32(o).astype(np.float64)
            assert np.array_equal(np.isnan(o), np.isnan(ref))
            assert np.array_equal(np.where(np.isinf(o), o, 0), np.where(np.isinf(ref), ref, 0))
            fin = np.isfinite(ref)
            err = np.linalg.norm(np.where(fin, o, 0) - np.where(fin, ref, 0), axis=-1)
            assert (err <= REL_L2[dtype] * np.linalg.norm(np.where(fin, ref, 0), axis=-1) + 1e-7).all()
