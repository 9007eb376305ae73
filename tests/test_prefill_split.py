"""Prefill units cut by keys: the launch list covers every query block's keys
once (CPU), and the kernels' results against the fp64 oracle (GPU)."""
import pytest
import torch

from parity import custom
from test_abi import _schedule, lib  # noqa: F401  (lib: fixture)
from test_gpu_parity import announce, assert_attention, hip_step, oracle_step, wl  # noqa: F401  (wl: fixture)

KEYS = 32  # keys per prefill tile


@pytest.mark.parametrize("hq,hkv,d,rows,cut", [
    (32, 8, 128, [(225, 1249, 1024), (1, 900, 899)], True),
    (32, 8, 128, [(64, 16448, 16384), (2, 40, 38), (700, 700, 0)], True),
    (8, 8, 128, [(200, 4200, 4000)], True),
    (16, 4, 256, [(300, 4300, 4000)], True),
    (12, 12, 64, [(3, 8195, 8192)], True),
    (8, 2, 64, [(33, 2000, 1000)], True),      # keys past the last query are masked
    (32, 8, 128, [(201, 501, 300)], False),    # no unit much longer than the smallest part
    (32, 8, 128, [(4096, 4096, 0)], False),    # fills the device
])
def test_units_cover_every_block(lib, hq, hkv, d, rows, cut):  # noqa: F811
    ql, kl, off = (list(x) for x in zip(*rows))
    _, pre, merge, ws, qs = _schedule(lib, ql, kl, off, hq=hq, hkv=hkv, d=d)
    g = hq // hkv
    nm, waves = {64: (4, 4), 128: (2, 4), 256: (1, 8)}[d]
    qpw = waves * (16 * nm // g)
    ranges, partial = {}, {}
    for row, h, qb, tiles, k0, parts, base, k1 in pre.tolist():
        nq = min(qpw, ql[row] - qb * qpw)
        end = min(kl[row], off[row] + qb * qpw + nq)
        assert k0 % KEYS == 0 and parts <= 0 and (parts < 0 or (k0, base, k1) == (0, 0, 0))
        stop = min(k1, end) if parts < 0 else end
        assert tiles == -(-(stop - k0) // KEYS)
        ranges.setdefault((row, h, qb), []).append((k0, stop))
        for i in range(nq if parts < 0 else 0):
            assert base - parts * i not in partial
            partial[base - parts * i] = (int(qs[row]) + qb * qpw + i, h, -parts)
    for (row, h, qb), r in ranges.items():
        r.sort()
        nq = min(qpw, ql[row] - qb * qpw)
        assert r[0][0] == 0 and r[-1][1] == min(kl[row], off[row] + qb * qpw + nq)
        assert all(a[1] == b[0] for a, b in zip(r, r[1:]))
    assert len(ranges) == sum(hkv * -(-q // qpw) for q in ql if q > 1)
    assert list(pre[:, 3]) == sorted(pre[:, 3], reverse=True)
    # the merge units read exactly the partials the units write
    read = {}
    for t, h, parts, base, _, _, queries, _ in merge.tolist():
        for i in range(queries):
            for k in range(parts):
                read[base + parts * i + k] = (t + i, h, parts)
    assert read == partial and bool(partial) == cut
    assert ws <= 64 << 20 and (len(partial) == 0 or ws >= (max(partial) + 1) * g * (d + 1) * 4)


ROWS = [
    [(225, 1249, 1024), (1, 900, 899), (1, 3000, 2999)],  # a budgeted chunk beside decode rows, one of them cut
    [(2, 4100, 4098), (33, 2047, 2014), (130, 700, 570)],  # the fewest queries; one query into a second block
    [(40, 1500, 1000), (31, 1024, 993)],                   # keys past the last query; parts of whole blocks
]


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (32, 8, 128, torch.bfloat16), (12, 12, 64, torch.float16), (8, 2, 64, torch.bfloat16), (16, 4, 256, torch.bfloat16),
    (16, 1, 128, torch.float16), (24, 8, 128, torch.bfloat16), (12, 4, 96, torch.float16),
])
def test_cut_units(cuda, sea, wl, hq, hkv, d, dtype):  # noqa: F811
    for spec in ROWS:
        w = custom(wl, spec, hq, hkv, d, dtype)
        T = wl.make_tensors(w, cuda)
        ref_o, ref_l = oracle_step(w, T)
        announce(f"cut prefill units Hq={hq} Hkv={hkv} D={d} {dtype} rows {spec}")
        meta = wl.metadata_tensors(w, cuda)
        o, l = hip_step(sea, wl, w, T, meta=meta)
        assert_attention(w, o, l, ref_o, ref_l)
        plan = list(meta["_schedules"].values())[0]
        assert plan[3] > 0 and plan[4] > 0  # merge units and their partials
        o2, l2 = hip_step(sea, wl, w, T, meta=meta)
        q = [i for i, x in enumerate(w.rows) if x.q_len > 1]  # prefill rows: the same bits on every call
        starts = w.arrays()[2]
        for i in q:
            sl = slice(int(starts[i]), int(starts[i]) + w.rows[i].q_len)
            assert torch.equal(o[sl], o2[sl]) and torch.equal(l[sl], l2[sl])
