"""Shared-prefix units beside prefill rows: as many as without them."""
import numpy as np
import pytest

from test_abi import GROUPS, _schedule, lib  # noqa: F401  (lib: fixture)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (64, 8, 128), (32, 8, 64), (24, 8, 128), (16, 4, 256)])
@pytest.mark.parametrize("rows,shared", [(64, 16384), (16, 32768), (64, 4096), (256, 1024), (5, 512)])
def test_prefix_units_do_not_depend_on_prefill_rows(lib, hq, hkv, d, rows, shared):  # noqa: F811
    k = [shared + 40 + 3 * i for i in range(rows)]
    nb = -(-max(k) // 16)
    count = []
    for chunks in ([], [(64, 0)], [(225, 1024)], [(512, 500)] * 8):
        ql, kl = [1] * rows + [c for c, _ in chunks], k + [c + p for c, p in chunks]
        off = [x - 1 for x in k] + [p for _, p in chunks]
        bt = np.arange(len(ql) * nb, dtype=np.int32).reshape(-1, nb)
        bt[:rows, :shared // 16] = bt[0, :shared // 16]
        *_, npx = _schedule(lib, ql, kl, off, hq=hq, hkv=hkv, d=d, bt=bt, prefix=True)
        count.append(npx)
    assert len(set(count)) == 1
    queries = {64: 4 * (64 * hkv // hq), 128: 4 * (32 * hkv // hq), 256: 8 * (16 * hkv // hq)}[d]  # of a prefix unit
    assert 0 < count[0] <= 2 * GROUPS + -(-rows // queries) * hkv
