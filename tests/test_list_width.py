"""A launch list says by its own decode unit count which work-groups it was
planned for: kvhot_paged_attention takes lists of 4 more than a multiple of 8
descriptors as groups of 4 (they share a launch with prefill units), others as
groups of 8, whatever partition_tokens it is passed."""
import numpy as np
import pytest

from test_abi import W, _check_decode_schedule, _schedule, lib  # noqa: F401  (lib: fixture)

MIXED_W = 4


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (12, 12, 64), (8, 1, 128), (24, 8, 128), (12, 4, 96), (16, 4, 256)])
@pytest.mark.parametrize("pt", [0, 32, 512])
def test_width_follows_from_the_unit_count(lib, hq, hkv, d, pt):  # noqa: F811
    g = hq // hkv
    if pt and (d == 96 or g & (g - 1)):
        pytest.skip("no lists with fixed partitions")
    rng = np.random.default_rng(hq + d + pt)
    for n in (1, 2, 3, 5, 8, 13, 30, 67):
        for chunks in ([], [(20, 30)], [(300, 0), (2, 4000)]):
            k = [int(x) for x in rng.integers(1, 40 << int(rng.integers(0, 7)), n)]
            ql, off = [1] * n + [c for c, _ in chunks], [x - 1 for x in k] + [p for _, p in chunks]
            kl = k + [c + p for c, p in chunks]
            dec, pre, merge, ws, qs = _schedule(lib, ql, kl, off, hq=hq, hkv=hkv, d=d, pt=pt)
            mixed = bool(chunks) and pt == 0 and d <= 128
            width = MIXED_W if len(dec) % W == MIXED_W else W
            assert len(dec) % width == 0 and width == (MIXED_W if mixed else W)
            merge = merge[merge[:, 6] == 0]  # (merge units of prefill units cut by keys apart)
            if mixed:
                ws = sum(int(x[2]) for x in merge) * g * (d + 1) * 4
            elif chunks:
                continue  # (workspace: the cut prefill units' partials too)
            _check_decode_schedule(dec, merge, ws, qs, width, dict(enumerate(k)), hkv, G=g, D=d, pt=pt)
