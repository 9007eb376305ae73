"""A step's launch list takes one run of the planner, or two where it is longer
than the list it was first given."""
import numpy as np
import pytest

from conftest import sea_module
from test_abi import _schedule, lib  # noqa: F401  (lib: fixture)


class _Counted:
    def __init__(self, mod):
        self.mod, self.runs = mod, 0

    def kvhot_paged_attention_schedule(self, *args):
        self.runs += 1
        return self.mod.kvhot_paged_attention_schedule(*args)


@pytest.mark.parametrize("rows,lo,hi,pt,runs", [(1, 1001, 1001, 0, 1), (4, 17, 130, 0, 1), (64, 128, 2048, 0, 1),
                                                (256, 64, 2048, 0, 1), (64, 8000, 9000, 32, 2)])
def test_runs_of_the_planner(lib, monkeypatch, rows, lo, hi, pt, runs):  # noqa: F811
    pak, _lib = sea_module("paged_attention_kernel"), sea_module("_lib")
    k = np.random.default_rng(rows).integers(lo, hi + 1, rows).astype(np.int32)
    q, qs, off = np.ones(rows, np.int32), np.arange(rows, dtype=np.int32), k - 1
    mb = int(-(-k.max() // 16))
    bt = (np.arange(rows * mb, dtype=np.int32) + 1000).reshape(rows, mb)
    counted = _Counted(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: counted)
    args = (q.ctypes.data, k.ctypes.data, qs.ctypes.data, off.ctypes.data, bt.ctypes.data, mb, rows, 32, 8, 128, 16, pt, 1, 2)
    units, (n_dec, n_pre, n_mrg, ws, n_pfx) = pak.plan_units(args, rows, int(k.max()), 8)
    assert counted.runs == runs
    dec, pre, merge, ws2, _ = _schedule(lib, q, k, off, pt=pt)
    assert (n_dec, n_pre, n_mrg, ws, n_pfx) == (len(dec), len(pre), len(merge), ws2, 0)
    assert len(units) == n_dec + n_pre + n_mrg and np.array_equal(units[n_dec + n_pre:], merge)


def test_the_graph_step_plans_once(lib, monkeypatch):  # noqa: F811
    graph, pak, _lib = sea_module("decode_graph"), sea_module("paged_attention_kernel"), sea_module("_lib")
    r, mb = 3, 70
    g = object.__new__(graph.DecodeStepGraph)
    g.r, g.max_blocks, g.shape = r, mb, (32, 8, 128, 16, 0, True, 2)
    a = np.zeros(4 * r + r * mb, np.int32)
    a[0:r], a[r:2 * r], a[2 * r:3 * r], a[3 * r:4 * r] = 1, [1000, 17, 300], range(r), [999, 16, 299]
    counted = _Counted(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: counted)
    monkeypatch.setattr(graph, "pinned_units", lambda units: units)
    units, counts = g._plan(a)
    assert counted.runs == 1 and len(units) == sum(counts[:3]) > 0
