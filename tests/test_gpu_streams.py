"""What one call keeps for later ones -- the step's launch list, the stream's
workspace -- under other streams and under graph capture."""
import math

import pytest
import torch

from conftest import sea_module
from parity import custom
from test_gpu_parity import announce, assert_attention, oracle_step, wl  # noqa: F401  (wl: fixture)

pytestmark = pytest.mark.gpu

ROWS = [(1, 900, 899), (1, 3000, 2999), (40, 2500, 2460), (1, 17, 16)]
SHAPES = [(32, 8, 128, torch.bfloat16), (24, 8, 128, torch.bfloat16), (8, 2, 64, torch.float32)]


def prepare(sea, wl, hq, hkv, d, dtype, cuda):  # noqa: F811
    w = custom(wl, ROWS, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda)
    ref = oracle_step(w, T)
    cache = sea._PagedKVCache(T.kv_cache)
    cache.write(T.new_k, T.new_v, 0, T.slot_mapping)
    kc, vc = cache.blocks(0)
    meta = wl.metadata_tensors(w, cuda)

    def call():
        return sea.paged_flash_attention(T.q, kc, vc, meta, hq, hkv, 1.0 / math.sqrt(d))

    torch.cuda.synchronize()
    return w, ref, meta, call


@pytest.mark.parametrize("hq,hkv,d,dtype", SHAPES)
def test_a_list_on_other_streams(cuda, sea, wl, hq, hkv, d, dtype):  # noqa: F811
    """A stream's first call waits for the list's copy, which the step's first
    call queued on its own stream; later ones run natively."""
    lib = sea_module("_lib")
    w, ref, meta, call = prepare(sea, wl, hq, hkv, d, dtype, cuda)
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = []
    for s in streams * 2:
        announce(f"one list, several streams Hq={hq} Hkv={hkv} D={d} {dtype}")
        with torch.cuda.stream(s):
            outs.append(call())
    torch.cuda.synchronize()
    for o, l in outs:
        assert_attention(w, o, l, *ref)
    if dtype is not torch.float32:
        ((event, ordered),) = meta["_schedule_streams"].values()
        assert ordered == {s.cuda_stream for s in streams}
    taken = []
    native = lib.native()

    class _Native:
        def attention(self, *args):
            taken.append(native.attention(*args))
            return taken[-1]

    for s, ordered in ((streams[1], True), (torch.cuda.Stream(), False)):
        lib._NATIVE = _Native()
        try:
            with torch.cuda.stream(s):
                o, l = call()
        finally:
            lib._NATIVE = native
        torch.cuda.synchronize()
        assert_attention(w, o, l, *ref)
        assert (taken[-1] is not None) == ordered


@pytest.mark.parametrize("hq,hkv,d,dtype", SHAPES)
@pytest.mark.parametrize("listed", [False, True])
def test_captured_calls(cuda, sea, wl, hq, hkv, d, dtype, listed):  # noqa: F811
    """A step's first call inside a capture, and one after its list was built:
    every replay, with eager work in between, gives the eager result, and the
    graph's workspace is its own."""
    pak = sea_module("paged_attention_kernel")
    w, ref, meta, call = prepare(sea, wl, hq, hkv, d, dtype, cuda)
    if listed:
        call()
        torch.cuda.synchronize()
    kept = dict(pak._WORKSPACES)
    graphs = []
    for _ in range(2):
        announce(f"captured call Hq={hq} Hkv={hkv} D={d} {dtype}, list there {listed}")
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = call()
        graphs.append((g, out))
    assert {k: v.data_ptr() for k, v in pak._WORKSPACES.items()} == {k: v.data_ptr() for k, v in kept.items()}
    assert bool(meta.get("_schedules")) == listed
    for rep in range(3):
        for g, (o, l) in graphs:
            o.fill_(float("nan"))
            l.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            announce(f"  replay {rep}")
            assert_attention(w, o, l, *ref)
        junk = [torch.full((1 << 20,), 1e30, device=cuda) for _ in range(4)]
        if rep:
            assert_attention(w, *call(), *ref)
        del junk
