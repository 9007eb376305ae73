"""kvhot_torch, the native side of the per-layer calls, against the Python
functions that take the calls it leaves alone: the same bits over the forms it
takes, and nothing done or raised for the others."""
import pytest
import torch

from conftest import sea_module
from parity import custom
from test_gpu_parity import announce, wl  # noqa: F401  (wl: fixture)

ROWS = [(20, 50, 30), (2, 17, 15), (37, 300, 263), (16, 16, 0)]  # prefill: the same bits on every call


class _Nothing:
    """Stands in for kvhot_torch and takes no call."""

    def __init__(self):
        self.calls = 0

    def _none(self, *args):
        self.calls += 1

    attention = append = layer = _none


class _Counted:
    """kvhot_torch, with the calls it took counted."""

    def __init__(self, mod):
        self.mod, self.taken, self.names = mod, 0, []

    def __getattr__(self, name):
        def call(*args):
            self.names.append(name)
            r = getattr(self.mod, name)(*args)
            self.taken += r is not None
            return r
        return call


def test_cpu_calls_are_left_alone():
    lib = sea_module("_lib")
    n = lib.native()
    q, kv = torch.zeros(2, 4, 64), torch.zeros(1, 2, 3, 16, 2, 64)
    k = torch.zeros(1, 2, 2, 64)
    slots = torch.zeros(2, dtype=torch.int64)
    assert n.append(kv, 2, 64, k, k, 0, slots) is None
    assert n.attention(q, kv[0, 0], kv[0, 1], {}, 4, 2, 0.1, True, 0, 1, {}) is None
    assert n.layer(kv, 2, 64, k, k, 0, slots, torch.zeros(1, 4, 2, 64), {}, 0.1, 0, 1, {}) is None
    for f in (n.append, n.attention, n.layer):  # too few arguments, and objects that are no tensors
        assert f() is None and f(*[None] * 13) is None


@pytest.mark.parametrize("answer,writes", [(None, 1), (False, 0)])
def test_a_refused_layer_appends_once(monkeypatch, answer, writes):
    """layer() answers None before the append and False after it."""
    runner, lib = sea_module("model_runner"), sea_module("_lib")
    calls = []

    class _Native:
        def layer(self, *args):
            return answer

    def _attention(*args, **kw):
        calls.append("attention")
        raise RuntimeError("refused")

    monkeypatch.setattr(lib, "_NATIVE", _Native())
    monkeypatch.setattr(runner._PagedKVCache, "write", lambda self, *args: calls.append("write"))
    monkeypatch.setattr(runner, "paged_flash_attention", _attention)

    class _Module:
        layer_idx = 0

    cache = runner._PagedKVCache(torch.zeros(1, 2, 3, 16, 2, 64))
    k = torch.zeros(1, 2, 2, 64)
    with pytest.raises(RuntimeError, match="refused"):
        runner.hip_paged_attention_forward(_Module(), torch.zeros(1, 4, 2, 64), k, k, None, 0.1, cache=cache,
                                           write_index=torch.zeros(2, dtype=torch.int64), paged_metadata={})
    assert calls == ["write"] * writes + ["attention"]


@pytest.mark.gpu
def test_attention_refused_after_the_append(cuda, sea, wl, monkeypatch):  # noqa: F811
    """A query whose head_dim is not unit-stride, which the library refuses:
    the step's K/V are appended once, and the refusal is raised."""
    lib = sea_module("_lib")
    w = custom(wl, ROWS, 8, 2, 64, torch.bfloat16)
    T = wl.make_tensors(w, cuda)
    cache = sea._PagedKVCache(T.kv_cache)
    meta = wl.metadata_tensors(w, cuda)
    kc, vc = cache.blocks(0)
    sea.paged_flash_attention(T.q, kc, vc, meta, 8, 2, 0.125)  # builds the launch list and the workspace
    native = _Counted(lib.native())
    monkeypatch.setattr(lib, "_NATIVE", native)

    class _Module:
        layer_idx = 0

    announce("attention refused after the append (append launch only)")
    q4 = T.q.transpose(0, 1).unsqueeze(0)
    bad = torch.stack([q4, q4], -1)[..., 0]
    assert bad.stride(-1) == 2
    with pytest.raises(Exception, match="unit-stride"):
        sea.hip_paged_attention_forward(_Module(), bad, T.new_k, T.new_v, None, 0.125, cache=cache,
                                        write_index=T.slot_mapping, paged_metadata=meta)
    torch.cuda.synchronize()
    assert native.names == ["layer", "attention"]  # (no append of its own)
    got = T.kv_cache[0].reshape(2, -1, 2, 64)[:, T.slot_mapping.long()]
    assert torch.equal(got[0], T.new_k[0].transpose(0, 1)) and torch.equal(got[1], T.new_v[0].transpose(0, 1))


def _layer(sea, w, T, meta, q4, k4, v4, slots, scale):
    class _Module:
        layer_idx = 0

    kv = T.kv_cache.clone()
    cache = sea._PagedKVCache(kv)
    o, none = sea.hip_paged_attention_forward(_Module(), q4, k4, v4, None, scale, cache=cache, write_index=slots,
                                              paged_metadata=meta)
    assert none is None
    kc, vc = cache.blocks(0)
    o2, l2 = sea.paged_flash_attention(q4.transpose(1, 2).squeeze(0), kc, vc, meta, w.num_q_heads, w.num_kv_heads, scale)
    return o, kv, o2, l2


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (32, 8, 128, torch.bfloat16), (12, 12, 64, torch.float32), (24, 8, 128, torch.float16), (16, 4, 96, torch.bfloat16),
])
@pytest.mark.parametrize("layout", ["kv-interleaved", "head-major", "token-major"])
def test_same_bits(cuda, sea, wl, hq, hkv, d, dtype, layout, monkeypatch):  # noqa: F811
    lib = sea_module("_lib")
    w = custom(wl, ROWS, hq, hkv, d, dtype)
    T = wl.make_tensors(w, cuda, layout=layout)
    t = T.q.shape[0]
    wide = torch.randn(1, hq + 3, t, 2 * d, device=cuda).to(dtype)  # a projection's rows with others between them
    queries = {"token-major": T.q.transpose(0, 1).unsqueeze(0), "heads apart": T.q.transpose(0, 1).unsqueeze(0).contiguous(),
               "strided": wide[:, 1:hq + 1, :, d:]}
    for name, q4 in queries.items():
        for sl in (T.slot_mapping, T.slot_mapping.int(), torch.stack([T.slot_mapping] * 2, 1)[:, 0]):
            announce(f"native call Hq={hq} Hkv={hkv} D={d} {dtype} {layout} q {name} slots {sl.dtype} {sl.stride()}")
            outs = []
            for native in (_Nothing(), _Counted(lib.native())):
                monkeypatch.setattr(lib, "_NATIVE", native)
                meta = wl.metadata_tensors(w, cuda)
                for _ in range(2):  # the first call builds the launch list
                    out = _layer(sea, w, T, meta, q4, T.new_k, T.new_v, sl, 1.0 / d ** 0.5)
                outs.append(out)
                monkeypatch.undo()
            torch.cuda.synchronize()
            assert native.taken >= (3 if sl.is_contiguous() else 2)
            for x, y in zip(*outs):
                assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype
                assert torch.equal(x, y)


@pytest.mark.gpu
def test_single_token_and_no_host_copies(cuda, sea, wl, monkeypatch):  # noqa: F811
    """One decode row (deterministic), with and without the metadata's host copies."""
    lib = sea_module("_lib")
    w = custom(wl, [(1, 77, 76)], 32, 8, 128, torch.bfloat16)
    T = wl.make_tensors(w, cuda)
    kc, vc = sea._PagedKVCache(T.kv_cache).blocks(0)
    outs = []
    for host in (True, False):
        for native in (_Nothing(), _Counted(lib.native())):
            monkeypatch.setattr(lib, "_NATIVE", native)
            meta = wl.metadata_tensors(w, cuda)
            if not host:
                meta = {k: v for k, v in meta.items() if not k.startswith("host_")}
            announce(f"native single token, host copies {host}")
            for _ in range(2):
                o, l = sea.paged_flash_attention(T.q, kc, vc, meta, 32, 8, 0.125, deterministic=True)
            torch.cuda.synchronize()
            outs.append((o, l))
            monkeypatch.undo()
        assert native.taken > 0
        assert all(torch.equal(x, y) for x, y in zip(*outs[-2:]))


@pytest.mark.gpu
def test_refused_calls_raise_as_before(cuda, sea, wl):  # noqa: F811
    w = custom(wl, ROWS, 8, 2, 64, torch.bfloat16)
    T = wl.make_tensors(w, cuda)
    cache = sea._PagedKVCache(T.kv_cache)
    kc, vc = cache.blocks(0)
    meta = wl.metadata_tensors(w, cuda)
    sea.paged_flash_attention(T.q, kc, vc, meta, 8, 2, 0.125)
    announce("refused calls (no launch)")

    def attention(q=T.q, k=kc, v=vc, m=meta, hq=8, hkv=2):
        sea.paged_flash_attention(q, k, v, m, hq, hkv, 0.125)

    for exc, kw in ((TypeError, dict(q=T.q.half())), (ValueError, dict(q=T.q[0])), (ValueError, dict(hq=4)),
                    (ValueError, dict(hkv=3)), (ValueError, dict(k=kc[:, :, :1])), (ValueError, dict(q=T.q.cpu())),
                    (TypeError, dict(m={**meta, "q_lens": meta["q_lens"].long()})),
                    (ValueError, dict(m={**meta, "k_lens": meta["k_lens"][:-1]})),
                    (ValueError, dict(m={**meta, "block_table": meta["block_table"].cpu()})),
                    (KeyError, dict(m={k: v for k, v in meta.items() if k != "q_starts"}))):
        with pytest.raises(exc):
            attention(**kw)
    k, s = T.new_k, T.slot_mapping
    for exc, args in ((ValueError, (k[0], T.new_v, 0, s)), (ValueError, (k[:, :1], T.new_v[:, :1], 0, s)),
                      (TypeError, (k.half(), T.new_v, 0, s)), (ValueError, (k, T.new_v, 0, s[:-1])),
                      (TypeError, (k, T.new_v, 0, s.float())), (ValueError, (k, T.new_v, 0, s.cpu())),
                      (IndexError, (k, T.new_v, 1, s)), (IndexError, (k, T.new_v, -1, s))):
        with pytest.raises(exc):
            cache.write(*args)
