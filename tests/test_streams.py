"""Streams of the torch-tensor calls: which handles are taken, and which
stream's allocator pool the call's own tensors come from (host logic only:
the launch, torch's streams and its allocator are stand-ins)."""
import contextlib
import ctypes

import pytest
import torch

import fmha_native_amd as fmha

CURRENT = 0x111000


class _Stream:
    def __init__(self, handle, external=False):
        self.cuda_stream, self.external = handle, external

    @property
    def _as_parameter_(self):  # as torch.cuda.Stream: what ctypes passes
        return ctypes.c_void_p(self.cuda_stream)


class _Tensor:
    """What the calls read of a device tensor; notes its pool and recorded streams."""
    is_cuda, device, dtype = True, torch.device("cpu"), torch.bfloat16

    def __init__(self, shape, pool):
        self.shape, self.pool, self.recorded = torch.Size(shape), pool, []

    def record_stream(self, s):
        self.recorded.append(s.cuda_stream)

    def data_ptr(self):
        return 1 << 20


class World:
    """The stand-ins: `made` holds every tensor allocated, `launches` every launch."""

    def __init__(self, monkeypatch, current=CURRENT, need=4096):
        self.stack, self.made, self.launches = [current], [], []

        @contextlib.contextmanager
        def use(s):
            self.stack.append(s.cuda_stream)
            yield
            self.stack.pop()

        def external(ptr, device=None):
            assert isinstance(ptr, int) and ptr != 0  # torch takes an int, and 0 for a stream of its own pool
            return _Stream(ptr, external=True)

        def empty(shape, **kw):
            t = _Tensor((shape,) if isinstance(shape, int) else shape, self.stack[-1])
            self.made.append(t)
            return t

        monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: _Stream(self.stack[-1]))
        monkeypatch.setattr(torch.cuda, "default_stream", lambda device=None: _Stream(0))
        monkeypatch.setattr(torch.cuda, "ExternalStream", external)
        monkeypatch.setattr(torch.cuda, "stream", use)
        monkeypatch.setattr(torch, "empty", empty)
        monkeypatch.setattr(fmha, "params_from_tensors", lambda *a: None)
        monkeypatch.setattr(fmha, "workspace_size", lambda p, b, c: need)
        launch = lambda stream: self.launches.append(ctypes.c_void_p.from_param(stream) and stream)
        monkeypatch.setattr(fmha, "fmha_fwd_d64_bf16", lambda p, b, c, stream: launch(stream))
        monkeypatch.setattr(fmha, "fmha_fwd_d64_bf16_ws", lambda p, b, c, ws, n, stream: launch(stream))

    def tensor(self, *shape):
        return _Tensor(shape, CURRENT)


@pytest.mark.parametrize("need", [0, 4096])
@pytest.mark.parametrize("stream,handle", [
    (None, CURRENT), (CURRENT, CURRENT), (0x222000, 0x222000), (ctypes.c_void_p(0x222000), 0x222000),
    (_Stream(0x222000), 0x222000), (0, 0), (ctypes.c_void_p(None), 0)])
def test_fmha_fwd_takes_every_form_of_stream(monkeypatch, stream, handle, need):
    """An int, a ctypes pointer or a torch stream, the null stream among them,
    whether or not the launch has a workspace."""
    w = World(monkeypatch, need=need)
    fmha.fmha_fwd(w.tensor(1, 2, 8, 64), w.tensor(1, 2, 9, 64), w.tensor(1, 2, 9, 64), stream=stream)
    (got,) = w.launches
    got = getattr(got, "_as_parameter_", got)
    assert (getattr(got, "value", got) or 0) == handle


@pytest.mark.parametrize("need", [0, 4096])
@pytest.mark.parametrize("stream", [0x222000, 0, _Stream(0x222000)])
def test_fmha_fwd_allocates_on_the_launch_stream(monkeypatch, stream, need):
    """O, LSE and the workspace come from the launch stream's pool, so that no
    block of the current stream's still in use there is written; the outputs
    are recorded for the current stream and the inputs for the launch's, so
    that neither is handed out again while the other stream uses it."""
    w = World(monkeypatch, need=need)
    handle = fmha._stream_handle(stream)
    q, k, v = w.tensor(1, 2, 8, 64), w.tensor(1, 2, 9, 64), w.tensor(1, 2, 9, 64)
    o, lse = fmha.fmha_fwd(q, k, v, return_lse=True, stream=stream)
    assert w.launches == [handle] and len(w.made) == (3 if need else 2)
    assert all(t.pool == handle for t in w.made)
    assert o.recorded == lse.recorded == [CURRENT]
    assert all(t.recorded == [handle] for t in (q, k, v))
    assert w.stack == [CURRENT]


@pytest.mark.parametrize("stream", [None, CURRENT])
def test_fmha_fwd_on_the_current_stream_records_nothing(monkeypatch, stream):
    w = World(monkeypatch)
    q, k, v = w.tensor(1, 2, 8, 64), w.tensor(1, 2, 9, 64), w.tensor(1, 2, 9, 64)
    fmha.fmha_fwd(q, k, v, return_lse=True, stream=stream)
    assert [t.pool for t in w.made] == [CURRENT] * 3
    assert not any(t.recorded for t in w.made + [q, k, v])


@pytest.mark.parametrize("given", [False, True])
def test_merge_allocates_on_the_launch_stream(monkeypatch, given):
    w = World(monkeypatch)
    monkeypatch.setattr(fmha, "fmha_merge_d64_bf16", lambda *a: w.launches.append(a[-1]))

    class Parts(_Tensor):
        def __init__(self, shape, dtype):
            super().__init__(shape, CURRENT)
            self.dtype = dtype

        dim = lambda self: len(self.shape)
        is_contiguous = lambda self: True
        __getitem__ = lambda self, i: Parts(self.shape[1:], self.dtype)
        numel = lambda self: self.shape.numel()

    o_parts, l_parts = Parts((2, 8, 64), torch.bfloat16), Parts((2, 8), torch.float32)
    out = (Parts((8, 64), torch.bfloat16), Parts((8,), torch.float32)) if given else (None, None)
    o, lse = fmha.merge_partials(o_parts, l_parts, *out, stream=0x222000)
    assert w.launches == [0x222000] and all(t.pool == 0x222000 for t in w.made)
    assert o.recorded == lse.recorded == [0x222000 if given else CURRENT]
    assert o_parts.recorded == l_parts.recorded == [0x222000]


@pytest.mark.gpu
def test_a_block_still_in_use_is_not_the_side_streams_workspace(monkeypatch):
    """Work pending on the current stream uses a block that was just freed; a
    call on another stream gets other memory for O, LSE and the workspace.
    The launch is replaced by a recorder, so nothing is written."""
    q = torch.zeros(2, 16, 1, 64, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(2, 4, 9000, 64, device="cuda", dtype=torch.bfloat16)
    need = fmha.workspace_size(fmha.params_from_tensors(q, k, k, torch.empty_like(q)), 2, 1)
    assert need > 0
    seen = []
    monkeypatch.setattr(fmha, "fmha_fwd_d64_bf16_ws", lambda p, b, c, ws, n, stream: seen.append((ws, n, stream)))
    side = torch.cuda.Stream()
    blocks = [torch.empty(need, dtype=torch.uint8, device="cuda"), torch.empty_like(q),
              torch.empty(q.shape[:-1], device="cuda")]
    spans = [(t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in blocks]
    torch.cuda.synchronize()
    torch.cuda._sleep(200_000_000)  # ~0.1 s of bounded work
    del blocks
    o, lse = fmha.fmha_fwd(q, k, k, causal=True, return_lse=True, stream=side)
    busy = not torch.cuda.current_stream().query()
    (ws, size, stream), = seen
    assert busy and (size, stream) == (need, side.cuda_stream)
    mine = [(ws, ws + need)] + [(t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in (o, lse)]
    assert not any(a < d and c < b for a, b in spans for c, d in mine)
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_fmha_fwd_on_a_side_stream_matches_the_current_one():
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(2, 16, 1, 64), rnd(2, 4, 9000, 64), rnd(2, 4, 9000, 64)
    want = fmha.fmha_fwd(q, k, v, causal=True, return_lse=True)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for stream in (side, side.cuda_stream, ctypes.c_void_p(side.cuda_stream)):
        got = fmha.fmha_fwd(q, k, v, causal=True, return_lse=True, stream=stream)
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with torch.cuda.stream(side):  # the null stream beside another current one
        got = fmha.fmha_fwd(q, k, v, causal=True, return_lse=True, stream=0)
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
