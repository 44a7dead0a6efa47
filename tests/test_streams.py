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
