"""Where sw.sddmm's scratch memory comes from, on a stand-in for torch.cuda (two
devices, which no test machine here has): the memory is taken on the stream
that the kernel runs on, or not at all."""
import contextlib
import ctypes
import types

import pytest

import sparsewavecomp_amd as sw


class _Stream:
    def __init__(self, device):
        self.device = device


def _fake_torch(capturing=False):
    state = types.SimpleNamespace(device=0, streams={0: "s0", 1: "s1"},
                                  taken=[], mode=0)

    @contextlib.contextmanager
    def stream(s):
        device, old = state.device, state.streams[s.device]
        state.device, state.streams[s.device] = s.device, s
        try:
            yield
        finally:
            state.device, state.streams[s.device] = device, old

    def empty(nbytes, dtype, device):
        # torch's allocator: the memory belongs to the current stream of the
        # device that it lies on; taken in relaxed mode, so that another
        # thread's capture is left alone
        assert state.mode == 2
        state.taken.append((device.index, state.streams[device.index]))
        return "memory"

    cuda = types.SimpleNamespace(
        Stream=_Stream, stream=stream,
        current_device=lambda: state.device,
        is_current_stream_capturing=lambda: capturing,
        OutOfMemoryError=MemoryError)
    return types.SimpleNamespace(cuda=cuda, uint8="u8", empty=empty), state


def _use(monkeypatch, torch, state):
    """The stand-in in torch's place, and one for the capture mode."""
    def exchange(ref):
        mode = ctypes.cast(ref, ctypes.POINTER(ctypes.c_int))
        state.mode, mode[0] = mode[0], state.mode
        return 0

    monkeypatch.setattr(sw, "_torch", torch)
    monkeypatch.setattr(sw, "load_library", lambda: types.SimpleNamespace(
        hipThreadExchangeStreamCaptureMode=exchange))


def _like(index):
    return types.SimpleNamespace(device=types.SimpleNamespace(index=index))


@pytest.mark.parametrize("operands,side,want", [
    (0, None, (0, "s0")),  # the plain call
    (1, None, None),       # operands on a device that is not current
    (1, 1, (1, "side")),   # a side stream of the operands' device
    (0, 1, None),          # a side stream of another device
])
def test_scratch_lies_on_the_launch_stream(monkeypatch, operands, side, want):
    torch, state = _fake_torch()
    _use(monkeypatch, torch, state)
    stream = None if side is None else _Stream(side)
    got = sw._workspace(64, _like(operands), stream)
    if want is None:
        assert got is None and state.taken == []
    else:
        assert got == "memory"
        device, on = state.taken[0]
        assert (device, "side" if on is stream else on) == want
    assert state.mode == 0


def test_no_scratch_under_capture_or_on_a_raw_stream(monkeypatch):
    torch, state = _fake_torch(capturing=True)
    _use(monkeypatch, torch, state)
    assert sw._workspace(64, _like(0), None) is None
    assert sw._workspace(64, _like(0), object()) is None
    assert state.taken == []
