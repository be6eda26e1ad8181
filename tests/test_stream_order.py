"""What the backend's calls are ordered behind and ahead of, on a model of streams and events (no GPU): every launch and
every op of the program carries the set of those that must have run before it."""
import ctypes as C

import pytest
import torch

from ferrite_amd import backend
from ferrite_amd.synth import MoeConfig


class Event:
    def __init__(self, *a, **k):
        self.before = set()

    def record(self, stream=None):
        self.before = set((stream or Sim.current).before)

    def synchronize(self):
        Sim.waited |= self.before


class Stream:
    def __init__(self, handle=None, **k):
        Sim.handles += 16
        self.cuda_stream = Sim.handles if handle is None else handle
        self.before, self.capturing = set(), False
        Sim.streams[self.cuda_stream] = self

    def __eq__(self, other):
        raise TypeError("streams are compared by their handles: torch's `stream != None` is False")

    __ne__ = __eq__

    def record_event(self, event=None):
        event = event or Event()
        event.record(self)
        return event

    def wait_event(self, event):
        self.before |= event.before

    def wait_stream(self, stream):
        self.wait_event(stream.record_event())

    def synchronize(self):
        Sim.waited |= self.before

    def op(self, name):
        """Queue something on this stream; returns what has run before it."""
        seen = set(self.before)
        self.before.add(name)
        return seen


class Sim:
    handles, streams, current, waited, launches = 4096, {}, None, set(), []


class Lib:
    """Every entry succeeds; one that is given a stream is a launch there."""

    def __getattr__(self, name):
        def entry(*args):
            if name.endswith("_bytes"):
                return 64
            handles = [a.value or 0 for a in args if type(a) is C.c_void_p]
            if handles and name not in ("ferrite_graph_begin", "ferrite_graph_end", "ferrite_graph_destroy"):
                stream = Sim.streams[handles[-1]]
                launch = f"launch {len(Sim.launches)}"
                Sim.launches.append((name, stream, stream.op(launch)))
            return backend.OK
        return entry


@pytest.fixture
def hip(monkeypatch):
    Sim.streams, Sim.waited, Sim.launches = {}, set(), []
    Sim.current = Stream(handle=0)
    for name, value in dict(is_available=lambda: True, set_device=lambda d: None, current_device=lambda: 0, Stream=Stream,
                            Event=Event, current_stream=lambda d=None: Sim.current,
                            is_current_stream_capturing=lambda: Sim.current.capturing).items():
        monkeypatch.setattr(torch.cuda, name, value)
    monkeypatch.setattr(backend, "load_library", lambda path=None: Lib())
    monkeypatch.setattr(backend.HipBackend, "_dev", lambda self, t, dtype, what: t)
    be = backend.HipBackend()
    be.device = torch.device("cpu")   # where the calls allocate
    return be


CFG = MoeConfig(4, 128, 4, 2, 128, 0, 1, 1)
z = torch.zeros


def _layer():
    layer = backend.MoeLayer(CFG, {}, z(64, dtype=torch.uint8))
    return layer, z(4, 128), z(4, 128), z(64, dtype=torch.uint8)


def _layer_call(hip):
    layer, x, out, ws = _layer()
    hip.moe_layer_dev_mxfp4(layer, x, out, workspace=ws)


def _static_call(hip):
    layer, x, out, _ = _layer()
    hip.moe_layer_dev_mxfp4_static(layer, x, out)


def _block_call(hip):
    layer, x, out, ws = _layer()
    hip.moe_block_mxfp4(layer, x, z(128), 1e-6, None, None, None, out, workspace=ws)


def _replay(hip):
    hip.begin_verify(backend.OpTrace([], graph_exec=Sim.current.cuda_stream))


CALLS = dict(
    matmul=lambda h: h.matmul(z(4, 8), z(6, 8), None, z(4, 6)),
    rmsnorm=lambda h: h.rmsnorm(z(4, 8), z(8), 1e-6, z(4, 8)),
    swiglu=lambda h: h.swiglu_limited(z(4, 8), 10.0, z(4, 4)),
    moe_route=lambda h: h.moe_route(z(4, 8), z(8), 2, 1.0, z(4, 2), z(4, 2)),
    hc_post=lambda h: h.hc_post(z(4, 8), z(4, 2, 8), z(4, 2), z(4, 2, 2)),
    moe_permute=lambda h: h.moe_permute(z(4, 2, dtype=torch.int32), 4),
    mxfp4_quant=lambda h: h.mxfp4_quant(z(4, 32)),
    mxfp4_dequant=lambda h: h.mxfp4_dequant(z(4, 16, dtype=torch.uint8), z(4, 1, dtype=torch.uint8)),
    act_quant=lambda h: h.act_quant_fp8(z(4, 32)),
    act_quant_x2=lambda h: h.act_quant_fp8_x2(z(4, 32)),
    pack_expert=lambda h: h.pack_expert(_layer()[0], 0),
    packed_dequant=lambda h: h.packed_dequant(_layer()[0], 0, 0),
    layer=_layer_call, layer_static=_static_call, block=_block_call, replay=_replay)


@pytest.mark.parametrize("call", CALLS)
def test_a_call_runs_between_the_ops_around_it(hip, call):
    """Inputs are made and outputs are read by torch ops on the current stream, with no synchronisation in between."""
    for side in (Sim.current, Stream()):
        Sim.current = side
        side.op("input")
        CALLS[call](hip)
        (_, _, seen), launch = Sim.launches[-1], f"launch {len(Sim.launches) - 1}"
        assert "input" in seen
        assert launch in side.op("output")


def test_calls_on_several_streams_run_one_after_the_other(hip):
    """They share workspaces and graphs, so no call may overtake one that was made before it."""
    streams = [Sim.current, Stream(), Stream(), hip.stream]
    for i in (0, 1, 0, 2, 1, 1, 3, 2, 3, 0):
        Sim.current = streams[i]
        (_replay if i == 2 else _layer_call)(hip)
        made = {f"launch {k}" for k in range(len(Sim.launches) - 1)}
        assert made <= Sim.launches[-1][2]
        hip.sync()
        assert f"launch {len(Sim.launches) - 1}" in Sim.waited


def test_work_on_the_backends_own_stream_is_ordered_with_the_calls(hip):
    _layer_call(hip)
    assert "launch 0" in hip.stream.op("mine")
    _layer_call(hip)
    assert "mine" in Sim.launches[-1][2]
    hip.stream.op("last")
    hip.sync()
    assert "last" in Sim.waited


def test_a_capture_records_on_one_stream(hip):
    _layer_call(hip)
    hip.begin_capture()
    for call in ("rmsnorm", "layer", "hc_post"):
        CALLS[call](hip)
        assert Sim.launches[-1][1].cuda_stream not in (0, None)
    assert len({s.cuda_stream for _, s, _ in Sim.launches[1:]}) == 1
    hip.end_capture()
    Sim.current.op("input")
    _replay(hip)
    assert "input" in Sim.launches[-1][2]
    assert f"launch {len(Sim.launches) - 1}" in Sim.current.op("output")


SHARED = ("layer", "layer_static", "block", "replay")   # calls that use memory other calls use too


@pytest.mark.parametrize("call", CALLS)
def test_a_capture_that_the_program_opened(hip, call):
    """Calls that share nothing are recorded on its stream, and nothing eager waits for them; the others are refused there."""
    Sim.current = side = Stream()
    CALLS["rmsnorm"](hip)
    side.capturing = True
    if call in SHARED:
        with pytest.raises(backend.FerriteError, match="capture"):
            CALLS[call](hip)
        assert len(Sim.launches) == 1
    else:
        CALLS[call](hip)
        assert Sim.launches[-1][1] is side and len(Sim.launches) == 2
    Sim.current = Stream()
    _layer_call(hip)
    assert Sim.launches[-1][2] == {"launch 0"}


@pytest.mark.parametrize("call", CALLS)
def test_a_capture_that_the_program_opened_on_the_backends_own_stream(hip, call):
    Sim.current = hip.stream
    Sim.current.capturing = True
    CALLS[call](hip)
    assert Sim.launches[-1][1] is Sim.current
