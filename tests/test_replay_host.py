"""Recorded passes on the host side, without a GPU: the library is a stub that notes its calls and runs recorded sequences
by reading their words, so what a recording holds and when it is used can be looked at call by call."""
import abc
import copy
import ctypes
import gc
import pickle
import threading
import weakref
from types import SimpleNamespace

import pytest
import torch

from maskedincrementeval_amd import _lib, ops, replay
from maskedincrementeval_amd import mask_incr_modules as mm
from maskedincrementeval_amd.event_frontend import EventFrames
from maskedincrementeval_amd.mask_incr_functional import IncrementReserve
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.e2depth_incr import E2VIDRecurrentIncr, UpsampleConvLayerIncr


class StubLib:
    """Answers every entry point with 0; `calls` holds (thread, name, arguments), recorded calls as their words."""

    def __init__(self, real):
        self._real = real
        self.calls = []
        self.mie_call_index, self.mie_call_signature = real.mie_call_index, real.mie_call_signature
        self.mie_conv_f32x3_takes = lambda *a: 0

    def __getattr__(self, name):
        if not name.startswith("mie_"):
            raise AttributeError(name)

        def fn(*args):
            self.calls.append((threading.get_ident(), name, args))
            return 0
        return fn

    def mie_run_calls(self, calls, n, inputs, n_inputs, stream):
        names = {self._real.mie_call_index(k.encode()): k for k in _lib.EXPORTS if self._real.mie_call_index(k.encode()) >= 0}
        for c in calls[:n]:
            words = list(ctypes.cast(c.args, ctypes.POINTER(ctypes.c_uint64))[:c.n_args])
            patches = ctypes.cast(c.patches, ctypes.POINTER(ctypes.c_int32))
            for p in range(c.n_patches):
                words[patches[2 * p]] = inputs[patches[2 * p + 1]]
            self.calls.append((threading.get_ident(), names[c.entry], words))
        return 0

    def named(self, name, thread=None):
        return [a for t, n, a in self.calls if n == name and thread in (None, t)]


@pytest.fixture
def stub(mie_lib, monkeypatch):
    """The package on CPU tensors over a StubLib."""
    s = StubLib(mie_lib)
    monkeypatch.setattr(_lib, "_lib", s)
    monkeypatch.setattr(ops, "_require_gpu", lambda t, name: None)
    monkeypatch.setattr(ops, "_stream", lambda t: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: SimpleNamespace(cuda_stream=0))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 0, raising=False)
    monkeypatch.setattr(replay, "_is_nhwc", lambda t: t.dim() == 4 and t.is_contiguous(memory_format=torch.channels_last))
    return s


def in_thread(fn):
    """fn() in another thread: its result, or its exception raised here."""
    box = []

    def body():
        try:
            box.append((fn(), None))
        except BaseException as e:
            box.append((None, e))
    t = threading.Thread(target=body)
    t.start()
    t.join(60)
    assert box, "the thread did not end"
    if box[0][1] is not None:
        raise box[0][1]
    return box[0][0]


def test_a_planning_pass_is_seen_by_its_own_thread_only(stub):
    ts = SimpleNamespace(ref=None, device=torch.device("cpu"), parent=None)

    def other():
        assert ops._phase is None and ops._plan_batch is None and ops.buffer_parity == 0
        assert ops.lib().mie_conv_masked_ws(1) == 0
        ops.build_mask_tiles(None, None, 1, 8, 8, 0, 1, 1, 0, ts)
        with ops.network_pass("compute"):
            pass
        return threading.get_ident()

    with ops.network_pass("plan"):
        ops.lib().mie_conv_masked_ws(0)                  # a planning pass: not made
        me = in_thread(other)
        assert not ops._plan_batch and ops._phase == "plan"
        ops._plan_batch.clear()
    assert stub.named("mie_conv_masked_ws") == stub.named("mie_conv_masked_ws", me) == [(1,)]
    assert len(stub.named("mie_build_mask_tiles", me)) == 1


def test_threads_record_side_by_side(stub):
    """Two threads record at the same time: each recording holds its thread's calls, all of them and no other's."""
    meet = threading.Barrier(2, timeout=30)

    def one(tag):
        def body():
            meet.wait()
            for i in range(20):
                assert ops.lib().mie_mul_dense(0, 0, 0, 100 * tag + i, 0, 0) == 0
                replay.keep(tag)
                if i % 5 == 0:
                    meet.wait()
            return tag
        result, program = replay._record([body], (), [], (), [])
        assert result == tag and program is not None and set(program.held[0]) == {tag}
        return program

    got = {}
    threads = [threading.Thread(target=lambda t=t: got.__setitem__(t, one(t))) for t in (1, 2)]
    [t.start() for t in threads]
    [t.join(60) for t in threads]
    for tag in (1, 2):
        del stub.calls[:]
        got[tag].run((), 0)
        assert [w[3] for w in stub.named("mie_mul_dense")] == [100 * tag + i for i in range(20)]


def _cl(*shape):
    return torch.randn(*shape).contiguous(memory_format=torch.channels_last)


def _conv(c=8, k=3):
    conv = mm.nnConvIncr(c, c, k, 1, k // 2)
    act = mm.nnReservedActivation(mm.leaky_relu_op(0.01), refine_mask=False)
    act.in_res.reservoir = _cl(1, c, 8, 8)
    return conv, act


def _programs(m):
    return [p for p in m.__dict__.get("_replay", {}).values() if isinstance(p, replay.Program)]


def _ptrs(words):
    """(x, x mask, addend) of a recorded mie_conv_masked_ws."""
    return words[0], words[1], words[17]


def test_an_addend_that_was_the_delta_when_recorded(stub):
    """The same tensor as the delta and as the addend in the recorded passes: later passes read each from where it is."""
    conv, act = _conv()
    c = _cl(1, 8, 8, 8)
    m = torch.ones(1, 1, 8, 8, dtype=torch.uint8)
    with torch.no_grad():
        for _ in range(3):
            conv.forward_fused([c, m], act, addend_incr=[c, m])
        for x in (_cl(1, 8, 8, 8), c, _cl(1, 8, 8, 8)):
            mask = m.clone()
            del stub.calls[:]
            conv.forward_fused([x, mask], act, addend_incr=[c, m])
            (words,) = stub.named("mie_conv_masked_ws")
            assert _ptrs(words) == (x.data_ptr(), mask.data_ptr(), c.data_ptr())
    assert [p.runs for p in _programs(conv)] == [3]


def test_a_recording_holds_no_input(stub):
    conv, act = _conv()
    gone = []
    with torch.no_grad():
        for _ in range(5):
            x, m = _cl(1, 8, 8, 8), torch.ones(1, 1, 8, 8, dtype=torch.uint8)
            gone += [weakref.ref(x), weakref.ref(m)]
            conv.forward_fused([x, m], act)
            del x, m
    del stub.calls[:]
    gc.collect()
    assert [p.runs for p in _programs(conv)] == [2] and not any(r() is not None for r in gone)
    sizes = [t for t in gc.get_objects() if type(t) is torch.Tensor and t.dtype == torch.uint8 and tuple(t.shape) == (1, 1, 8, 8)]
    assert len(sizes) == 1          # the tile set's own pixel mask; no copy of an input's


def test_a_pass_that_hands_an_input_on_is_walked_and_hands_on_the_callers(stub):
    x, m = _cl(1, 8, 8, 8), torch.ones(1, 1, 8, 8, dtype=torch.uint8)

    def body(pair):
        ops.lib().mie_mul_dense(pair[0].data_ptr(), 0, 0, 1, 0, 0)
        return [pair[0], (pair[1], {"mask": pair[1]})]
    result, program = replay._record([body], ([x, m],), [(0, 0), (0, 1)], (), [])
    assert program is None and result[0] is x and result[1][0] is m and result[1][1]["mask"] is m


def test_a_planning_pass_asks_the_library_for_its_shapes(stub):
    """What decides a layer's kernels is asked in the planning pass as in the compute pass: both walk the same layers."""
    stub.mie_conv_f32x3_takes = lambda *args: 1
    for phase in (None, "plan", "compute"):
        with ops.network_pass(phase):
            assert ops.f32x3_takes(5, 1, 256, 0, 128), phase


def _network():
    net = E2VIDRecurrentIncr().eval()
    x = _cl(1, 5, 16, 16)
    for _ in range(4):
        net.forward_refresh_reservoirs(x, None)
    return net, x


def test_a_mask_of_the_callers_may_lie_anywhere(stub):
    """Steps whose mask is a new tensor each time: recorded once, and the plan reads the mask of the pass at hand."""
    with torch.no_grad():
        net, _ = _network()
        for i in range(8):
            m = torch.ones(1, 1, 16, 16, dtype=torch.bool if i % 2 else torch.uint8)
            x = _cl(1, 5, 16, 16)
            del stub.calls[:]
            net([x, m], None)
            if i < 6:
                continue
            (plan,) = stub.named("mie_build_mask_plan")
            arr = ctypes.cast(plan[0], ctypes.POINTER(_lib.MiePlanOp))
            assert m.data_ptr() in [arr[k].in_mask for k in range(plan[1])]
            assert stub.named("mie_conv_masked_ws")[0][:2] == [x.data_ptr(), m.data_ptr()]
    assert sorted(p.runs for p in _programs(net)) == [1, 1, 1]      # two kinds of mask, and the refresh


def test_inputs_never_seen_again_push_no_recording_out(stub):
    with torch.no_grad():
        net, x = _network()
        assert [p.runs for p in _programs(net)] == [1]
        alive = []
        for _ in range(3 * replay.MAX_RECORDINGS):
            states = [[_cl(1, c, s, s)] * 2 for c, s in ((64, 8), (128, 4), (256, 2))]
            net([x, None], [[[h, None], [c, None]] for h, c in states])
            alive.append(states)
        net.forward_refresh_reservoirs(x, None)
    assert [p.runs for p in _programs(net)] == [2]
    assert len(net.__dict__["_replay"].waiting) <= replay.MAX_RECORDINGS


def _step(net, size=16):
    net([_cl(1, 5, size, size), None], None)


def test_an_assignment_ends_the_recordings_that_read_the_object_and_no_other(stub):
    with torch.no_grad():
        a, b = (_network()[0] for _ in range(2))
        layer, act = _conv()
        for _ in range(4):
            _step(a), _step(b)
            layer.forward_fused([_cl(1, 8, 8, 8), None], act)
        mm.set_input_threshold(b, None)
        act.in_res.reservoir = _cl(1, 8, 8, 8)
        assert [p.valid() for p in _programs(a)] == [True, True]
        assert [p.valid() for p in _programs(b)] == [False, False]
        assert [p.valid() for p in _programs(layer)] == [False]
        for change in (lambda n: setattr(n.unetrecurrent.decoders[1].activation, "op", torch.tanh),
                       lambda n: setattr(n.unetrecurrent.encoders[0].recurrent_block.cell_res, "reservoir", None),
                       lambda n: delattr(n.unetrecurrent.head.conv2d, "path")):
            net = _network()[0]
            [_step(net) for _ in range(4)]
            assert all(p.valid() for p in _programs(net)) and len(_programs(net)) == 2
            change(net)
            assert not any(p.valid() for p in _programs(net))


def test_a_new_frame_size_frees_the_reservoirs_of_the_former_one(stub):
    with torch.no_grad():
        net, _ = _network()
        [_step(net) for _ in range(5)]
        reserves = [r for m in net.modules() for r in vars(m).values() if isinstance(r, IncrementReserve)]
        old = [weakref.ref(r.reservoir) for r in reserves if r.reservoir is not None]
        assert len(old) > 10
        net.forward_refresh_reservoirs(_cl(1, 5, 32, 32), None)
        assert not any(r() is not None for r in old)
        [_step(net, 32) for _ in range(4)]
    res = net.unetrecurrent.head.activation.in_res           # (what notes its readers stays copyable)
    for twin in (copy.deepcopy(res), pickle.loads(pickle.dumps(res))):
        assert torch.equal(twin.reservoir, res.reservoir)
        twin.reservoir = None
    assert all(p.valid() for p in _programs(net)[-1:])


@pytest.mark.parametrize("cls,name", [(mm.nnConvIncr, "_incr_forward"), (mm.nnConvIncr, "lossy_input"), (mm._IncrBuffers, "_delta_buf"),
                                      (mm._ConvIncrMixin, "_conv_tile_set"), (mm.nnReluIncr, "forward")])
def test_a_replaced_method_gets_its_calls(stub, monkeypatch, cls, name):
    """Also one that recordings do not go through by name, a mixin's, and one set on a class that inherited it."""
    with torch.no_grad():
        net, layer = _network()[0], mm.nnConvIncr(8, 8, 3, 1, 1)
        one = lambda: (_step(net), layer([_cl(1, 8, 8, 8), None]))
        [one() for _ in range(5)]
        assert all(len(_programs(m)) and all(p.valid() for p in _programs(m)) for m in (net, layer))
        seen, real = [], getattr(cls, name)
        inherited = name not in vars(cls)
        with monkeypatch.context() as patch:
            patch.setattr(cls, name, lambda self, *args, **kw: (seen.append(1), real(self, *args, **kw))[1])
            for _ in range(6):
                del seen[:]
                one()
                assert seen or cls is mm.nnReluIncr
            assert not any(p.valid() for p in _programs(net))
        assert (name in vars(cls)) != inherited
        before = len(stub.named("mie_conv_masked_ws"))
        for _ in range(40):
            one()
        assert any(p.valid() for p in _programs(net)) and len(stub.named("mie_conv_masked_ws")) > before


def test_a_method_replaced_in_an_object_gets_its_calls(stub):
    with torch.no_grad():
        net, _ = _network()
        [_step(net) for _ in range(5)]
        conv, seen = net.unetrecurrent.resblocks[0].conv1, []
        real = conv._incr_forward
        conv._incr_forward = lambda *args, **kw: (seen.append(1), real(*args, **kw))[1]
        for _ in range(8):
            del seen[:]
            _step(net)
            assert seen


def test_a_subclass_of_a_module_may_be_abstract_and_changes_nothing_for_others():
    class Mine(mm.nnConvIncr, abc.ABC):
        count = 0
    before = replay.WatchedType.changes
    Mine.count += 1
    assert Mine(4, 4, 3).weight.shape == (4, 4, 3, 3) and replay.WatchedType.changes == before


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_event_frames_are_copied_with_buffers_of_their_own(stub, dtype):
    frames = EventFrames(20, 12, device="cpu", dtype=dtype)
    frames.set_events(torch.zeros(3, 4, dtype=torch.float64))
    entry = "mie_events_to_frame" if dtype == torch.float32 else "mie_events_to_frame_bf16"
    frames.delta(0.0, 0.1)
    for twin in (copy.deepcopy(frames), pickle.loads(pickle.dumps(frames))):
        del stub.calls[:]
        out, mask = twin.delta(0.0, 0.1)
        (args,) = stub.named(entry)
        assert args[0] == twin._events.data_ptr() != frames._events.data_ptr()
        assert args[-3:-1] == (out.data_ptr(), mask.data_ptr()) and out.data_ptr() != frames._delta.data_ptr()


def test_a_workspace_per_stream(stub, monkeypatch):
    """Two streams never share a split workspace, whoever recorded what where; captured launches have one of their own."""
    at = [1]
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: at[0], raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, device=None, **kw: empty(*a, **kw))
    monkeypatch.setattr(ops, "_split_ws", {})
    monkeypatch.setattr(ops, "_captured_ws", {})
    monkeypatch.setattr(ops, "SPLIT_WORKSPACE_BYTES", 4096)
    dev = torch.device("cpu")
    got = {}
    for stream in (1, 2, 1, 2):
        at[0] = stream
        got.setdefault(stream, ops.split_workspace(dev))
        assert got[stream] is ops.split_workspace(dev)
    assert got[1] is not got[2]
    with monkeypatch.context() as patch:
        patch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        captured = ops.split_workspace(dev)
        at[0] = 1
        assert captured is ops.split_workspace(dev) and captured is not got[1] and captured is not got[2]

    def body(x):
        ptr, size = ops._workspace_args(None, True, dev)
        ops.lib().mie_upconv_masked_ws(x.data_ptr(), None, None, None, 64, 4, 4, 0, 0, 64, 5, 2, 32, None, 0, None, None, 0, 0.0, 0, ptr, size, 0)
        return None

    x = _cl(1, 64, 4, 4)
    at[0] = 1
    _, program = replay._record([body], (x,), [(0, None)], (), [])
    for stream in (1, 2, 3, 1):
        at[0] = stream
        del stub.calls[:]
        program.run([x.data_ptr()], dev)
        assert stub.named("mie_upconv_masked_ws")[0][20] == ops.split_workspace(dev).data_ptr()
    for stream in range(10, 60):
        at[0] = stream
        ops.split_workspace(dev)
    assert len(ops._split_ws) <= ops.SPLIT_WORKSPACES


def test_a_plan_is_for_the_tile_sets_at_hand(stub):
    """A tile set that shares some of its addresses with a former one is not planned as that one; plans made for buffers
    that are gone do not pile up."""
    def planned(*sets):
        with ops.network_pass("plan"):
            for ts in sets:
                ops.build_mask_tiles(None, None, 1, 16, 16, _lib.FOOT_CONV, 3, 1, 1, ts)
        arr, n, _ = stub.named("mie_build_mask_plan")[-1]
        return [bytes(op.out) for op in arr[:n]]

    a, b = (TileMask(1, 16, 16, "cpu") for _ in range(2))
    assert planned(a, b) == planned(a, b) == [bytes(a.c_struct), bytes(b.c_struct)]
    other = torch.zeros_like(a.flags)
    a.c_struct.flags = other.data_ptr()
    assert planned(a, b) == [bytes(a.c_struct), bytes(b.c_struct)]
    for _ in range(3 * ops.PLAN_CACHE):
        a.c_struct.flags += 64
        planned(a)
    assert len(ops._plan_cache) <= ops.PLAN_CACHE


def test_decoder_layers_take_the_form_without_lists_where_the_plane_is_dense(stub, monkeypatch):
    monkeypatch.setattr(ops, "upconv2x_takes", lambda *args: True)
    monkeypatch.setattr(ops, "upconv_takes", lambda *args: True)

    def taken(layer, x_mask, skip_mask, skip=True):
        x, y = _cl(1, 64, 8, 8), _cl(1, 64, 8, 8)
        layer.activation.in_res.reservoir = _cl(1, 32, 16, 16)
        del stub.calls[:]
        layer([x, x_mask], [y, skip_mask] if skip else None)
        return [n for _, n, _ in stub.calls if n.startswith("mie_upconv")]

    mask = torch.ones(1, 1, 8, 8, dtype=torch.uint8)
    with torch.no_grad():
        layer = UpsampleConvLayerIncr(64, 32, 5, padding=2)
        lists, dense = ["mie_upconv_masked_ws"], ["mie_upconv2x_masked"]
        assert taken(layer, mask, mask) == taken(layer, mask, None, skip=False) == lists
        assert taken(layer, None, mask) == taken(layer, mask, None) == taken(layer, None, None, skip=False) == dense
        layer.dense_plane = True
        assert taken(layer, mask, mask) == dense
        assert all(d.dense_plane for d in E2VIDRecurrentIncr().unetrecurrent.decoders)


def test_layers_are_recorded_one_by_one_only_where_their_network_is_not(stub):
    inner = lambda net: [m for m in net.modules() if m is not net and m.__dict__.get("_replay") is not None]
    with torch.no_grad():
        net, _ = _network()
        for _ in range(6):
            _step(net)
            assert not inner(net)
        alive = []
        for i in range(replay.WALKS + 8):        # (states at new addresses each time: passes that are never recorded)
            alive.append([[_cl(1, c, s, s), _cl(1, c, s, s)] for c, s in ((64, 8), (128, 4), (256, 2))])
            net([_cl(1, 5, 16, 16), None], [[[h, None], [c, None]] for h, c in alive[-1]])
            assert bool(inner(net)) == (i >= replay.WALKS)
        assert any(p.runs for m in inner(net) for p in _programs(m))
        assert not ops._pass.walking
