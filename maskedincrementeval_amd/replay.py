"""Recorded steps: the library calls of a module or a whole network, noted once and handed over as one sequence.

A step makes the same calls every time: buffers, tile sets, filters and reservoirs stay where they are, only the input
tensors move.  Walking the modules costs the host 15-25 us per call (shape checks, pointers, buffer look-ups, argument
conversion) where the kernels behind it take 5-20 us, so the plain calls of small and medium frames were bound by Python:
an E2Depth-incr step at 64x96 took 596 us for 230 us of kernels.  The third pass over an input of one shape is
therefore recorded (`Recording`: every call of the library with its arguments), and later passes hand the sequence
to mie_run_calls with the pointers of their inputs filled in -- about 3 us a call, the launch itself.

A recording stands for the Python pass as long as everything that pass read is what it was:
  * attributes of the package's modules it went through and which reservoir tensor an IncrementReserve of theirs holds:
    an assignment ends the recordings that read the object, and what they hold is freed (`Watched`);
  * weights: the parameter objects, their addresses and version counters;
  * the settings and functions of `ops` (a program or a test that replaces one gets its calls);
  * the package's module classes (a method replaced by an instrumented one gets its calls), forward hooks, and the
    members of module containers.
Otherwise the pass runs in Python again and is recorded anew.  A pass that runs any torch operation of its own
(a conversion, a concat, the allocation of a buffer) is never recorded, nor one on a planning stream or inside a
planning pass, nor under graph capture.  It is recorded on copies of its inputs, so that what is an input is known by
its address.  Recordings hold references to every tensor whose address they use.
"""
import abc
import collections
import ctypes
import functools
import operator
import os
import struct
import threading
import weakref

import torch
from torch.utils._python_dispatch import TorchDispatchMode

from . import _lib
from ._lib import check

enabled = os.environ.get("MIE_REPLAY", "1") != "0"      # read once
MAX_RECORDINGS = 8          # per module, least recently used first out
# While a pass waits to be recorded, the passes inside it (its layers') do not look for recordings of their own; once this
# many passes in a row were walked it is one that is not recorded, and its layers are.
WALKS = 4
_recording = {}             # thread identity -> the Recording that thread is making
_SILENT = frozenset(("training", "states"))     # assignments no incremental pass depends on


class _Readers(list):
    """Weak references to the programs that read an object.  Copies and pickles of the object start without any."""

    def __deepcopy__(self, memo):
        return _Readers()

    def __reduce__(self):
        return _Readers, ()


# attributes that Python itself puts on classes (copying an object adds __slotnames__)
_NOT_CODE = frozenset(("__abstractmethods__", "__annotations__", "__doc__", "__dict__", "__weakref__", "__slotnames__"))


class WatchedType(abc.ABCMeta):
    """Class of the package's module classes and mixins: notes when an attribute of one is replaced, whoever does it.  (Of
    ABCMeta, so that a caller's subclass may be an abstract one, too.)"""
    changes = 0              # replacements so far, in all classes of the package
    defined = {}             # class of the package -> its attributes as they were written
    looked_at = {}           # class -> (changes, as_written) when last looked at

    def __init__(cls, *args, **kw):
        super().__init__(*args, **kw)
        if cls.__module__.split(".")[0] == __package__:
            WatchedType.defined[cls] = WatchedType.code_of(cls)

    def code_of(cls):
        return {k: v for k, v in vars(cls).items() if k not in _NOT_CODE and not k.startswith("_abc_")}

    def __setattr__(cls, name, value):
        if cls in WatchedType.defined and name not in _NOT_CODE:
            WatchedType.changes += 1
        super().__setattr__(name, value)

    def __delattr__(cls, name):
        if cls in WatchedType.defined:
            WatchedType.changes += 1
        super().__delattr__(name)

    def as_written(cls):
        """Whether this class and the package's classes it comes from are what their sources say."""
        seen = WatchedType.looked_at.get(cls)
        if seen is None or seen[0] != WatchedType.changes:
            same = True
            for c in cls.__mro__:
                was = WatchedType.defined.get(c)
                if was is not None:
                    now = WatchedType.code_of(c)
                    same = same and now.keys() == was.keys() and all(now[k] is was[k] for k in was)
            seen = WatchedType.looked_at[cls] = (WatchedType.changes, same)
        return seen[1]


_methods = {}                # class -> (changes, names of what can be called on it)


def _methods_of(cls):
    seen = _methods.get(cls)
    if seen is None or seen[0] != WatchedType.changes:
        names = frozenset(k for c in cls.__mro__ for k, v in vars(c).items() if callable(v))
        seen = _methods[cls] = (WatchedType.changes, names)
    return seen[1]


class Watched(metaclass=WatchedType):
    """First base of the package's modules and reservoirs: an assignment to an attribute ends the programs that read the
    object, before the attribute changes."""

    def __setattr__(self, name, value):
        if name not in _SILENT:
            outdate(self)
        super().__setattr__(name, value)

    def __delattr__(self, name):
        outdate(self)
        super().__delattr__(name)


def outdate(obj):
    for ref in obj.__dict__.pop("_replay_readers", ()):
        program = ref()
        if program is not None:
            program.end()


_PLAIN = frozenset((dict, collections.OrderedDict, set, bool, int, float, str, type(None), torch.Tensor))


def _watched_in(modules):
    """The watched objects a pass over these modules reads: themselves, and the reservoirs they hold."""
    found = {id(m): m for m in modules if isinstance(type(m), WatchedType)}
    for m in modules:
        for x in vars(m).values():
            if type(x) not in _PLAIN:
                for y in (x if type(x) in (list, tuple) else (x,)):
                    if isinstance(type(y), WatchedType):
                        found[id(y)] = y
    return found.values()


class ValueDependentMask(RuntimeError):
    """A mask that depends on values met inside a planning pass."""


# ---- what the pass reads outside the modules -----------------------------------------------------------------
_ops_globals = _ops_pass = None
_get_functions = _get_settings = None
_functions = ()


def bind_ops(namespace, pass_state, functions, settings):
    """Called once by ops: its namespace, the state of a thread's pass, and the names a pass goes through / depends on."""
    global _ops_globals, _ops_pass, _get_functions, _get_settings, _functions
    _ops_globals, _ops_pass = namespace, pass_state
    _get_functions, _get_settings = operator.itemgetter(*functions), operator.itemgetter(*settings)
    _functions = _get_functions(namespace)


def _idle() -> bool:
    """Whether ops is in its ordinary state for this thread: no planning pass, no planning stream, no pending threshold
    mask -- and its functions are its own."""
    s = _ops_pass
    return (s.phase is None and s.planner is None and not s.pending_thr and s.buffer_parity == 0
            and _get_functions(_ops_globals) == _functions)


# ---- recording ------------------------------------------------------------------------------------------------
# questions to the library, answered in every phase and never recorded
PASS_THROUGH = frozenset(("mie_last_error_string", "mie_tile_capacity", "mie_version", "mie_conv_f32x3_takes",
                          "mie_conv_needs_no_workspace", "mie_conv_gates_needs_no_workspace", "mie_upconv_needs_no_workspace",
                          "mie_f16x2_takes_upconv2x", "mie_all_phases_upconv2x"))
_VIEWS = frozenset(("aten::permute", "aten::detach", "aten::view", "aten::slice", "aten::select", "aten::alias",
                    "aten::as_strided", "aten::t", "aten::transpose", "aten::unsqueeze", "aten::squeeze",
                    "aten::expand", "aten::_reshape_alias", "aten::_unsafe_view", "aten::split", "aten::unbind"))


class _TorchWatch(TorchDispatchMode):
    """Notes torch operations other than views."""

    def __init__(self):
        super().__init__()
        self.seen = None

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func._schema.name not in _VIEWS:
            self.seen = func
        return func(*args, **(kwargs or {}))


class Recording:
    """The library as a pass sees it while it is recorded: makes every call and notes the ones that succeed."""

    def __init__(self, real, watch):
        self._real, self.watch = real, watch
        self.calls, self.keep, self.effects = [], [], []
        self.workspace = None

    def __getattr__(self, name):
        fn = getattr(self._real, name)
        if name in PASS_THROUGH or not name.startswith("mie_"):
            return fn

        def noted(*args):
            rc = fn(*args)
            if rc == 0:
                self.calls.append((name, args))
            return rc
        return noted


def current():
    """The Recording this thread is making, or None."""
    return _recording.get(threading.get_ident()) if _recording else None


def lib():
    """The library, or the recording of it this thread is making."""
    if _recording:
        r = _recording.get(threading.get_ident())
        if r is not None:
            return r
    return _lib.lib()


def keep(obj):
    """While a pass is recorded: its recording holds on to `obj`, whose address it uses."""
    if _recording:
        r = _recording.get(threading.get_ident())
        if r is not None:
            r.keep.append(obj)
    return obj


def apart(fn):
    """fn(), which runs torch operations that are no part of a pass being recorded."""
    r = current()
    if r is None:
        return fn()
    seen = r.watch.seen
    result = fn()
    r.watch.seen = seen
    return result


def shared_workspace(ws):
    """While a pass is recorded: notes that `ws` is the workspace of the stream at hand; a replay takes its own stream's."""
    r = current()
    if r is not None:
        r.workspace = ws
    return ws


def effect(fn, *args):
    """fn(*args), now and on every replay of the pass: for changes of host state the pass makes."""
    r = current()
    if r is not None:
        r.effects.append((fn, args))
    return fn(*args)


def _bits(kind, value):
    """The word of a floating-point argument."""
    return struct.unpack("<I", struct.pack("<f", value))[0] if kind == "f" else struct.unpack("<Q", struct.pack("<d", value))[0]


_signatures = {}


def _signature(name):
    s = _signatures.get(name)
    if s is None:
        real = _lib.lib()
        idx = real.mie_call_index(name.encode())
        s = _signatures[name] = (idx, real.mie_call_signature(idx).decode()) if idx >= 0 else None
    return s


def _copy(v):
    """A fresh list / tuple / dict structure around the same tensors and tile sets."""
    t = type(v)
    if t is list:
        return [_copy(x) for x in v]
    if t is tuple:
        return tuple([_copy(x) for x in v])
    if t is dict:
        return {k: _copy(x) for k, x in v.items()}
    return v


class _Inputs:
    """Copies of the inputs of a pass, which the pass is recorded on.  No other tensor lies where they lie, so an argument
    with an address of theirs came from that input: the same argument given as anything else, too (a tensor that is the
    delta in one place and the addend in another), has its own address there."""

    def __init__(self, args, free):
        self.args, self.given, self.copies = list(args), [], []
        for i, j in free:
            given = self.args[i] if j is None else self.args[i][j]
            copy = given.detach().clone()
            self.given.append(given)
            self.copies.append(copy)
            if j is None:
                self.args[i] = copy
            else:
                self.args[i] = list(self.args[i])
                self.args[i][j] = copy
        self.spans = [(c.data_ptr(), c.data_ptr() + c.numel() * c.element_size()) for c in self.copies]
        self.lo, self.hi = min([lo for lo, _ in self.spans], default=0), max([hi for _, hi in self.spans], default=0)

    def slot(self, address):
        """Which input starts at `address`; None: it lies in none."""
        if not address or not self.lo <= address < self.hi:
            return None
        for k, (lo, hi) in enumerate(self.spans):
            if lo <= address < hi:
                if address != lo:
                    raise _NotRecordable("an address inside an input")
                return k
        return None

    def holds(self, t):
        at = t.data_ptr()
        return self.lo <= at < self.hi and any(lo <= at < hi for lo, hi in self.spans)

    def refuse(self, what, *addresses):
        for a in addresses:
            if a and self.lo <= a < self.hi and self.slot(a) is not None:
                raise _NotRecordable(what)

    def refuse_in(self, value):
        """No part of a result or of a change of host state may be an input: the next pass has others."""
        if torch.is_tensor(value):
            self.refuse("an input is handed on", value.data_ptr())
        elif isinstance(value, (list, tuple)):
            for x in value:
                self.refuse_in(x)
        elif isinstance(value, dict):
            self.refuse_in(list(value.values()))
        elif hasattr(value, "c_struct"):
            self.refuse_set(value.c_struct)

    def give_back(self, value):
        """A result with the inputs it hands on, in place of their copies."""
        if type(value) in (list, tuple):
            return type(value)([self.give_back(x) for x in value])
        if type(value) is dict:
            return {k: self.give_back(x) for k, x in value.items()}
        for given, copy in zip(self.given, self.copies):
            if value is copy:
                return given
        return value

    def refuse_set(self, ts):
        self.refuse("a tile set over an input", ts.pixmask, ts.tiles, ts.stale, ts.counts, ts.flags)


class Program:
    """A recorded pass that can be run again."""

    def __init__(self, rec, inputs, result, tree, static):
        self.effects, self.result = rec.effects, result
        self.runs, self.alive = 0, True
        self.plan_masks = []         # (op of a plan, its field, input): set before each run
        self.held = [[k for k in rec.keep if not (torch.is_tensor(k) and inputs.holds(k))], static]
        workspace = None if rec.workspace is None else rec.workspace.data_ptr()
        calls = (_lib.MieCall * len(rec.calls))()
        for call, (name, args) in zip(calls, rec.calls):
            idx, sig = _signature(name)
            words = (ctypes.c_uint64 * max(1, len(sig)))()
            patches = []
            for i, (kind, value) in enumerate(zip(sig, args)):
                if kind == "i" or kind == "l":
                    words[i] = value & 0xFFFFFFFFFFFFFFFF
                    continue
                if value is None or kind == "f" or kind == "d":
                    words[i] = 0 if value is None else _bits(kind, value)
                    continue
                if kind == "t":
                    inputs.refuse_set(value._obj)
                elif isinstance(value, ctypes.Array):       # the ops of a plan: this program's own array of them
                    value = type(value).from_buffer_copy(value)
                    for op in value:
                        inputs.refuse_set(op.out)
                        for field in ("in_mask", "in_mask2"):
                            slot = inputs.slot(getattr(op, field))
                            if slot is not None:
                                self.plan_masks.append((op, field, slot))
                if not isinstance(value, int):
                    self.held.append(value)
                    words[i] = ctypes.addressof(getattr(value, "_obj", value))
                    continue
                words[i] = value
                slot = inputs.slot(value)
                if slot is not None:
                    if kind == "w":
                        raise _NotRecordable("an input is written")
                    patches += [i, slot]
                elif kind == "w" and value == workspace:
                    patches += [i, len(inputs.copies)]          # one input more: the workspace of the stream it runs on
            pa = (ctypes.c_int32 * max(1, len(patches)))(*patches)
            call.entry, call.n_args, call.n_patches = idx, len(sig), len(patches) // 2
            call.args, call.patches = ctypes.addressof(words), ctypes.addressof(pa)
            self.held += [words, pa]
        self.calls, self.n = calls, len(rec.calls)
        self.uses_workspace = workspace is not None
        self.n_inputs = len(inputs.copies) + (1 if self.uses_workspace else 0)
        self.words_type = ctypes.c_uint64 * max(1, self.n_inputs)
        self.fn = _lib.lib().mie_run_calls
        self._guards(tree)

    # what the pass depended on
    def _guards(self, tree):
        mods = []
        for m in tree:
            mods.extend(m.modules())
        mods = list({id(m): m for m in mods}.values())
        self.settings = _get_settings(_ops_globals)
        self.hooks = [d for m in mods for d in (m._forward_hooks, m._forward_pre_hooks)]
        self.hooks += [torch.nn.modules.module._global_forward_hooks, torch.nn.modules.module._global_forward_pre_hooks]
        if any(self.hooks) or not all(_methods_of(type(m)).isdisjoint(vars(m)) for m in mods):
            raise _NotRecordable("hooked, or a method replaced in an object")
        classes = {type(m) for m in mods}
        for c in classes:
            if c.__module__.split(".")[0] not in (__package__, "torch"):
                raise _NotRecordable("a class of the caller's")
            if isinstance(c, WatchedType) and not c.as_written():
                raise _NotRecordable("a class with something replaced")
        self.changes = WatchedType.changes
        self.torch_classes = [c for c in classes if not isinstance(c, WatchedType)]
        self.forwards = [c.forward for c in self.torch_classes]
        self.containers = [m._modules for m in mods if m._modules]
        self.members = [list(d.values()) for d in self.containers]
        self.param_dicts = [m._parameters for m in mods if m._parameters]
        self.params = [p for d in self.param_dicts for p in d.values()]
        self.tensors = [p for p in self.params if p is not None]
        self.addresses = [p.data_ptr() for p in self.tensors]
        self.versions = [p._version for p in self.tensors]
        me = weakref.ref(self)
        for w in _watched_in(mods):
            readers = w.__dict__.setdefault("_replay_readers", _Readers())
            readers[:] = [r for r in readers if r() is not None] + [me]

    def end(self):
        """Never valid again; lets go of everything it held."""
        self.alive = False
        self.held = self.effects = self.result = self.calls = None
        self.plan_masks, self.tensors, self.params, self.param_dicts, self.members, self.containers = [], [], [], [], [], []

    def valid(self) -> bool:
        return (self.alive and self.changes == WatchedType.changes and _get_settings(_ops_globals) == self.settings and not any(self.hooks)
                and [p.data_ptr() for p in self.tensors] == self.addresses
                and [p._version for p in self.tensors] == self.versions
                and all(map(operator.is_, [p for d in self.param_dicts for p in d.values()], self.params))
                and [list(d.values()) for d in self.containers] == self.members
                and [c.forward for c in self.torch_classes] == self.forwards)

    def run(self, pointers, device):
        self.runs += 1
        # (an effect, or another thread, may end this program meanwhile)
        calls, held, effects, result = self.calls, self.held, self.effects, self.result
        for op, field, slot in self.plan_masks:
            setattr(op, field, pointers[slot])
        if self.uses_workspace:
            ws = _ops_globals["split_workspace"](device)
            pointers = [*pointers, ws.data_ptr()]
        check(self.fn(calls, self.n, self.words_type(*pointers), self.n_inputs, torch._C._cuda_getCurrentRawStream(device)))
        for fn, args in effects:
            fn(*args)
        return _copy(result)


class _NotRecordable(Exception):
    pass


class _Cache(collections.OrderedDict):
    """Recordings of one module, by method and input.  Copies and pickles of a module start without any.  `waiting`: the
    passes that have none (yet), apart, so that inputs that are never seen again push no recording out."""

    def __init__(self):
        super().__init__()
        self.waiting = collections.OrderedDict()
        self.walks = 0           # passes walked since the last one that ran from a recording

    def keep(self, key, entry):
        if type(entry) is Program:
            self.waiting.pop(key, None)
            while len(self) >= MAX_RECORDINGS and key not in self:
                self.popitem(last=False)
            self[key] = entry
        else:
            self.pop(key, None)
            while len(self.waiting) >= MAX_RECORDINGS:
                self.waiting.popitem(last=False)
            self.waiting[key] = entry

    def __deepcopy__(self, memo):
        return _Cache()

    def __reduce__(self):
        return _Cache, ()


class _Waiting:
    """A pass that is not recorded (yet): how often it was seen, and when it is tried next."""
    __slots__ = ("seen", "next", "step")

    def __init__(self):
        self.seen, self.next, self.step = 0, 3, 2


def _record(fns, args, free, tree, static):
    """One pass, recorded if it can be: (result, Program or None).  free: positions (argument, index in it or None) of
    the inputs that may lie elsewhere in the next pass."""
    me = threading.get_ident()
    for k, fn in enumerate(fns):
        inputs, watch = _Inputs(args, free), _TorchWatch()
        rec = Recording(_lib.lib(), watch)
        _recording[me], _ops_pass.walking = rec, True
        try:
            with watch:
                result = fn(*inputs.args)
        except ValueDependentMask:
            if k + 1 == len(fns):
                raise
            continue
        finally:
            del _recording[me]
            _ops_pass.walking = False
        if watch.seen is not None or any(_signature(name) is None for name, _ in rec.calls):
            return inputs.give_back(result), None
        try:
            inputs.refuse_in(result)
            inputs.refuse_in([effect_args for _, effect_args in rec.effects])
            return result, Program(rec, inputs, _copy(result), tree, static)
        except _NotRecordable:
            return inputs.give_back(result), None


def _static_key(v, held):
    if v is None or isinstance(v, (int, float, str, bool)):
        return v
    if torch.is_tensor(v):
        return (v.data_ptr(), v.shape, v.stride(), v.dtype)
    if isinstance(v, (list, tuple)):
        return tuple([_static_key(x, held) for x in v])
    held.append(v)
    return id(v)


def _is_nhwc(t) -> bool:
    return (t.dim() == 4 and t.is_cuda and t.dtype in (torch.float32, torch.bfloat16)
            and t.is_contiguous(memory_format=torch.channels_last))


def replayed(record=None, dense=0, masked=1, trees=()):
    """Decorator of a pass: method(self, *args).  The first `dense` arguments are dense tensors and the next `masked`
    ones Masked pairs (or None); those and plain mask tensors of the pairs may live anywhere, everything else has to be
    the same object or memory to be the same pass.  trees: positions of further
    arguments that are modules the pass reads.  record: name of another method to record in place of this one, tried
    first, with the same result (ValueDependentMask: it does not apply)."""
    def decorate(method):
        @functools.wraps(method)
        def wrapped(self, *args, **kw):
            if kw or not enabled or _ops_pass.walking or not _idle():
                return method(self, *args, **kw)
            key, pointers, free, held, device = [method.__name__], [], [], [], None
            for i, a in enumerate(args):
                if a is not None and i < dense + masked:
                    x = a if i < dense else a[0]
                    if not torch.is_tensor(x) or not _is_nhwc(x):
                        return method(self, *args)
                    pointers.append(x.data_ptr())
                    free.append((i, None if i < dense else 0))
                    device = x.device.index
                    key += (x.shape, x.dtype, device)
                    m = None if i < dense or len(a) < 2 else a[1]
                    if torch.is_tensor(m):
                        n, _, h, w = x.shape
                        if (m.dtype not in (torch.uint8, torch.bool) or m.shape != (n, 1, h, w) or not m.is_contiguous()
                                or m.device != x.device):
                            return method(self, *args)
                        pointers.append(m.data_ptr())
                        free.append((i, 1))
                        key.append(m.dtype)
                    else:
                        key.append(_static_key(m, held))
                else:
                    key.append(_static_key(a, held))
            if not pointers or len(set(pointers)) != len(pointers) or 0 in pointers:
                return method(self, *args)
            key = tuple(key)
            cache = self.__dict__.get("_replay")
            if cache is None:
                cache = self.__dict__["_replay"] = _Cache()
            ent = cache.get(key)
            if ent is not None:
                if ent.valid():
                    cache.move_to_end(key)
                    cache.walks = 0
                    return ent.run(pointers, device)
                # outdated: recorded anew like a new one, or later and later if recordings here never last
                w = _Waiting()
                if ent.runs < 16:
                    w.step = w.next = ent.step
                cache.keep(key, w)
                ent = w
            else:
                ent = cache.waiting.get(key)
                if ent is None:
                    ent = _Waiting()
                    cache.keep(key, ent)
            ent.seen += 1
            if ent.seen < ent.next or torch.cuda.is_current_stream_capturing():
                cache.walks += 1
                if cache.walks > WALKS:
                    return method(self, *args)
                _ops_pass.walking = True
                try:
                    return method(self, *args)
                finally:
                    _ops_pass.walking = False
            # tried again after twice as many passes each time, so that a pass that cannot be recorded, or whose
            # surroundings change all the time, costs little more than it did
            ent.step = min(2 * ent.step, 256)
            ent.next = ent.seen + ent.step
            fns = ([getattr(self, record)] if record else []) + [functools.partial(method, self)]
            result, program = _record(fns, args, free, (self,) + tuple(args[i] for i in trees), held)
            if program is not None:
                program.step = ent.step
                cache.keep(key, program)
            return result
        return wrapped
    return decorate
