"""The work a program built on this package has it do, as a list of measurable cases.

A case is a dict of plain values; `prepare` makes what the program holds before the call (the network or layer with
its weights, reservoirs already filled by a dense refresh, inputs resident in HBM), `run` is one call as the program
makes it, and `work` says what the call cannot do without.  Kinds:

step      one incremental frame through a network.  mode: "call" is the plain module call, launched eagerly, as the
          per-frame loops of the evaluation drivers make it; "graph" replays a captured step (one graph per resident
          input, tile sets planned first); "ahead" replays the two captured halves through ops.LookaheadStepper, the
          next step's tile sets planned beside this step (what bench.py times).
          state: the recurrent state deltas of a step are fed to the next one.
refresh   the dense pass that fills the reservoirs (every 20-100 frames of a sequence).
chain     one conv layer with its fused activation and a second activation with a refined mask, called as modules.
events    the event front end: the frame delta of two sliding windows and its pixel mask.

Inputs change from call to call and sum to zero over four calls, so that a sequence of any length stays bounded.
"""
import math

import torch
import torch.nn.functional as F

from maskedincrementeval_amd import mask_incr_modules as mm
from maskedincrementeval_amd import ops
from maskedincrementeval_amd.e2depth_incr import E2VIDRecurrentIncr
from maskedincrementeval_amd.event_frontend import EventFrames
from maskedincrementeval_amd.evflownet_incr import MultiResUNetRecurrentIncr
from maskedincrementeval_amd.synthetic import MovingEdges, random_events, seed_module_


def _step(name, net, n, h, w, density, dtype, mode, decoder="upsample", state=False):
    return {"name": name, "kind": "step", "net": net, "n": n, "h": h, "w": w, "density": density, "dtype": dtype,
            "mode": mode, "decoder": decoder, "state": state}


def listed():
    return [
        # the smallest frame the tests step a whole network on: what one call costs when the arithmetic is nothing
        _step("e2depth 64x96 call", "e2depth", 1, 64, 96, 0.05, "f32", "call"),
        # the recurrent loop with its state fed back, on a small sensor crop
        _step("e2depth 128x128 state", "e2depth", 1, 128, 128, 0.05, "f32", "call", state=True),
        # the headline frame (346x260 sensor, padded), called plainly frame by frame as the evaluation drivers do
        _step("e2depth 264x352 call", "e2depth", 1, 264, 352, 0.05, "f32", "call"),
        # the same frame as the benchmark runs it: graphs, next step's tile sets planned beside the step
        _step("e2depth 264x352 ahead", "e2depth", 1, 264, 352, 0.05, "f32", "ahead"),
        # an odd frame: planes of 25x35 ... 200x280 (no multiple of a tile), two streams, bf16
        _step("e2depth 2x200x280 bf16 graph", "e2depth", 2, 200, 280, 0.10, "bf16", "graph"),
        # eight VGA event streams in bf16, quiet scene: the batched serving configuration
        _step("e2depth 8x480x640 bf16 ahead", "e2depth", 8, 480, 640, 0.01, "bf16", "ahead"),
        # the same eight streams with a moving camera, called plainly: the largest case
        _step("e2depth 8x480x640 bf16 call", "e2depth", 8, 480, 640, 0.20, "bf16", "call"),
        # optical flow, both decoder kinds, moving edges; many small layers
        _step("evflownet 256 tconv call", "evflownet", 1, 256, 256, 0.03, "f32", "call", decoder="transposed"),
        _step("evflownet 256 up graph", "evflownet", 1, 256, 256, 0.03, "f32", "graph"),
        # the dense refresh of the headline frame
        {"name": "e2depth 264x352 refresh", "kind": "refresh", "net": "e2depth", "n": 1, "h": 264, "w": 352, "dtype": "f32"},
        # one layer of a network assembled from the modules: conv 3x3 64->64, LeakyReLU, ReLU
        {"name": "chain 64ch 132x176", "kind": "chain", "n": 1, "c": 64, "h": 132, "w": 176, "density": 0.05, "dtype": "f32"},
        # 60 000 events of a 346x260 sensor into a 5-bin voxel-grid delta
        {"name": "events 346x260 60k", "kind": "events", "h": 260, "w": 346, "events": 60000, "dtype": "f32"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _side(rng, lo, hi, mult):
    return max(lo, int(_log(rng, lo, hi + mult - 1)) // mult * mult)


def draw(rng):
    kind = rng.choices(["e2depth", "evflownet", "refresh", "chain", "events"], [10, 4, 2, 2, 1])[0]
    dtype = rng.choice(["f32", "bf16"])
    if kind == "events":
        h, w = int(_log(rng, 60, 480)), int(_log(rng, 80, 640))
        return {"kind": kind, "h": h, "w": w, "events": int(_log(rng, 1000, 1000000)), "dtype": dtype}
    if kind == "chain":
        return {"kind": kind, "n": rng.choice([1, 1, 2, 4]), "c": rng.choice([32, 64, 128]), "h": int(_log(rng, 30, 260)),
                "w": int(_log(rng, 40, 340)), "density": round(_log(rng, 0.005, 0.3), 4), "dtype": dtype}
    # three halvings of the plane (four for evflownet) that the decoders undo: sides in multiples of 8 (16)
    mult = 16 if kind == "evflownet" else 8
    most = 8 * 480 * 640 if dtype == "bf16" else 8 * 480 * 640 // 4     # pixels of a step, by what a pixel costs
    if kind == "evflownet":
        most //= 4
    while True:
        n = rng.choice([1, 1, 1, 2, 3, 4, 8])
        h, w = _side(rng, 64, 480, mult), _side(rng, 64, 640, mult)
        if n * h * w <= most:
            break
    if kind == "refresh":
        return {"kind": kind, "net": rng.choice(["e2depth", "e2depth", "evflownet"]) if h % 16 == w % 16 == 0 else "e2depth",
                "n": min(n, 2), "h": h, "w": w, "dtype": dtype}
    net = kind
    mode = rng.choice(["call", "graph", "ahead"])
    c = _step("", net, n, h, w, round(_log(rng, 0.005, 0.2), 4), dtype, mode,
              decoder=rng.choice(["upsample", "transposed"]) if net == "evflownet" else "upsample",
              state=net == "e2depth" and mode == "call" and rng.random() < 0.25)
    del c["name"]
    return c


# ---- inputs --------------------------------------------------------------------------------------------------
_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _blobs(n, h, w, density, gen):
    """(n, 1, h, w) bool: exactly round(density * h * w) active pixels per sample in smooth blobs (white noise under a
    Gaussian of 4 pixels, thresholded)."""
    r, sigma = 12, 4.0
    f = F.pad(torch.rand((n, 1, h, w), generator=gen, device=gen.device), (r, r, r, r), mode="reflect")
    taps = [math.exp(-0.5 * (i / sigma) ** 2) for i in range(-r, r + 1)]
    f = sum(t * f[:, :, i:i + h] for i, t in enumerate(taps))
    f = sum(t * f[:, :, :, i:i + w] for i, t in enumerate(taps))
    keep = max(1, round(density * h * w))
    top = f.reshape(n, -1).topk(keep, dim=1).indices
    m = torch.zeros((n, h * w), dtype=torch.bool, device=gen.device).scatter_(1, top, True)
    return m.reshape(n, 1, h, w)


def _voxel_deltas(c, gen, count):
    """Event-count deltas: Poisson(2) events of random polarity per bin on the blob mask, times 0.1."""
    out = []
    for _ in range(count):
        m = _blobs(c["n"], c["h"], c["w"], c["density"], gen)
        shape = (c["n"], 5, c["h"], c["w"])
        k = torch.poisson(torch.full(shape, 2.0, device=gen.device), generator=gen)
        sign = torch.randint(0, 2, shape, generator=gen, device=gen.device).float() * 2 - 1
        out.append(0.1 * k * sign * m)
    return out


def _edges(c, seed):
    """Generators of the moving-edge event images, with the number of segments that fires about `density`."""
    segments = max(1, round(17 * c["density"] / 0.03 * (c["h"] * c["w"]) ** 0.5 / 256))
    return [MovingEdges(c["h"], c["w"], segments=segments, seed=seed * 64 + b) for b in range(c["n"])]


def _edge_deltas(c, seed, count):
    gens = _edges(c, seed)
    return [torch.cat([g.step()[0] for g in gens], 0) for _ in range(count)]


def _nhwc(t, c):
    return t.to("cuda").to(_DTYPES[c["dtype"]]).contiguous(memory_format=torch.channels_last)


def _cycle(ds):
    """Two deltas and their negatives: four inputs that sum to zero."""
    return ds + [-d for d in ds]


def _network(c):
    planned = {"async_masks": True, "plan_first": True} if c.get("mode") in ("graph", "ahead") else {}
    if c["net"] == "evflownet":
        net = MultiResUNetRecurrentIncr(num_bins=4, decoder=c.get("decoder", "upsample"), **planned)
    else:
        net = E2VIDRecurrentIncr(**planned)
    return seed_module_(net, seed=1).to("cuda").eval()


def _refresh(c, net, x):
    return net.forward_refresh_reservoirs(x) if c["net"] == "evflownet" else net.forward_refresh_reservoirs(x, None)


def _bins(c):
    return 4 if c["net"] == "evflownet" else 5


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    with torch.no_grad():
        if c["kind"] == "events":
            ev = random_events(c["events"], c["w"], c["h"], 0.0, 0.1, seed=int(seed) % (1 << 31))
            frames = EventFrames(c["w"], c["h"], dtype=_DTYPES[c["dtype"]])
            frames.set_events(ev)
            return {"case": c, "frames": frames, "i": 0}
        if c["kind"] == "chain":
            shape = (c["n"], c["c"], c["h"], c["w"])
            conv = seed_module_(mm.nnConvIncr(c["c"], c["c"], 3, 1, 1), seed=2).to("cuda").eval()
            leaky = mm.nnReservedActivation(mm.leaky_relu_op(0.01), refine_mask=False)
            relu = mm.nnReluIncr()
            ins = []
            for _ in range(2):
                m = _blobs(c["n"], c["h"], c["w"], c["density"], gen)
                d = _nhwc(0.2 * torch.randn(shape, generator=gen, device="cuda") * m, c)
                ins.append((d, m.to(torch.uint8)))
            ins += [(-d, m) for d, m in ins]
            x0 = _nhwc(torch.randn(shape, generator=gen, device="cuda"), c)
            relu.forward_refresh_reservoirs(conv.forward_refresh_fused(x0, leaky))
            return {"case": c, "conv": conv, "leaky": leaky, "relu": relu, "ins": ins, "i": 0}
        net = _network(c)
        frame = 0.5 * torch.randn((c["n"], _bins(c), c["h"], c["w"]), generator=gen, device="cuda")
        if c["kind"] == "refresh":
            frames = [_nhwc(frame, c), _nhwc(frame.flip(3), c)]
            _refresh(c, net, frames[1])
            if c["net"] == "evflownet":
                net.states = [None] * net.num_states
            return {"case": c, "net": net, "frames": frames, "i": 0}
        if c["net"] == "evflownet":
            deltas = _edge_deltas(c, int(seed) % (1 << 24), 2)
        else:
            deltas = _voxel_deltas(c, gen, 2)
        s = {"case": c, "net": net, "deltas": _cycle([_nhwc(d, c) for d in deltas]), "prev": None, "i": 0}
        _refresh(c, net, _nhwc(frame, c))
        if c["mode"] == "ahead":
            s["stepper"] = ops.LookaheadStepper("cuda:0")
            _warm_and_capture_halves(s)
        elif c["mode"] == "graph":
            _warm_and_capture(s)
        return s


def _call(s, i):
    c, net = s["case"], s["net"]
    if c["net"] == "evflownet":
        return net([s["deltas"][i], None])
    out = net([s["deltas"][i], None], s["prev"])
    if c["state"]:
        s["prev"] = out[1]
    return out


def _warm_and_capture(s):
    s["graphs"], s["outs"] = [], []
    for i in range(4):
        _call(s, i)
    torch.cuda.synchronize()
    for i in range(4):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            s["outs"].append(_call(s, i))
        s["graphs"].append(g)


def _warm_and_capture_halves(s):
    net, deltas, stepper = s["net"], s["deltas"], s["stepper"]
    compute = lambda i: net.forward_planned([deltas[i % 4], None], i % 2)      # noqa: E731
    plan = lambda i: net.plan_ahead([deltas[i % 4], None], i % 2)              # noqa: E731
    for i in range(4):
        stepper.step(i, lambda: compute(i), lambda: plan(i + 1))
    torch.cuda.synchronize()
    s["graphs"], s["outs"], s["plans"] = [], [], [None] * 4
    for i in range(4):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            s["outs"].append(compute(i))
        s["graphs"].append(g)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            plan(i + 1)
        s["plans"][(i + 1) % 4] = g


# ---- one pass ------------------------------------------------------------------------------------------------
def _outputs(s, r):
    """What the caller of a step gets and what it leaves behind: the prediction deltas and the recurrent state deltas,
    the accumulated cell states and the pre-activations of the predictions."""
    net = s["net"]
    if s["case"]["net"] == "evflownet":
        return {"flow": [p[0] for p in r], "pred": [p.activation.in_res.reservoir for p in net.preds]}
    pred, states = r
    u = net.unetrecurrent
    return {"image": pred[0], "h": [st[0][0] for st in states], "c": [st[1][0] for st in states],
            "cell": [e.recurrent_block.cell_res.reservoir for e in u.encoders], "pred": u.activation.in_res.reservoir}


def run(state):
    s, c = state, state["case"]
    i = s["i"]
    s["i"] = i + 1
    with torch.no_grad():
        if c["kind"] == "events":
            t0 = 0.005 * (i % 8)
            return s["frames"].delta(t0, t0 + 0.01)
        if c["kind"] == "chain":
            d, m = s["ins"][i % 4]
            out, ts = s["relu"](s["conv"].forward_fused([d, m], s["leaky"]))
            return {"out": out, "mask": ts.pixmask, "leaky": s["leaky"].in_res.reservoir, "relu": s["relu"].in_res.reservoir}
        if c["kind"] == "refresh":
            if c["net"] == "evflownet":
                s["net"].states = [None] * s["net"].num_states      # a new sequence
                flow = _refresh(c, s["net"], s["frames"][i % 2])
                return {"flow": flow, "states": list(s["net"].states)}
            pred, states = _refresh(c, s["net"], s["frames"][i % 2])
            return {"image": pred, "states": [list(st) for st in states]}
        if c["mode"] == "call":
            return _outputs(s, _call(s, i % 4))
        if c["mode"] == "graph":
            s["graphs"][i % 4].replay()
        else:
            s["stepper"].step(i, s["graphs"][i % 4].replay, s["plans"][(i + 1) % 4].replay)
        return _outputs(s, s["outs"][i % 4])


# ---- what a pass cannot do without ---------------------------------------------------------------------------
def _reach(m, k, s=1):
    return F.max_pool2d(m, k, s, k // 2)


def _grow(m, k):
    """Pixels of the doubled plane that a bilinear up-sampling and a k x k conv reach."""
    return _reach(F.interpolate(_reach(m, 3), scale_factor=2), k)


class _Count:
    def __init__(self, es):
        self.es, self.bytes, self.flops = es, 0.0, 0.0

    def conv(self, m_out, cin, cout, k, reservoir=True, taps=None):
        """A conv over the active pixels of m_out: its products, its filter read once, its reservoir read and written."""
        a = float(m_out.sum())
        t = k * k if taps is None else taps
        self.flops += 2.0 * a * cin * cout * t
        self.bytes += cin * cout * k * k * self.es + (8.0 * a * cout if reservoir else 0.0)

    def move(self, m, c, size):
        self.bytes += float(m.sum()) * c * size


def _e2depth_work(w, m0):
    w.bytes += m0.numel() * 5 * w.es                         # the frame or delta itself
    m = _reach(m0, 5)
    w.conv(m, 5, 32, 5)
    head, blocks, ch = m, [], 32
    for _ in range(3):
        m = _reach(m, 5, 2)
        w.conv(m, ch, 2 * ch, 5)
        ch *= 2
        m = _reach(m, 3)
        w.conv(m, ch, 4 * ch, 3)
        w.move(m, ch, 8 + 4 + 2 * w.es)                       # cell reservoir, previous cell, h and c handed out
        blocks.append(m)
    for _ in range(4):
        m = _reach(m, 3)
        w.conv(m, ch, ch, 3)
    for b in reversed(blocks):
        m = _grow(torch.maximum(m, b), 5)
        w.conv(m, ch, ch // 2, 5)
        ch //= 2
    m = torch.maximum(m, head)
    w.conv(m, 2 * ch, 1, 1)
    w.move(m, 1, w.es)


def _evflownet_work(w, m0, transposed):
    w.bytes += m0.numel() * 4 * w.es
    m, blocks, ch = m0, [], 4
    for cout in (64, 128, 256, 512):
        m = _reach(m, 3, 2)
        w.conv(m, ch, cout, 3)
        m = _reach(m, 3)
        w.conv(m, cout, 2 * cout, 3)
        blocks.append(m)
        ch = cout
    for _ in range(4):
        m = _reach(m, 3)
        w.conv(m, ch, ch, 3)
    lead = 0
    for b, cout in zip(reversed(blocks), (256, 128, 64, 32)):
        m = torch.maximum(m, b)
        m = _reach(F.interpolate(m, scale_factor=2), 3) if transposed else _grow(m, 3)
        w.conv(m, lead + 2 * ch, cout, 3, taps=9 / 4 if transposed else None)
        w.conv(m, cout, 2, 1)
        w.move(m, 2, w.es)
        ch, lead = cout, 2


def work(case):
    c = case
    es = 2 if c["dtype"] == "bf16" else 4
    w = _Count(es)
    if c["kind"] == "events":
        p = (c["h"] + 4) * (c["w"] + 6)                       # reflection padding of 2 and 3 pixels a side
        return {"bytes": 32.0 * c["events"] + p * (5 * es + 1), "flops": 0.0}
    gen = torch.Generator().manual_seed(1)
    if c["kind"] == "refresh":
        m0 = torch.ones((c["n"], 1, c["h"], c["w"]))
    elif c.get("net") == "evflownet":
        m0 = torch.cat([g.step()[1] for g in _edges(c, 1)], 0).float()
    else:
        m0 = _blobs(c["n"], c["h"], c["w"], c["density"], gen).float()
    if c["kind"] == "chain":
        m = _reach(m0, 3)
        w.conv(m, c["c"], c["c"], 3)
        w.move(m0, c["c"], es)
        w.move(m, c["c"], 8 + es)                             # second reservoir, delta handed out
        w.bytes += 2.0 * m.numel()                            # masks
    elif c["net"] == "evflownet":
        _evflownet_work(w, m0, c.get("decoder") == "transposed")
    else:
        _e2depth_work(w, m0)
    return {"bytes": w.bytes, "flops": w.flops}


def tolerance(case):
    if case["dtype"] == "bf16":
        # deltas are rounded to 8 bits of mantissa after every layer
        return {"rel": 1e-2, "max": 0.5, "differ": 2e-3}
    if case["kind"] in ("chain", "events"):
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}
    if case["kind"] == "refresh":
        return {"rel": 1e-5, "max": 1e-3}
    # fifteen layers of 32-bit sums whose deltas are differences of activations: sums taken in another order alone
    # differ by up to 5e-5
    return {"rel": 1e-4, "max": 5e-3}
