"""GPU parity of EVFlowNet-incr (ConvGRU encoders, concat skips, multi-scale flow heads) against the
CPU oracle, for both decoder kinds, through the C ABI.  fp32: rtol 1e-4, atol 1e-5."""
import numpy as np
import pytest
import torch

from maskedincrementeval_amd import ops
from maskedincrementeval_amd.evflownet_incr import ConvGRUIncr, MultiResUNetRecurrentIncr
from maskedincrementeval_amd.synthetic import MovingEdges, gaussian_delta, seed_module_
from oracle import mask_oracle as mo
from tolerances import BF16_RTOL, bf16_atol
from oracle.evflownet_oracle import EVFlowNetOracle, _ConvGRU
import mask_chain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cl(t):
    return t.to(DEV).contiguous(memory_format=torch.channels_last)


def _close(got, ref, what="", rtol=1e-4, atol=1e-5):
    got = got.detach().cpu()
    err = (got - ref).abs().max().item()
    assert torch.allclose(got, ref, rtol=rtol, atol=atol), "%s max|diff| = %.3e" % (what, err)


@pytest.mark.parametrize("fuse,stacked,one_launch", [(True, True, "never"), (True, True, "always"), (True, True, "in turn"), (True, False, "never"),
                                                     (False, False, "never")])
@pytest.mark.parametrize("c", [64, 32, 12])
def test_convgru_module_matches_oracle(fuse, stacked, one_launch, c):
    # stacked: both gate convs as one conv of 2*hid channels + mie_convgru_gates_incr, or (one_launch) mie_conv_gru_masked, on the
    # kernel for planes of few tiles (c = 64) and the general one (32); c = 12 keeps the conv off the matrix-core path and the gate kernel
    # on 4-channel vectors
    n, h, w = 1, 20, 28
    cell = seed_module_(ConvGRUIncr(c, c, 3, fuse=fuse, stacked=stacked), 41).to(DEV).eval()
    params = {"g." + k: v for k, v in cell.state_dict().items()}
    ref = _ConvGRU({k: v.cpu() for k, v in params.items()}, "g", c)
    x = torch.randn(n, c, h, w, generator=torch.Generator().manual_seed(42))
    with torch.no_grad():
        hd, _ = cell.forward_refresh_reservoirs(_cl(x), None)
    _close(hd, ref.refresh(x, None), "refresh")
    for step in range(4):
        d, m = gaussian_delta(n, c, h, w, 0.08, 0.3, seed=4300 + step)
        cell.one_launch = one_launch == "always" or (one_launch == "in turn" and step % 2 == 0)
        with torch.no_grad():
            dh, _ = cell([_cl(d), m.to(DEV)], None)
        torch.cuda.synchronize()
        _close(dh[0], ref.incr(d), "step %d" % step)
        # clean-delta invariant: nothing outside the 3x3 footprint of the input mask
        foot = torch.from_numpy(mo.footprint_conv(m[:, 0].numpy(), 3, 1, 1)).bool().unsqueeze(1)
        assert torch.count_nonzero(dh[0].cpu() * (~foot)) == 0
    assert ("gru_gates" in str(list(cell._ib().keys()))) == (fuse and stacked and (c == 12 or one_launch != "always"))


def _run(decoder, h, w, steps, edges, fuse=True):
    model = seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder=decoder, fuse=fuse), seed=51).to(DEV).eval()
    oracle = EVFlowNetOracle(model.state_dict(), decoder=decoder)
    x0 = torch.randn(1, 4, h, w, generator=torch.Generator().manual_seed(52)) * 0.5
    with torch.no_grad():
        acc = [p.clone() for p in model.forward_refresh_reservoirs(_cl(x0))]
    acc_ref = oracle.refresh(x0)
    for a, b in zip(acc, acc_ref):
        _close(a, b, "refresh")
    gen = MovingEdges(h, w, seed=53) if edges else None
    x = x0.clone()
    prev_lists, sets_checked = {}, 0
    for step in range(steps):
        if edges:
            d, m = gen.step()
        else:
            d, m = gaussian_delta(1, 4, h, w, 0.05, 0.3, seed=5400 + step)
        with torch.no_grad(), mask_chain.BuildRecorder() as rec:
            preds = model([_cl(d), None])           # the reference drivers pass no mask
        torch.cuda.synchronize()
        ref = oracle.incr(d)
        for s, (a, b) in enumerate(zip(preds, ref)):
            _close(a[0], b, "step %d scale %d" % (step, s))
        acc = [a + p[0] for a, p in zip(acc, preds)]
        acc_ref = [a + b for a, b in zip(acc_ref, ref)]
        x = x + d
        pm = mo.pixel_mask(d.numpy(), 0.0)
        enc0 = model.encoders[0].conv.conv2d._tile_set("out_act" if fuse else "out", 1, h // 2, w // 2, torch.device(DEV))
        want = mo.tile_list(mo.footprint_conv(pm, 3, 2, 1))
        assert np.array_equal(enc0.active_tiles().cpu().numpy(), want)
        if fuse:
            # every tile set of the step in situ (pixel mask, ascending tile list, stale list) against the chained
            # footprints of the input pixel mask, and the named layers against the chain of the network definition
            seeds = {model._pix_buf("input", 1, h, w, torch.device(DEV)).data_ptr(): pm}
            sets_checked += mask_chain.check_recorded_builds(rec.calls, seeds, prev_lists, "step %d" % step)
            sets_checked += mask_chain.check_evflownet_layers(model, pm, "step %d" % step)
    assert not fuse or sets_checked >= 30 * steps
    for a, b in zip(acc, acc_ref):
        _close(a, b, "accumulated")
    return model, acc, x


@pytest.mark.parametrize("decoder", ["upsample", "transposed"])
@pytest.mark.parametrize("fuse", [True, False])
def test_evflownet_small_matches_oracle(decoder, fuse):
    _run(decoder, 64, 96, steps=3, edges=False, fuse=fuse)


@pytest.mark.parametrize("decoder", ["upsample", "transposed"])
def test_evflownet_config4_moving_edges_and_dense_identity(decoder):
    # benchmark configuration 4: 1x4x256x256, moving-edge deltas (~3 % density); transposed-conv decoders as the
    # configuration words it, up-sampling decoders as the reference file has them
    model, acc, x = _run(decoder, 256, 256, steps=3, edges=True)
    _dense_identity(decoder, acc, x)


def _dense_identity(decoder, acc, x):
    fresh = seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder=decoder), seed=51).to(DEV).eval()
    with torch.no_grad():
        dense = fresh.forward_refresh_reservoirs(_cl(x))
    for a, b in zip(acc, dense):
        _close(a, b.cpu(), "refresh + increments vs dense")


@pytest.mark.parametrize("decoder", ["upsample", "transposed"])
def test_evflownet_config4_100_steps_of_accumulation(decoder):
    # benchmark configuration 4 as it is worded: 100 moving-edge frames at 1x4x256x256 accumulated into the same
    # reservoirs; every step and flow scale against the CPU oracle, every tile set of every step against the mask
    # oracle, and refresh + the 100 increments == dense forward on the accumulated input
    model, acc, x = _run(decoder, 256, 256, steps=100, edges=True)
    _dense_identity(decoder, acc, x)


def test_evflownet_50_steps_of_accumulation():
    # 50 moving-edge frames accumulated into the same reservoirs: parity per step and scale, and refresh + the 50
    # increments == dense forward on the accumulated input; reduced frame (64x96: bottleneck planes of 4x6 pixels,
    # every small-plane form of the conv runs)
    model, acc, x = _run("upsample", 64, 96, steps=50, edges=True)
    fresh = seed_module_(MultiResUNetRecurrentIncr(num_bins=4), seed=51).to(DEV).eval()
    with torch.no_grad():
        dense = fresh.forward_refresh_reservoirs(_cl(x))
    for a, b in zip(acc, dense):
        _close(a, b.cpu(), "refresh + 50 increments vs dense")


@pytest.mark.parametrize("decoder", ["upsample", "transposed"])
def test_evflownet_bf16_matches_fp32_oracle(decoder):
    # bf16 deltas and weights, fp32 reservoirs: every flow scale within rtol 2e-2 of its range (tanh output)
    h, w = 64, 96
    bf = torch.bfloat16
    model = seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder=decoder), seed=51).to(DEV).eval()
    oracle = EVFlowNetOracle(model.state_dict(), decoder=decoder)
    x0 = torch.randn(1, 4, h, w, generator=torch.Generator().manual_seed(52)) * 0.5
    with torch.no_grad():
        acc = [p.float().clone() for p in model.forward_refresh_reservoirs(_cl(x0).to(bf))]
    acc_ref = oracle.refresh(x0)
    for a, b in zip(acc, acc_ref):
        _close(a, b, "refresh", rtol=BF16_RTOL, atol=bf16_atol(b))
    for step in range(3):
        d, m = gaussian_delta(1, 4, h, w, 0.05, 0.3, seed=5400 + step)
        with torch.no_grad():
            preds = model([_cl(d).to(bf), None])
        torch.cuda.synchronize()
        ref = oracle.incr(d)
        for s, (a, b) in enumerate(zip(preds, ref)):
            assert a[0].dtype == bf
            # a step's flow delta is a 1x1 conv over up to 256 channels of bf16-rounded deltas about ten times
            # its own size: the cancellation multiplies the relative error (measured 2 - 12 roundoffs of the
            # delta's largest value, most at the coarsest scale where the delta is smallest); 16 allowed.
            # The accumulated flow below is held to 3 roundoffs of its range.
            _close(a[0].float(), b, "step %d scale %d" % (step, s), rtol=BF16_RTOL, atol=bf16_atol(b, 16.0))
        acc = [a + p[0].float() for a, p in zip(acc, preds)]
        acc_ref = [a + b for a, b in zip(acc_ref, ref)]
    for a, b in zip(acc, acc_ref):
        _close(a, b, "accumulated", rtol=BF16_RTOL, atol=bf16_atol(b))


@pytest.mark.parametrize("decoder", ["upsample", "transposed"])
def test_evflownet_planning_stream_and_pass_reproduce_inline_planning(decoder):
    # tile sets built on the planning stream in a planning pass, replayed from a HIP graph, against inline
    # planning with eager launches: same kernels over the same tiles, so every flow scale agrees bit for bit
    h, w, steps = 64, 96, 7
    a = seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder=decoder, async_masks=True, plan_first=True),
                     seed=51).to(DEV).eval()
    s = seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder=decoder), seed=51).to(DEV).eval()
    x0 = torch.randn(1, 4, h, w, generator=torch.Generator().manual_seed(52)) * 0.5
    deltas = [_cl(gaussian_delta(1, 4, h, w, 0.03 + 0.03 * (i % 3), 0.3, seed=5600 + i)[0]) for i in range(steps)]
    static_in = _cl(torch.zeros(1, 4, h, w))
    with torch.no_grad():
        a.forward_refresh_reservoirs(_cl(x0))
        s.forward_refresh_reservoirs(_cl(x0))
        refs = [[p[0].clone() for p in s([d, None])] for d in deltas]
        got, g, g_out = [], None, None
        for i, d in enumerate(deltas):
            static_in.copy_(d)
            if i == 2:
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    g_out = [p[0] for p in a([static_in, None])]
            if g is not None:
                g.replay()
                got.append([t.clone() for t in g_out])
            else:
                got.append([p[0].clone() for p in a([static_in, None])])
        torch.cuda.synchronize()
    for i in range(steps):
        for sc, (x, y) in enumerate(zip(got[i], refs[i])):
            assert torch.equal(x, y), "step %d scale %d max|diff| = %.3e" % (i, sc, (x - y).abs().max().item())


def test_concat_layers_refuse_the_planning_stream():
    # the un-fused transposed-conv decoders concatenate with torch ops on the compute stream, which would read
    # pixel masks the planning stream is still writing: refused, and the planner is unwound
    h, w = 32, 48
    m = seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder="transposed", async_masks=True, fuse=False),
                     seed=51).to(DEV).eval()
    with torch.no_grad():
        m.forward_refresh_reservoirs(_cl(torch.randn(1, 4, h, w, generator=torch.Generator().manual_seed(1))))
        with pytest.raises(NotImplementedError, match="asynchronous mask planning"):
            m([_cl(gaussian_delta(1, 4, h, w, 0.05, 0.3, seed=2)[0]), None])
    assert ops._planner is None and ops._phase is None


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("decoder", ["transposed", "upsample"])
@pytest.mark.parametrize("x3", ["f16x2", "bf16x3"])
def test_a_step_planned_under_one_setting_runs_under_another(x3, decoder, dtype, monkeypatch):
    # ops.f32_matmul is chosen per call, also between a plan and its step: which tile sets the step needs follows it.  (Deltas are
    # differences of values of order one: sums in another order, all that a plan of the other setting changes, show as some 1e-7)
    h, w = 64, 96
    a, b = (seed_module_(MultiResUNetRecurrentIncr(num_bins=4, decoder=decoder), seed=3).to(DEV).eval() for _ in range(2))
    gen = MovingEdges(h, w, seed=5)
    native = "native"
    with torch.no_grad():
        x0 = _cl(torch.randn(1, 4, h, w, generator=torch.Generator().manual_seed(1))).to(dtype)
        a.forward_refresh_reservoirs(x0), b.forward_refresh_reservoirs(x0)
        for i, (planned, run) in enumerate([(x3, x3), (x3, native), (native, native), (native, x3), (native, native), (native, x3), (x3, native), (x3, x3)]):
            d = _cl(gen.step()[0]).to(dtype)
            monkeypatch.setattr(ops, "f32_matmul", planned)
            a.plan_ahead([d, None], i % 2)
            monkeypatch.setattr(ops, "f32_matmul", run)
            got, want = a.forward_planned([d, None], i % 2), b([d, None])
            torch.cuda.synchronize()
            for (g, _), (v, _) in zip(got, want):
                assert (g - v).abs().max() <= (2e-6 if dtype == torch.float32 else 0), i
