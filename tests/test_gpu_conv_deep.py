"""Convs on planes of few tiles in one launch without a workspace (csrc/mie_conv_deep.hip) against fp64, beside the split form."""
import pytest
import torch
import torch.nn.functional as F

from maskedincrementeval_amd import _lib, ops
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.synthetic import gaussian_delta, he_normal_conv_weight

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(t):
    return ops.as_nhwc(t.to(DEV).contiguous(memory_format=torch.channels_last))


# chunks of 32 channels: fewer, as many and more than the 8 waves, 1, 2, 4 or 8 of them a chunk, of one input or two; planes of one
# pixel, of less than two rows or columns of a tile, of whole tiles; the last shapes at which two rows a workgroup, four, and the
# form itself are taken (256 workgroups), and the first beyond
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k,s,n,c1,c2,cout,h,w,pad", [(3, 1) + shape for shape in [
    (1, 64, 0, 32, 1, 1, 1), (2, 64, 64, 64, 3, 2, 1), (1, 192, 0, 32, 5, 9, 1), (1, 256, 128, 96, 13, 11, 0), (1, 320, 0, 32, 9, 7, 2),
    (1, 512, 0, 64, 16, 17, 1), (3, 256, 64, 32, 12, 8, 3), (1, 128, 0, 256, 16, 16, 1), (1, 64, 0, 256, 16, 24, 1),
    (1, 64, 64, 512, 16, 16, 1), (1, 64, 0, 512, 16, 24, 1), (2, 64, 0, 512, 16, 16, 1), (1, 128, 0, 512, 24, 24, 1),
    (1, 64, 0, 256, 32, 32, 1), (1, 96, 64, 256, 31, 29, 1), (1, 128, 64, 256, 31, 29, 1), (1, 64, 0, 256, 32, 33, 1), (1, 512, 32, 512, 16, 25, 1)]] + [(5, 2) + shape for shape in [
        (1, 32, 0, 32, 1, 1, 2), (1, 32, 0, 64, 1, 1, 2), (2, 64, 32, 64, 6, 5, 2), (1, 96, 0, 32, 17, 33, 1), (1, 96, 0, 64, 17, 33, 1), (1, 128, 0, 256, 16, 24, 2), (1, 32, 0, 64, 127, 128, 2),
        (1, 64, 0, 128, 64, 64, 2), (1, 32, 0, 64, 136, 128, 2)]] + [(3, 2) + shape for shape in [
        (1, 64, 0, 32, 1, 1, 1), (2, 64, 32, 64, 5, 18, 1), (1, 64, 32, 48, 19, 21, 1), (1, 128, 0, 512, 15, 16, 1), (1, 256, 64, 128, 31, 29, 1), (1, 64, 0, 256, 64, 64, 1),
        (1, 64, 32, 64, 128, 127, 0), (1, 64, 0, 256, 64, 66, 1)]])
def test_whole_contraction_in_a_workgroup(k, s, n, c1, c2, cout, h, w, pad, dtype):
    cin, bf = c1 + c2, dtype == torch.bfloat16
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    wt = q(he_normal_conv_weight(cout, cin, k, 21))
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    ho, wo = ops.conv_out_size(h, w, k, s, pad)
    ts = TileMask(n, ho, wo, DEV)
    tiles = ts.capacity
    takes = _lib.lib().mie_conv_needs_no_workspace(k, s, c1, c2, cout, tiles, _lib.DTYPE_BF16 if bf else _lib.DTYPE_F32_BF16X3)
    # (bf16 of other chunks of channels, and slabs of columns, than the matrix cores take: the VALU, not named)
    whole = lambda c, m: c1 % c == 0 and c2 % c == 0 and cout % m == 0
    matrix = whole(64, 32) or (s == 2 and whole(32, 64)) if bf else whole(32, 16 if (k, s) == (3, 2) else 32)
    assert takes == (matrix and tiles * (cout // 16) <= 256 and not (not bf and (k, s) == (3, 1) and tiles * (cout // 16) > 128 and cin > 512))
    outs = [ops.new_nhwc(n, cout, ho, wo, DEV, dtype) for _ in range(2)]
    r0 = torch.randn(n, cout, ho, wo, generator=torch.Generator().manual_seed(5))
    ress = [_dev(r0) for _ in range(2)]
    ref = r0.double()
    tol = torch.zeros_like(ref)
    split = torch.full((ops.SPLIT_WORKSPACE_BYTES // 4,), float("nan"), device=DEV)
    err = [0.0, 0.0]
    for step, dens in enumerate((0.3, 0.04, 1.0)):
        d, m = gaussian_delta(n, cin, h, w, dens, 0.5, seed=300 + step)
        d = q(d)
        live = F.max_pool2d(F.pad(m.float(), (pad,) * 4), k, s) > 0
        add = q(gaussian_delta(n, cout, ho, wo, 1.0, 0.3, seed=400 + step)[0]) * live if step else None
        dm = m.to(DEV)
        x = torch.where(m.bool(), d, torch.full((), float("nan")))       # what an inactive pixel holds is not read
        x1, x2 = _dev(x[:, :c1]).to(dtype), _dev(x[:, c1:]).to(dtype) if c2 else None
        ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_CONV, k, s, pad, ts)
        sums = F.conv2d(d.double(), wt.double(), padding=pad, stride=s) + (0 if add is None else add.double())
        bound = F.conv2d(d.double().abs(), wt.double().abs(), padding=pad, stride=s) + (0 if add is None else add.double().abs())
        # three fp32 roundings of sum |x||w|, as for the other forms, and the reservoir's own, step upon step
        before, tol = tol, tol + 4e-7 * bound + 2.0 ** -23 * (ref.abs() + sums.abs())
        for i, ws in enumerate((None, split)):
            ops.conv_masked(x1, dm, x2, None if x2 is None else dm, filt, k, s, pad, ts, outs[i], ress[i], _lib.ACT_RELU, 0.0,
                            _lib.PATH_MFMA if takes and ws is None else _lib.PATH_AUTO, None if add is None else _dev(add).to(dtype), workspace=ws)
            torch.cuda.synchronize()
            off = (ress[i].cpu().double() - (ref + sums)).abs()
            assert (off <= tol).all(), (step, i)
            want = (ref + sums).clamp(min=0) - ref.clamp(min=0)
            got = outs[i].cpu().double()
            assert ((got - want).abs() <= (before + tol) * (1 + 2.0 ** -8) + (2.0 ** -8 if bf else 0.0) * want.abs()).all(), (step, i)
            assert not got[~live.expand_as(got)].any()
            err[i] += off.norm().item()
        ref = ref + sums
    assert err[0] <= 1.1 * err[1], err
    if takes:
        y, res = ops.new_nhwc(n, cout, ho, wo, DEV, dtype), ops.new_nhwc(n, cout, ho, wo, DEV)
        bias = torch.randn(cout, generator=torch.Generator().manual_seed(6))
        every = TileMask(n, ho, wo, DEV)
        ops.build_mask_tiles(None, None, n, ho, wo, _lib.FOOT_CONV, 1, 1, 0, every)
        ops.conv_refresh(_dev(d[:, :c1]).to(dtype), _dev(d[:, c1:]).to(dtype) if c2 else None, filt, bias.to(DEV), k, s, pad, every, y, res)
        want = F.conv2d(d.double(), wt.double(), bias.double(), padding=pad, stride=s)
        assert ((res.cpu().double() - want).abs() <= 4e-7 * bound + 2.0 ** -23 * want.abs()).all()


def _split_workspace():
    return torch.full((ops.SPLIT_WORKSPACE_BYTES // 4,), float("nan"), device=DEV)


@pytest.mark.parametrize("k", [3, 5])
def test_infinite_deltas_pass_the_strided_form(k):
    # as through the split form, whose sums are taken again in fp32 where they are not finite
    c, cout, h, w = 64, 32, 9, 12
    wt = he_normal_conv_weight(cout, c, k, 4)
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    x = torch.randn(1, c, h, w, generator=torch.Generator().manual_seed(1))
    x[0, 3, 4, 5], x[0, 7, 0, 0] = float("inf"), 3.4e38
    ts = TileMask(1, 5, 6, DEV)
    ops.build_mask_tiles(None, None, 1, 5, 6, _lib.FOOT_CONV, 1, 1, 0, ts)
    got = []
    for ws in (None, _split_workspace()):
        out = ops.new_nhwc(1, cout, 5, 6, DEV)
        ops.conv_masked(_dev(x), None, None, None, filt, k, 2, k // 2, ts, out, workspace=ws)
        got.append(out.cpu())
    fin = torch.isfinite(got[1])
    assert (torch.isfinite(got[0]) == fin).all() and not fin.all() and torch.equal(got[0].isnan(), got[1].isnan())
    ref = F.conv2d(x.double(), wt.double(), padding=k // 2, stride=2)
    bound = F.conv2d(x.double().abs(), wt.double().abs(), padding=k // 2, stride=2)
    assert ((got[0].double() - ref).abs()[fin] <= (4e-7 * bound)[fin]).all()


# one and two inputs of 2, 3, 8 and 16 chunks; two, four and eight rows a workgroup (256 workgroups each), and planes of a few pixels
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,hid,two,h,w", [(1, 64, False, 1, 1), (2, 64, True, 3, 9), (1, 64, True, 32, 31), (1, 128, True, 16, 16), (1, 128, False, 13, 24),
                                           (1, 256, True, 8, 8), (1, 256, False, 8, 12), (1, 256, True, 16, 15)])
def test_gates_conv_in_one_launch(n, hid, two, h, w, dtype):
    bf = dtype == torch.bfloat16
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    gen = torch.Generator().manual_seed(11)
    cin = 2 * hid if two else hid
    wt = q(he_normal_conv_weight(4 * hid, cin, 3, 31))
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    ts = TileMask(n, h, w, DEV)
    assert _lib.lib().mie_conv_gates_needs_no_workspace(hid, cin - hid, hid, ts.capacity, _lib.DTYPE_BF16 if bf else _lib.DTYPE_F32_BF16X3)
    r0, cp0, cc0 = (torch.randn(n, c, h, w, generator=gen) for c in (4 * hid, hid, hid))
    err = [0.0, 0.0]
    x, m = gaussian_delta(n, cin, h, w, 0.2, 0.5, seed=61)
    dp, mp = gaussian_delta(n, hid, h, w, 0.3, 0.3, seed=62)
    x, dp = q(x), q(dp)
    live = F.max_pool2d(m.float(), 3, 1, 1) > 0
    dm, dpm = m.to(DEV), (mp.bool() & live).to(torch.uint8).to(DEV)
    dp = dp * dpm.cpu() if two else torch.zeros_like(dp)
    x1 = torch.where(m.bool(), x, torch.full((), float("nan")))
    sums = F.conv2d(x.double(), wt.double(), padding=1)
    bound = 4e-7 * F.conv2d(x.double().abs(), wt.double().abs(), padding=1) + 2.0 ** -23 * (r0.double().abs() + sums.abs())
    for i, kw in enumerate((dict(one_launch=True), dict(workspace=_split_workspace()))):
        ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_CONV, 3, 1, 1, ts)
        gr, cpr, cr = _dev(r0), _dev(cp0), _dev(cc0)
        dh, dc = (ops.new_nhwc(n, hid, h, w, DEV, dtype) for _ in range(2))
        ops.conv_gates_incr(_dev(x1[:, :hid]).to(dtype), dm, _dev(x1[:, hid:]).to(dtype) if two else None, dm if two else None, filt, ts, gr,
                            _dev(dp).to(dtype) if two else None, dpm if two else None, cpr, cr, dh, dc, **kw)
        torch.cuda.synchronize()
        off = (gr.cpu().double() - r0.double() - sums).abs()
        assert (off <= bound).all(), i
        err[i] = off.norm().item()
        # the chain, from the gates it left: each of its evaluations within 2e-7, none multiplied by more than |cell values| + 1
        g0, g1 = (t.double().reshape(n, hid, 4, h, w).unbind(2) for t in (r0, gr.cpu()))
        act = lambda g: (g[0].sigmoid(), g[1].sigmoid(), g[2].sigmoid(), g[3].tanh())
        (i0, f0, o0, t0), (i1, f1, o1, t1) = act(g0), act(g1)
        c0, p0, p1 = cc0.double(), cp0.double(), cp0.double() + dp.double()
        want_c = (i1 * t1 - i0 * t0) + (f1 * p1 - f0 * p0)
        want_h = o1 * (c0 + want_c).tanh() - o0 * c0.tanh()
        tol = 2e-6 * (2 + p1.abs() + p0.abs() + c0.abs())
        for got, want in ((dc, want_c), (dh, want_h)):
            got = got.cpu().double()
            assert ((got - want).abs()[live.expand_as(got)] <= (tol + (2.0 ** -8 * want.abs() if bf else 0))[live.expand_as(got)]).all(), i
            assert not got[~live.expand_as(got)].any()
        assert ((cr.cpu().double() - c0 - want_c * live).abs() <= tol).all() and ((cpr.cpu().double() - p1).abs() <= 1e-6 * (1 + p1.abs())).all()
    assert err[0] <= 1.1 * err[1], err


# sources of one pixel to those of 256 workgroups with two, four and (bf16) eight rows; 2, 3, 4 and 8 chunks; one source or two
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,cout,two,h,w", [(1, 64, 32, True, 1, 1), (2, 128, 64, True, 3, 5), (1, 64, 96, False, 9, 7), (1, 128, 64, True, 16, 16), (1, 128, 32, True, 31, 32),
                                              (1, 64, 32, True, 64, 32), (1, 128, 64, False, 32, 31)])
def test_up_sampling_conv_in_one_launch(n, c, cout, two, h, w, dtype):
    bf = dtype == torch.bfloat16
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    wt = q(he_normal_conv_weight(cout, c, 5, 41))
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    H, W = 2 * h, 2 * w
    up, ts = TileMask(n, H, W, DEV), TileMask(n, H, W, DEV)
    takes = _lib.lib().mie_upconv_needs_no_workspace(c, cout, ts.capacity, _lib.DTYPE_BF16 if bf else _lib.DTYPE_F32_BF16X3)
    assert takes == (ts.capacity * (cout // 16) <= (256 if bf else 128))
    r0 = torch.randn(n, cout, H, W, generator=torch.Generator().manual_seed(5))
    (a, ma), (b, mb) = (gaussian_delta(n, c, h, w, d, 0.5, seed=70 + i) for i, d in enumerate((0.3, 0.1)))
    a, b = q(a), q(b)
    z = (a.double() + b.double() if two else a.double())
    big = lambda t: F.interpolate(t, scale_factor=2, mode="bilinear", align_corners=False)
    x = big(z)
    live = F.max_pool2d(F.max_pool2d(F.interpolate(F.max_pool2d((ma | mb if two else ma).float(), 3, 1, 1), scale_factor=2), 3, 1, 1), 5, 1, 2) > 0
    sums = F.conv2d(x, wt.double(), padding=2)
    # three fp32 roundings of sum |x||w| and three of the blended values'; bf16: these rounded to 8 bits
    bound = (4e-7 + 4e-7 + (2.0 ** -8 if bf else 0)) * F.conv2d(big((a.abs() + b.abs() if two else a.abs()).double()), wt.double().abs(), padding=2)
    nan = lambda t, m: torch.where(m.bool(), t, torch.full((), float("nan")))
    da, db = _dev(nan(a, ma)).to(dtype), _dev(nan(b, mb)).to(dtype) if two else None
    dma, dmb = ma.to(DEV), mb.to(DEV) if two else None
    err = []
    for ws in (None, _split_workspace()):
        ops.build_mask_tiles(dma, dmb, n, h, w, _lib.FOOT_UP2X, 0, 0, 0, up)
        ops.build_mask_tiles(up, None, n, H, W, _lib.FOOT_CONV, 5, 1, 2, ts)
        out, res = ops.new_nhwc(n, cout, H, W, DEV, dtype), _dev(r0)
        ops.upconv_masked(da, dma, db, dmb, filt, 5, 2, ts, out, res, _lib.ACT_RELU, 0.0, workspace=ws)
        torch.cuda.synchronize()
        off = (res.cpu().double() - r0.double() - sums).abs()
        assert (off <= bound + 2.0 ** -23 * (r0.double().abs() + sums.abs())).all()
        want = (r0.double() + sums).clamp(min=0) - r0.double().clamp(min=0)
        got = out.cpu().double()
        assert ((got - want).abs() <= bound + 2.0 ** -22 * (r0.double().abs() + sums.abs()) + (2.0 ** -8 if bf else 0.0) * want.abs()).all()
        assert not got[~live.expand_as(got)].any()
        err.append(off.norm().item())
    assert err[0] <= 1.1 * err[1], err


# layers of more input channels than the one-launch form is the faster one for: what a call without a word on workspaces gives is the
# split form's result (3x3 stride 2 in fp32: the fp32 instruction's), whatever the shared workspace holds
@pytest.mark.parametrize("kind,dtype,c1,c2", [("c31", torch.float32, 512, 64), ("c31", torch.bfloat16, 1024, 576), ("c32", torch.float32, 256, 256), ("c32", torch.bfloat16, 960, 0),
                                              ("c52", torch.float32, 192, 0), ("c52", torch.bfloat16, 256, 256), ("gates", torch.float32, 640, 64),
                                              ("gates", torch.bfloat16, 1088, 1024), ("up", torch.bfloat16, 512, 0)])
def test_layers_of_many_channels_are_split(kind, dtype, c1, c2):
    n, h, w, cout = 1, 11, 13, 64
    k, s = {"c31": (3, 1), "c32": (3, 2), "c52": (5, 2), "gates": (3, 1), "up": (5, 1)}[kind]
    code = _lib.DTYPE_BF16 if dtype == torch.bfloat16 else _lib.DTYPE_F32_BF16X3
    ho, wo = (2 * h, 2 * w) if kind == "up" else ops.conv_out_size(h, w, k, s, k // 2)
    ts, lib = TileMask(n, ho, wo, DEV), _lib.lib()
    assert not (lib.mie_upconv_needs_no_workspace(c1, cout, ts.capacity, code) if kind == "up" else
                lib.mie_conv_gates_needs_no_workspace(c1, c2, cout // 4, ts.capacity, code) if kind == "gates" else
                lib.mie_conv_needs_no_workspace(k, s, c1, c2, cout, ts.capacity, code))
    filt = ops.ConvFilter(he_normal_conv_weight(cout, c1 + c2, k, 3).permute(1, 2, 3, 0).contiguous().to(DEV))
    d, m = gaussian_delta(n, c1 + c2, h, w, 0.3, 0.5, seed=8)
    x, x2, dm = _dev(d[:, :c1]).to(dtype), _dev(d[:, c1:]).to(dtype) if c2 else None, m.to(DEV)
    got = []
    for ws in (None, _split_workspace()):
        ops.split_workspace(torch.device(DEV)).fill_(float("nan"))
        out, res = ops.new_nhwc(n, cout, ho, wo, DEV, dtype), ops.new_nhwc(n, cout, ho, wo, DEV)
        if kind == "up":
            up = TileMask(n, ho, wo, DEV)
            ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_UP2X, 0, 0, 0, up)
            ops.build_mask_tiles(up, None, n, ho, wo, _lib.FOOT_CONV, 5, 1, 2, ts)
            ops.upconv_masked(x, dm, None, None, filt, 5, 2, ts, out, res, _lib.ACT_RELU, 0.0, workspace=ws)
            got.append((out, res))
            assert not ops.upconv2x_takes(x, cout, 5, 1, 2, filt)
        elif kind == "gates":
            ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_CONV, k, s, k // 2, ts)
            cells = [ops.new_nhwc(n, cout // 4, h, w, DEV) for _ in range(2)] + [ops.new_nhwc(n, cout // 4, h, w, DEV, dtype) for _ in range(2)]
            ops.conv_gates_incr(x, dm, x2, None if x2 is None else dm, filt, ts, res, None, None, *cells, workspace=ws, one_launch=True)
            got.append((res, *cells))
        else:
            ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_CONV, k, s, k // 2, ts)
            ops.conv_masked(x, dm, x2, None if x2 is None else dm, filt, k, s, k // 2, ts, out, res, _lib.ACT_RELU, 0.0, workspace=ws)
            got.append((out, res))
        assert torch.isfinite(ops.split_workspace(torch.device(DEV))).any() == (ws is None)
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and torch.equal(a, b)
    assert got[0][-1 if kind == "gates" else 0].any()
