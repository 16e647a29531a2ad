"""fp32 deltas in two fp16 terms whose values do not fit a workgroup's scale, in every form that takes them, with its epilogue: gates, ConvGRU, fused
activation with reservoir and addend, up-sampled and transposed convs, refreshes.  Reservoirs and outputs against fp64; where values are not
finite, against the fp32 instruction.  No counterpart in the reference, whose convs have one arithmetic."""
import pytest
import torch
import torch.nn.functional as F

from maskedincrementeval_amd import _lib, ops
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.synthetic import he_normal_conv_weight

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
WHAT = ["pixels", "channels", "filter", "not finite"]


def _dev(t):
    return ops.as_nhwc(t.to(DEV).contiguous(memory_format=torch.channels_last))


@pytest.fixture(autouse=True)
def setting():
    old = ops.f32_matmul
    yield
    ops.f32_matmul = old


def _rnd(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def _unfit(what, x, wt, cin_at):
    """Input and filter (its input channels along `cin_at`) with what does not fit: other rows of the plane 2^-30 of the rest, channels of 2^-8 to 1,
    some filter rows of 1e-12, or infinities and NaN."""
    x, wt, c = x.clone(), wt.clone(), x.shape[1]
    if what == "pixels":
        x[:, :, 1::2] *= 2.0 ** -30
    elif what == "channels":
        x *= (2.0 ** (8.0 * torch.arange(c) / c - 8.0)).view(1, -1, 1, 1)
    elif what == "filter":
        wt.narrow(cin_at, c // 2, 8).mul_(1e-12)
    else:
        x[0, 1, x.shape[2] // 2, 0], x[0, c - 1, 0, -1], x[0, c // 2, -1, x.shape[3] // 2] = float("inf"), float("nan"), -3.4e38
    return x, wt


def _mask(n, h, w, seed):
    m = torch.rand(n, 1, (h + 7) // 8, (w + 7) // 8, generator=torch.Generator().manual_seed(seed)) < 0.6
    return F.interpolate(m.float(), scale_factor=8)[:, :, :h, :w].to(torch.uint8).contiguous()


def _poison(x, m):
    """What an inactive pixel holds is not read."""
    return torch.where(m.bool(), x, torch.full((), float("nan")))


def _same_not_finite(run, outs):
    """The fp32 instruction's not finite values, and only these; what is finite is near to its values: both are within 4e-7 of sum |x||w|, of
    up to 1e3 * 3.4e38 where the huge value comes in, of about 1e3 elsewhere."""
    for a, b in zip(outs, run("native")):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
        fine = torch.isfinite(b)
        assert (((a - b).abs() <= 1e-5 + 1e-5 * b.abs()) | (b.abs() > 1e30) | (a.abs() > 1e30))[fine].all()


def _act(z, kind):
    return torch.relu(z) if kind == _lib.ACT_RELU else z


def _check(run, what, res0, sums, bound, kind=_lib.ACT_RELU, extra=None):
    """run(mode) -> (delta, reservoir).  Sums within 4e-7 of sum |x||w| (fp32 roundings), the reservoir with its own rounding, the increment of
    an activation of slope 1 within both reservoirs' errors."""
    outs = run("f16x2")
    if what == "not finite":
        return _same_not_finite(run, outs)
    z = sums if extra is None else sums + extra.double()
    tol = 4e-7 * bound + 2.0 ** -23 * (res0.abs() + z.abs() + (0 if extra is None else extra.abs()))
    delta, res = outs
    assert ((res - (res0.double() + z)).abs() <= tol).all(), ((res - (res0.double() + z)).abs() / tol).max()
    want = _act(res0.double() + z, kind) - _act(res0.double(), kind)
    assert ((delta - want).abs() <= 2 * tol).all(), ((delta - want).abs() / tol).max()


def _both(f, x, w):
    return f(x.double(), w.double()), f(x.double().abs(), w.double().abs())


# whole (slabs of 32, 64, 128 columns, four and eight waves), split, in one launch
@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("c1,c2,cout,k,stride,h,w", [(64, 0, 64, 3, 1, 70, 75), (128, 128, 256, 3, 1, 33, 44), (64, 64, 128, 3, 1, 66, 88), (64, 0, 128, 5, 2, 80, 100),
                                                     (64, 64, 64, 5, 2, 132, 140), (64, 0, 32, 5, 1, 33, 47), (512, 512, 256, 3, 1, 17, 9), (256, 256, 128, 3, 1, 16, 16)])
def test_conv_with_reservoir_addend_and_masks(c1, c2, cout, k, stride, h, w, what):
    cin = c1 + c2
    x, wt = _unfit(what, _rnd(1, cin, h, w, seed=1), he_normal_conv_weight(cout, cin, k, 7), 1)
    m, ho, wo = _mask(1, h, w, 3), *ops.conv_out_size(h, w, k, stride, k // 2)
    ts = TileMask(1, ho, wo, DEV)
    ops.build_mask_tiles(m.to(DEV), None, 1, h, w, _lib.FOOT_CONV, k, stride, k // 2, ts)
    live = ts.pixmask.cpu().bool()
    res0, extra = _rnd(1, cout, ho, wo, seed=2), _rnd(1, cout, ho, wo, seed=4) * live
    p, filt = _poison(x, m), ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))

    def run(mode):
        ops.f32_matmul = mode
        res, out = _dev(res0).clone(), ops.new_nhwc(1, cout, ho, wo, DEV).zero_()
        ops.conv_masked(_dev(p[:, :c1]), m.to(DEV), _dev(p[:, c1:]) if c2 else None, m.to(DEV) if c2 else None, filt, k, stride, k // 2, ts, out, res,
                        _lib.ACT_RELU, path=_lib.PATH_MFMA, addend=_dev(extra))
        return out.cpu().double(), res.cpu().double()
    sums, bound = _both(lambda a, b: F.conv2d(a, b, stride=stride, padding=k // 2), torch.where(m.bool(), x, torch.zeros(())), wt)
    _check(run, what, res0, sums, bound, extra=extra)


@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("c1,c2,cout,h,w", [(64, 0, 64, 70, 75), (128, 128, 256, 33, 44)])
def test_refresh_conv(c1, c2, cout, h, w, what):
    x, wt = _unfit(what, _rnd(1, c1 + c2, h, w, seed=1), he_normal_conv_weight(cout, c1 + c2, 3, 7), 1)
    bias, filt = _rnd(cout, seed=5), ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    ts = TileMask(1, h, w, DEV)
    ops.build_mask_tiles(None, None, 1, h, w, _lib.FOOT_CONV, 1, 1, 0, ts)

    def run(mode):
        ops.f32_matmul = mode
        res, out = (ops.new_nhwc(1, cout, h, w, DEV) for _ in range(2))
        ops.conv_refresh(_dev(x[:, :c1]), _dev(x[:, c1:]) if c2 else None, filt, bias.to(DEV), 3, 1, 1, ts, out, res, _lib.ACT_RELU)
        return out.cpu().double(), res.cpu().double()
    sums, bound = _both(lambda a, b: F.conv2d(a, b, padding=1), x, wt)
    _check(run, what, torch.zeros(1, cout, h, w), sums, bound, extra=bias.view(1, -1, 1, 1).expand(1, -1, h, w))


# one kernel over the blended tile: whole, and split on planes of few tiles
@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("c,cout,h,w", [(64, 32, 33, 37), (64, 64, 70, 90), (128, 128, 44, 40), (256, 128, 16, 16)])
def test_up_sampled_conv(c, cout, h, w, what):
    a, wt = _unfit(what, _rnd(1, c, h, w, seed=1), he_normal_conv_weight(cout, c, 5, 7), 1)
    b = a.roll(1, 0) if what == "not finite" else _unfit(what, _rnd(1, c, h, w, seed=6), wt, 1)[0]
    m = _mask(1, h, w, 3)
    t0, ts = TileMask(1, 2 * h, 2 * w, DEV), TileMask(1, 2 * h, 2 * w, DEV)
    ops.build_mask_tiles(m.to(DEV), m.to(DEV), 1, h, w, _lib.FOOT_UP2X, 0, 0, 0, t0)
    ops.build_mask_tiles(t0, None, 1, 2 * h, 2 * w, _lib.FOOT_CONV, 5, 1, 2, ts)
    res0, filt = _rnd(1, cout, 2 * h, 2 * w, seed=2), ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))

    def run(mode):
        ops.f32_matmul = mode
        res, out = _dev(res0).clone(), ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV).zero_()
        ops.upconv_masked(_dev(_poison(a, m)), m.to(DEV), _dev(_poison(b, m)), m.to(DEV), filt, 5, 2, ts, out, res, _lib.ACT_RELU)
        return out.cpu().double(), res.cpu().double()
    up = lambda t: F.interpolate(t.double() * m, scale_factor=2, mode="bilinear", align_corners=False)      # noqa: E731
    if what == "not finite":
        return _check(run, what, res0, None, None)
    sums, bound = F.conv2d(up(a + b), wt.double(), padding=2), F.conv2d(up(a.abs() + b.abs()), wt.double().abs(), padding=2)
    _check(run, what, res0, sums, 1.5 * bound)      # (the blend's roundings: 6e-7, as in the decoders of test_gpu_f16x2.py)


@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("c,cout,h,w", [(128, 64, 66, 88), (64, 32, 72, 123), (256, 128, 20, 21)])
def test_decoder_at_input_resolution_and_its_refresh(c, cout, h, w, what):
    a, wt = _unfit(what, _rnd(1, c, h, w, seed=1), he_normal_conv_weight(cout, c, 5, 7), 1)
    t0, ts = TileMask(1, 2 * h, 2 * w, DEV), TileMask(1, 2 * h, 2 * w, DEV)
    ops.build_mask_tiles(None, None, 1, h, w, _lib.FOOT_UP2X, 0, 0, 0, t0)
    ops.build_mask_tiles(t0, None, 1, 2 * h, 2 * w, _lib.FOOT_CONV, 5, 1, 2, ts)
    res0, bias = _rnd(1, cout, 2 * h, 2 * w, seed=2), _rnd(cout, seed=5)
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    assert _lib.lib().mie_f16x2_takes_upconv2x(1, h, w, c, cout)
    ops.f32_matmul = "f16x2"
    res, out = _dev(res0).clone(), ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV)
    fill, dense = ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV), ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV)
    ops.upconv2x_masked(_dev(a), None, None, None, filt, ts, out, res, _lib.ACT_RELU)
    ops.upconv2x_refresh(_dev(a), None, filt, bias.to(DEV), ts, dense, fill, _lib.ACT_RELU)
    outs, filled = (out.cpu().double(), res.cpu().double()), (dense.cpu().double(), fill.cpu().double())
    up = lambda t: F.interpolate(t.double(), scale_factor=2, mode="bilinear", align_corners=False)      # noqa: E731
    if what == "not finite":      # (not finite wherever a value that is not comes in, by a weight that may be zero: around its pixel)
        near = F.conv2d(F.pad((~torch.isfinite(a) | (a.abs() > 1e38)).any(1, keepdim=True).float(), (2, 2, 2, 2)), torch.ones(1, 1, 5, 5))
        far = (F.interpolate(near, scale_factor=2) == 0).expand(1, cout, -1, -1)
        for got in (*outs, *filled):
            assert torch.isfinite(got[far]).all() and (~torch.isfinite(got)).any()
        return
    sums, bound = F.conv2d(up(a), wt.double(), padding=2), F.conv2d(up(a.abs()), wt.double().abs(), padding=2)
    _check(lambda mode: outs, what, res0, sums, 1.5 * bound)
    _check(lambda mode: filled, what, torch.zeros_like(res0), sums, 1.5 * bound, extra=bias.view(1, -1, 1, 1).expand_as(res0))


# with a leading part (two more channels in front), and the refresh
@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("c1,c2,cout,h,w,lead", [(64, 64, 32, 100, 125, True), (64, 64, 64, 150, 170, True), (128, 64, 64, 66, 88, False), (1024, 512, 64, 8, 7, False)])
def test_transposed_conv(c1, c2, cout, h, w, lead, what):
    cin, z = c1 + c2, 2 if lead else 0
    x, wt = _unfit(what, _rnd(1, cin, h, w, seed=1), _rnd(cin, cout, 3, 3, seed=8) * (8.0 / (cin * 9)) ** 0.5, 0)
    x = torch.cat([_rnd(1, z, h, w, seed=9), x], 1)
    wt = torch.cat([_rnd(z, cout, 3, 3, seed=10) * 0.1, wt])
    ho, wo, m = 2 * h, 2 * w, _mask(1, h, w, 3)
    filt = ops.ConvFilter(wt.permute(0, 2, 3, 1).contiguous().to(DEV))
    wide = filt.rows(z, z + cin)
    ts, blocks, all_ts, all_blocks = TileMask(1, ho, wo, DEV), TileMask(1, h, w, DEV), TileMask(1, ho, wo, DEV), TileMask(1, h, w, DEV)
    for mask, t, b in ((m.to(DEV), ts, blocks), (None, all_ts, all_blocks)):
        ops.build_mask_tiles(mask, None, 1, h, w, _lib.FOOT_TCONV, 3, 2, 1, t)
        ops.build_mask_tiles(t, None, 1, ho, wo, _lib.FOOT_CONV, 2, 2, 0, b)
    res0, bias, p = _rnd(1, cout, ho, wo, seed=2), _rnd(cout, seed=5), _poison(x, m)

    def run(mode):
        ops.f32_matmul = mode
        res, out = _dev(res0).clone(), ops.new_nhwc(1, cout, ho, wo, DEV).zero_()
        part = mode != "native" and lead
        add = None
        if lead and not part:      # (its increments from a call of their own)
            add = ops.new_nhwc(1, cout, ho, wo, DEV).zero_()
            ops.tconv_masked(_dev(p[:, :z]), m.to(DEV), filt.rows(0, z), 3, 2, 1, ts, add)
        ops.tconv2x_masked(_dev(p[:, z:z + c1]), m.to(DEV), _dev(p[:, z + c1:]), m.to(DEV), wide, 3, ts, blocks, out, res, _lib.ACT_RELU, addend=add,
                           lead=(_dev(p[:, :z]), m.to(DEV), filt.rows(0, z)) if part else None)
        return out.cpu().double(), res.cpu().double()

    def refresh(mode):
        ops.f32_matmul = mode
        res, out = (ops.new_nhwc(1, cout, ho, wo, DEV) for _ in range(2))
        ops.tconv2x_refresh(_dev(x[:, z:z + c1]), _dev(x[:, z + c1:]), wide, bias.to(DEV), 3, all_ts, all_blocks, out, res, _lib.ACT_RELU)
        return out.cpu().double(), res.cpu().double()
    up = lambda a, b: F.conv_transpose2d(a, b, stride=2, padding=1, output_padding=1)      # noqa: E731
    _check(run, what, res0, *_both(up, torch.where(m.bool(), x, torch.zeros(())), wt))
    if what != "not finite" or cin < 1024:      # (that one's refresh has no workspace to split over: three terms, which make NaN of infinities)
        _check(refresh, what, torch.zeros_like(res0), *_both(up, x[:, z:], wt[z:]), extra=bias.view(1, -1, 1, 1).expand_as(res0))


# whole (slabs of 32 to 128, eight waves at 128 + 128 -> 256 columns), split, in one launch in two terms
@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("c1,c2,hid,h,w,one", [(64, 64, 64, 66, 70, False), (128, 128, 64, 33, 44, False), (64, 0, 16, 64, 96, False), (256, 256, 128, 33, 44, False),
                                               (128, 128, 64, 12, 20, False), (256, 256, 64, 16, 16, True)])
def test_convlstm_gates(c1, c2, hid, h, w, one, what):
    cin, cols = c1 + c2, 4 * hid
    x, wt = _unfit(what, _rnd(1, cin, h, w, seed=1), he_normal_conv_weight(cols, cin, 3, 7), 1)
    m = _mask(1, h, w, 3)
    ts = TileMask(1, h, w, DEV)
    ops.build_mask_tiles(m.to(DEV), m.to(DEV) if c2 else None, 1, h, w, _lib.FOOT_CONV, 3, 1, 1, ts)
    res0, cp, cell = _rnd(1, cols, h, w, seed=2), _rnd(1, hid, h, w, seed=4), _rnd(1, hid, h, w, seed=5)
    p, filt = _poison(x, m), ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))

    def run(mode):
        ops.f32_matmul = mode
        g, r1, r2 = _dev(res0).clone(), _dev(cp).clone(), _dev(cell).clone()
        dh, dc = (ops.new_nhwc(1, hid, h, w, DEV).zero_() for _ in range(2))
        ops.conv_gates_incr(_dev(p[:, :c1]), m.to(DEV), _dev(p[:, c1:]) if c2 else None, m.to(DEV) if c2 else None, filt, ts, g, None, None, r1, r2, dh, dc,
                            one_launch=one)
        return tuple(t.cpu().double() for t in (g, dh, dc, r2))
    outs = run("f16x2")
    if what == "not finite":
        return _same_not_finite(run, outs)
    sums, bound = _both(lambda a, b: F.conv2d(a, b, padding=1), torch.where(m.bool(), x, torch.zeros(())), wt)
    tol = 4e-7 * bound + 2.0 ** -23 * (res0.abs() + sums.abs())
    assert ((outs[0] - res0.double() - sums).abs() <= tol).all(), ((outs[0] - res0.double() - sums).abs() / tol).max()
    # the states against the fp32 instruction's, whose gates lie within 1e-6 of sum |x||w| and these: sigmoid and tanh of slopes 1/4 and 1, cells of
    # up to 6, four gates a channel
    near = 8.0 * 2 * (1e-6 * bound + 2.0 ** -23 * (res0.abs() + sums.abs())).view(1, hid, 4, h, w).sum(2) + 1e-6
    for a, b in zip(outs[1:], run("native")[1:]):
        assert ((a - b).abs() <= near).all(), ((a - b).abs() / near).max()


@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("cin,hid,h,w", [(64, 32, 90, 93), (64, 64, 90, 93), (512, 64, 16, 16)])
def test_convgru(cin, hid, h, w, what):
    x, wt = _unfit(what, _rnd(1, cin, h, w, seed=1), he_normal_conv_weight(2 * hid, cin, 3, 7), 1)
    m, order = _mask(1, h, w, 3), ops.gru_interleave_index(hid)
    filt = ops.ConvFilter(wt[order].permute(1, 2, 3, 0).contiguous().to(DEV))
    stacked = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    ts = TileMask(1, h, w, DEV)
    ops.build_mask_tiles(m.to(DEV), None, 1, h, w, _lib.FOOT_CONV, 3, 1, 1, ts)
    res0, p = _rnd(1, 2 * hid, h, w, seed=2), _poison(x, m)

    def run(mode):
        ops.f32_matmul = mode
        u, c = (_dev(r).clone() for r in res0.split(hid, 1))
        dh = ops.new_nhwc(1, hid, h, w, DEV).zero_()
        if mode != "native":
            assert ops.conv_gru_takes(cin, cin, hid, torch.float32)
            ops.conv_gru_incr(_dev(p), m.to(DEV), filt, ts, u, c, dh)
        else:
            both = ops.new_nhwc(1, 2 * hid, h, w, DEV)
            ops.conv_masked(_dev(p), m.to(DEV), None, None, stacked, 3, 1, 1, ts, both)
            ops.convgru_gates_incr(both, u, c, dh, ts)
        return torch.cat([u, c], 1).cpu().double(), dh.cpu().double()
    outs = run("f16x2")
    if what == "not finite":
        return _same_not_finite(run, outs)
    sums, bound = _both(lambda a, b: F.conv2d(a, b, padding=1), torch.where(m.bool(), x, torch.zeros(())), wt)
    tol = 4e-7 * bound + 2.0 ** -23 * (res0.abs() + sums.abs())
    assert ((outs[0] - res0.double() - sums).abs() <= tol).all()
    state = lambda r: r[:, :hid].sigmoid() * r[:, hid:].tanh()      # noqa: E731
    want = state(res0.double() + sums) - state(res0.double())
    # sigmoid and tanh carry the errors of their arguments with slopes of 1/4 and 1; their own errors are some 2^-24 (16 of them) of values below 2
    assert ((outs[1] - want).abs() <= 0.25 * tol[:, :hid] + tol[:, hid:] + 16 * 2.0 ** -24 * 2).all()
