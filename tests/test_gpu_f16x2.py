"""The two-term fp16 form of the fp32 matrix-core convs (MIE_DTYPE_F32_F16X2): filter copy, error against fp64 beside three bf16
terms, and the inputs that do not fit the scale of a workgroup.  No counterpart in the reference, whose convs have one arithmetic."""
import pytest
import torch
import torch.nn.functional as F

from maskedincrementeval_amd import _lib, ops
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.synthetic import he_normal_conv_weight

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(t):
    return ops.as_nhwc(t.to(DEV).contiguous(memory_format=torch.channels_last))


def _filt(w_oihw):
    return ops.ConvFilter(w_oihw.permute(1, 2, 3, 0).contiguous().to(DEV))


@pytest.fixture
def setting():
    old = ops.f32_matmul
    yield
    ops.f32_matmul = old


@pytest.mark.parametrize("top,bottom,fits", [(1.0, 1e-8, 1.0), (1e-12, 1e-20, 1.0), (3e10, 100.0, 1.0), (1.0, 1e-9, 0.0), (1e-20, 1e-32, 0.0),
                                             (float("inf"), 1.0, 0.0), (float("nan"), 1.0, 0.0), (0.0, 0.0, 1.0)])
def test_filter_copy(top, bottom, fits):
    cin, k, cout = 32, 3, 40
    g = torch.Generator().manual_seed(1)
    w = (torch.rand(cin, k, k, cout, generator=g) + 0.5) * (1.0 if top != 0.0 else 0.0)
    w = w * (min(top, 3e38) if top == top and top != 0.0 else 1.0) * 0.6
    w[8:16, 1, 1, 5] = bottom * torch.rand(8, generator=g).clamp_min(0.5)          # a small group
    w[3, 0, 0, 0], w[16:24, 2, 2, 7] = top, 0.0
    raw = ops.pack_filter(w.contiguous().to(DEV), f16x2=True).cpu()
    m = w.numel()
    assert raw.numel() == 14 * m + _lib.F16X2_END_BYTES
    three = raw[:6 * m].view(torch.bfloat16).view(cin // 16, k * k, 3, 2, cout, 8).permute(2, 0, 3, 5, 1, 4).reshape(3, cin, k, k, cout)
    terms = raw[6 * m:10 * m].view(torch.float16).view(cin // 16, k * k, 2, 2, cout, 8).permute(2, 0, 3, 5, 1, 4).reshape(2, cin, k, k, cout).double()
    values = raw[10 * m:14 * m].view(torch.float32).view(cin // 16, k * k, 2, 2, cout, 4).permute(0, 3, 2, 5, 1, 4).reshape(cin, k, k, cout)
    end = raw[14 * m:14 * m + 16].view(torch.float32)
    assert torch.equal(values.nan_to_num(nan=7.0), w.nan_to_num(nan=7.0))
    assert end[1].item() == fits
    if fits:
        assert torch.equal(three.double().sum(0), w.double()) or top < 1e-30
        back = (terms[0] + terms[1] / 2048) * end[0].double()
        # 23 bits, and where a value lies far below the largest of its filter what the fp16 subnormals leave
        assert ((back - w.double()).abs() <= w.double().abs() * 2.0 ** -23 + 2.0 ** -36 * end[0].double()).all()
        mant = torch.frexp(end[0])[0].item()
        assert mant == 0.5 and (top == 0.0 or 2.0 ** 14 <= (w.abs().max() / end[0]).item() < 2.0 ** 15)


def _conv(x, wt, k, stride, mode, c1=None, xm=None, path=_lib.PATH_MFMA, workspace=None):
    n, cin, h, w = x.shape
    c1 = cin if c1 is None else c1
    ho, wo = ops.conv_out_size(h, w, k, stride, k // 2)
    ts = TileMask(n, ho, wo, DEV)
    ops.build_mask_tiles(xm, None, n, h, w, _lib.FOOT_CONV, k, stride, k // 2, ts)
    out = ops.new_nhwc(n, wt.shape[0], ho, wo, DEV)
    ops.f32_matmul = mode
    ops.conv_masked(_dev(x[:, :c1]), xm, None if c1 == cin else _dev(x[:, c1:]), None if c1 == cin else xm, _filt(wt), k, stride, k // 2, ts, out,
                    path=path, workspace=workspace)
    torch.cuda.synchronize()
    return out.cpu().double()


# planes of more than 256 slabs of 16 columns, or more channels than the one-launch form: k_conv_mfma, whole and (the three with a workspace) split
SHAPES = [(32, 32, 3, 1, 136, 130, None), (64, 64, 3, 1, 70, 75, None), (128, 128, 3, 1, 41, 47, 64), (256, 256, 3, 1, 33, 44, None),
          (256, 512, 3, 1, 34, 39, 128), (64, 32, 5, 1, 33, 47, None), (128, 128, 5, 1, 34, 42, None), (32, 64, 5, 2, 131, 133, None),
          (128, 256, 5, 2, 66, 88, None), (1024, 256, 3, 1, 17, 9, None), (256, 32, 5, 1, 16, 16, None), (512, 64, 5, 2, 17, 16, 256),
          # eight waves a workgroup (up to 256 of them): slabs of 32, 64 and 128, two and many chunks; inputs that are no whole chunks of it
          (64, 128, 5, 2, 80, 100, None), (96, 128, 5, 2, 79, 101, 32), (512, 1024, 3, 1, 30, 44, 256), (320, 256, 3, 1, 33, 47, 64), (256, 256, 3, 1, 33, 44, 96),
          # the one-launch form from 512 channels on: two, four and eight rows a workgroup, waves of two and three chunks
          (512, 64, 3, 1, 7, 9, None), (512, 64, 3, 1, 16, 24, 192), (576, 128, 3, 1, 24, 20, None), (512, 128, 3, 1, 31, 33, 256)]


@pytest.mark.parametrize("cin,cout,k,stride,h,w,c1", SHAPES)
def test_error_against_fp64_beside_three_terms(cin, cout, k, stride, h, w, c1, setting):
    g = torch.Generator().manual_seed(cin + h)
    x = torch.randn(1, cin, h, w, generator=g) * torch.rand(1, 1, h, w, generator=g)
    wt = he_normal_conv_weight(cout, cin, k, 7)
    ref = F.conv2d(x.double(), wt.double(), stride=stride, padding=k // 2)
    bound = F.conv2d(x.double().abs(), wt.double().abs(), stride=stride, padding=k // 2)
    err = {}
    for mode in ("bf16x3", "f16x2"):
        e = (_conv(x, wt, k, stride, mode, c1) - ref).abs()
        err[mode] = (e.norm() / ref.norm()).item(), (e / bound).max().item()
    # the norm of the error is that of some thousand outputs at least; a single output's may be either way
    assert err["f16x2"][0] <= err["bf16x3"][0] and err["f16x2"][1] < 4e-7, err


@pytest.mark.parametrize("cin,cout,k,stride,h,w,c1", SHAPES)
def test_scaled_inputs_give_scaled_outputs(cin, cout, k, stride, h, w, c1, setting):
    """The scale follows the data: inputs times a power of two, the same bits."""
    g = torch.Generator().manual_seed(cin)
    x = torch.randn(1, cin, h, w, generator=g)
    wt = he_normal_conv_weight(cout, cin, k, 7)
    one = _conv(x, wt, k, stride, "f16x2", c1)
    for e in (-27, 30):
        assert torch.equal(_conv(x * 2.0 ** e, wt * 2.0 ** -e, k, stride, "f16x2", c1), one)
        assert torch.equal(_conv(x * 2.0 ** e, wt, k, stride, "f16x2", c1), one * 2.0 ** e)


@pytest.mark.parametrize("cin,cout,k,stride,h,w,c1", SHAPES)
@pytest.mark.parametrize("what", ["below", "above", "not finite", "filter", "first chunk zero", "second input only"])
def test_values_that_do_not_fit_the_scale(cin, cout, k, stride, h, w, c1, what, setting):
    """Every value of the result within 4e-7 of sum |x||w|, three fp32 roundings, as the fp32 instruction has it; non-finite ones
    where an fp32 conv has them, and only there."""
    g = torch.Generator().manual_seed(cin + k)
    x, wt = torch.randn(1, cin, h, w, generator=g), he_normal_conv_weight(cout, cin, k, 7)
    if what == "below":
        x[:, :, h // 2:] *= 1e-13
    elif what == "above":
        x[:, cin // 2:] *= 1e6
    elif what == "filter":
        wt[:, : cin // 2] *= 1e-10
    elif what == "first chunk zero":
        x[:, :32] = 0.0
        x *= 1e-3
    elif what == "second input only":
        x[:, : cin // 2] *= 1e-12
    else:
        x[0, 1, 2, 3], x[0, cin - 1, h - 1, w - 1], x[0, 0, h // 2, 0], x[0, cin // 2, h // 2, w - 2] = float("inf"), float("-inf"), float("nan"), 3.4e38
    got = _conv(x, wt, k, stride, "f16x2", c1)
    ref = F.conv2d(x.double(), wt.double(), stride=stride, padding=k // 2)
    bound = F.conv2d(x.double().abs(), wt.double().abs(), stride=stride, padding=k // 2)
    if what == "not finite":
        want = F.conv2d(x, wt, stride=stride, padding=k // 2)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        assert torch.equal(got[torch.isinf(want)].float(), want[torch.isinf(want)])
        fine = torch.isfinite(want) & torch.isfinite(ref)
    else:
        fine = torch.isfinite(ref)
        assert torch.isfinite(got).all()
    assert ((got - ref).abs() <= 4e-7 * bound)[fine].all(), ((got - ref).abs() / bound)[fine].max()


def test_masked_pixels_do_not_count(setting):
    """What lies under a cleared mask byte is neither multiplied nor looked at for the scale."""
    g = torch.Generator().manual_seed(3)
    x, wt = torch.randn(1, 64, 70, 75, generator=g), he_normal_conv_weight(64, 64, 3, 7)
    m = (torch.rand(1, 1, 70, 75, generator=g) < 0.5).to(torch.uint8)
    clean = _conv(x * m, wt, 3, 1, "f16x2", xm=m.to(DEV))
    junk = torch.where(m.bool().expand_as(x), x, torch.full((), float("inf")))
    assert torch.equal(_conv(junk, wt, 3, 1, "f16x2", xm=m.to(DEV)), clean)


def _up2x(a, b, wt, mode, out=None):
    n, c, h, w = a.shape
    ts = TileMask(n, 2 * h, 2 * w, DEV)
    ops.build_mask_tiles(None, None, n, 2 * h, 2 * w, _lib.FOOT_CONV, 5, 1, 2, ts)
    out = ops.new_nhwc(n, wt.shape[0], 2 * h, 2 * w, DEV)
    ops.f32_matmul = mode
    ops.upconv2x_masked(_dev(a), None, None if b is None else _dev(b), None, _filt(wt), ts, out)
    torch.cuda.synchronize()
    return out.cpu().double()


# decoders at the resolution of their inputs: 32 columns a workgroup (up to 256 of them) and 64; blocks in part, strips and corners; 64 and 96
# channels on many blocks: all phases in a workgroup
@pytest.mark.parametrize("c,cout,h,w,two", [(128, 64, 32, 32, True), (128, 64, 66, 88, True), (256, 128, 33, 44, True), (256, 64, 9, 11, False),
                                            (160, 32, 21, 37, True), (128, 96, 2, 40, True), (128, 32, 10, 3, False),
                                            (64, 32, 72, 123, True), (96, 64, 63, 66, False)])
@pytest.mark.parametrize("what", ["fits", "below", "above", "not finite", "filter"])
def test_decoders_at_the_resolution_of_their_inputs(c, cout, h, w, two, what, setting):
    g = torch.Generator().manual_seed(c + h)
    a = torch.randn(1, c, h, w, generator=g) * torch.rand(1, 1, h, w, generator=g)
    b = torch.randn(1, c, h, w, generator=g) if two else None
    wt = he_normal_conv_weight(cout, c, 5, 7)
    if what == "below":
        a[:, :, h // 2:] *= 1e-13
        b = None if b is None else b * (torch.arange(h).view(1, 1, h, 1) < h // 2)
    elif what == "above":
        a[:, c // 2:] *= 1e6
    elif what == "filter":
        wt[:, : c // 2] *= 1e-10
    elif what == "not finite":
        a[0, 1, h // 2, w // 2], a[0, c - 1, 0, 0] = float("inf"), float("nan")
    up = lambda t: F.interpolate(t.double(), scale_factor=2, mode="bilinear", align_corners=False)      # noqa: E731
    s = a if b is None else a + b
    size = a.abs() if b is None else a.abs() + b.abs()
    ref, bound = F.conv2d(up(s), wt.double(), padding=2), F.conv2d(up(size), wt.double().abs(), padding=2)
    got = _up2x(a, b, wt, "f16x2")
    if what == "not finite":
        # (the phases' windows are the clamped taps': zero coefficients times an infinity make NaN of some outputs beside an fp32 conv's)
        bad = torch.zeros(1, 1, h, w)
        bad[0, 0, h // 2, w // 2] = bad[0, 0, 0, 0] = 1.0
        near = F.max_pool2d(F.interpolate(F.max_pool2d(bad, 5, 1, 2), scale_factor=2), 3, 1, 1).bool().expand_as(got)
        assert torch.isfinite(got[~near]).all() and not torch.isfinite(got[~torch.isfinite(ref)]).any()
        fine = ~near
    else:
        fine = torch.ones_like(got, dtype=torch.bool)
    # the combined weights are rounded sums of up to 25, the sum of the inputs is rounded: five fp32 roundings
    assert ((got - ref).abs() <= 6e-7 * bound + 1e-30)[fine].all(), ((got - ref).abs() / bound)[fine].max()
    if what == "fits":
        three = _up2x(a, b, wt, "bf16x3")
        assert (got - ref).norm() <= (three - ref).norm()


# transposed convs: 32 and 64 columns a workgroup, planes cut off at both edges, split (more than 1408 channels on few blocks, 5x5)
@pytest.mark.parametrize("c1,c2,cout,h,w,k", [(64, 64, 32, 127, 131, 3), (128, 0, 64, 132, 176, 3), (64, 64, 64, 160, 159, 3), (1024, 512, 64, 8, 7, 3),
                                              (64, 64, 32, 90, 93, 5), (256, 64, 32, 9, 8, 5)])
@pytest.mark.parametrize("what", ["fits", "below", "above", "not finite", "second input only"])
def test_transposed_convs(c1, c2, cout, h, w, k, what, setting):
    g = torch.Generator().manual_seed(c1 + h)
    cin = c1 + c2
    x = torch.randn(1, cin, h, w, generator=g)
    wt = torch.randn(cin, cout, k, k, generator=g) * (8.0 / (cin * k * k)) ** 0.5
    if what == "below":
        x[:, :, h // 2:] *= 1e-13
    elif what == "above":
        x[:, cin // 2:] *= 1e6
    elif what == "second input only":
        x[:, :c1] = 0.0
        x *= 1e-6
    elif what == "not finite":
        x[0, 1, h // 2, w // 2], x[0, cin - 1, 0, 0], x[0, 5, h - 1, w - 1] = float("inf"), float("nan"), float("-inf")
    up = lambda x_, w_: F.conv_transpose2d(x_, w_, stride=2, padding=k // 2, output_padding=1)      # noqa: E731
    ref, bound = up(x.double(), wt.double()), up(x.double().abs(), wt.double().abs())
    filt = ops.ConvFilter(wt.permute(0, 2, 3, 1).contiguous().to(DEV))
    ts, blocks = TileMask(1, 2 * h, 2 * w, DEV), TileMask(1, h, w, DEV)
    ops.build_mask_tiles(None, None, 1, h, w, _lib.FOOT_TCONV, k, 2, k // 2, ts)
    ops.build_mask_tiles(ts, None, 1, 2 * h, 2 * w, _lib.FOOT_CONV, 2, 2, 0, blocks)
    got = {}
    for mode in ("bf16x3", "f16x2"):
        ops.f32_matmul = mode
        out = ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV)
        ops.tconv2x_masked(_dev(x[:, :c1]), None, _dev(x[:, c1:]) if c2 else None, None, filt, k, ts, blocks, out)
        torch.cuda.synchronize()
        got[mode] = out.cpu().double()
    fine = torch.isfinite(ref)
    if what == "not finite":
        want = up(x, wt)
        assert torch.equal(torch.isnan(got["f16x2"]), torch.isnan(want)) and torch.equal(torch.isinf(got["f16x2"]), torch.isinf(want))
    assert ((got["f16x2"] - ref).abs() <= 4e-7 * bound)[fine].all(), ((got["f16x2"] - ref).abs() / bound)[fine].max()
    if what == "fits":
        assert (got["f16x2"] - ref).norm() <= (got["bf16x3"] - ref).norm()


def _halves(x, factor):
    """The lower half of the plane `factor` times the upper one: outputs far enough down see small values only, in workgroups that
    see the large ones too."""
    return x * torch.where(torch.arange(x.shape[2]) < x.shape[2] // 2, 1.0, factor).view(1, 1, -1, 1)


# (from where the two terms hold all of a value to far behind where they hold nothing; 4e-7, 6e-7 as in the tests above)
FACTORS = [2.0 ** -22, 2.0 ** -24, 1e-8, 1e-9, 1e-10, 1e-11, 2.0 ** -40]


@pytest.mark.parametrize("cin,cout,k,stride,h,w,c1", SHAPES)
def test_no_digits_lost_below_the_largest_value(cin, cout, k, stride, h, w, c1, setting):
    g = torch.Generator().manual_seed(cin + w)
    x0, wt = torch.randn(1, cin, h, w, generator=g), he_normal_conv_weight(cout, cin, k, 7)
    for factor in FACTORS:
        x = _halves(x0, factor)
        ref = F.conv2d(x.double(), wt.double(), stride=stride, padding=k // 2)
        bound = F.conv2d(x.double().abs(), wt.double().abs(), stride=stride, padding=k // 2)
        e = (_conv(x, wt, k, stride, "f16x2", c1) - ref).abs()
        assert (e <= 4e-7 * bound).all(), (factor, (e / bound).max())


@pytest.mark.parametrize("c,cout,h,w,two", [(128, 64, 66, 88, True), (256, 128, 33, 44, True), (256, 64, 9, 11, False), (64, 32, 72, 123, True), (96, 64, 63, 66, False)])
def test_no_digits_lost_below_the_largest_value_decoders(c, cout, h, w, two, setting):
    g = torch.Generator().manual_seed(c + w)
    a0, b0, wt = torch.randn(1, c, h, w, generator=g), torch.randn(1, c, h, w, generator=g), he_normal_conv_weight(cout, c, 5, 7)
    up = lambda t: F.interpolate(t.double(), scale_factor=2, mode="bilinear", align_corners=False)      # noqa: E731
    for factor in FACTORS:
        a, b = _halves(a0, factor), _halves(b0, factor)
        s, size = (a + b, a.abs() + b.abs()) if two else (a, a.abs())
        ref, bound = F.conv2d(up(s), wt.double(), padding=2), F.conv2d(up(size), wt.double().abs(), padding=2)
        e = (_up2x(a, b if two else None, wt, "f16x2") - ref).abs()
        assert (e <= 6e-7 * bound).all(), (factor, (e / bound).max())


def _tconv(x, c1, wt, k, mode):
    (_, cin, h, w), cout = x.shape, wt.shape[1]
    filt = ops.ConvFilter(wt.permute(0, 2, 3, 1).contiguous().to(DEV))
    ts, blocks = TileMask(1, 2 * h, 2 * w, DEV), TileMask(1, h, w, DEV)
    ops.build_mask_tiles(None, None, 1, h, w, _lib.FOOT_TCONV, k, 2, k // 2, ts)
    ops.build_mask_tiles(ts, None, 1, 2 * h, 2 * w, _lib.FOOT_CONV, 2, 2, 0, blocks)
    ops.f32_matmul = mode
    out = ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV)
    ops.tconv2x_masked(_dev(x[:, :c1]), None, _dev(x[:, c1:]) if c1 < cin else None, None, filt, k, ts, blocks, out)
    torch.cuda.synchronize()
    return out.cpu().double()


def _tconv_ref(x, wt, k):
    up = lambda x_, w_: F.conv_transpose2d(x_, w_, stride=2, padding=k // 2, output_padding=1)      # noqa: E731
    return up(x.double(), wt.double()), up(x.double().abs(), wt.double().abs())


TCONVS = [(64, 64, 32, 127, 131, 3), (128, 0, 64, 132, 176, 3), (1024, 512, 64, 8, 7, 3), (64, 64, 32, 90, 93, 5)]


@pytest.mark.parametrize("c1,c2,cout,h,w,k", TCONVS)
def test_no_digits_lost_below_the_largest_value_transposed(c1, c2, cout, h, w, k, setting):
    g = torch.Generator().manual_seed(c1 + w)
    x0, wt = torch.randn(1, c1 + c2, h, w, generator=g), torch.randn(c1 + c2, cout, k, k, generator=g) * (8.0 / ((c1 + c2) * k * k)) ** 0.5
    for factor in FACTORS:
        x = _halves(x0, factor)
        ref, bound = _tconv_ref(x, wt, k)
        e = (_tconv(x, c1, wt, k, "f16x2") - ref).abs()
        assert (e <= 4e-7 * bound).all(), (factor, (e / bound).max())


def _leading_zero(x, c1, scale):
    """`scale` times x with the leading channels of each input zero, up to half of them: the chunks that a scale is first taken from."""
    x = x * scale
    for lo, hi in ((0, c1), (c1, x.shape[1])):
        x[:, lo:lo + min(64, (hi - lo) // 2)] = 0.0
    return x


@pytest.mark.parametrize("cin,cout,k,stride,h,w,c1", SHAPES)
def test_leading_channels_zero(cin, cout, k, stride, h, w, c1, setting):
    g = torch.Generator().manual_seed(cin + 5)
    x0, wt = torch.randn(1, cin, h, w, generator=g), he_normal_conv_weight(cout, cin, k, 7)
    for scale in (1e-4, 1e-5, 1e-6, 1e-7):
        x = _leading_zero(x0, cin if c1 is None else c1, scale)
        ref = F.conv2d(x.double(), wt.double(), stride=stride, padding=k // 2)
        bound = F.conv2d(x.double().abs(), wt.double().abs(), stride=stride, padding=k // 2)
        e = (_conv(x, wt, k, stride, "f16x2", c1) - ref).abs()
        assert (e <= 4e-7 * bound).all(), (scale, (e / bound).max())


@pytest.mark.parametrize("c,cout,h,w", [(128, 64, 66, 88), (256, 128, 33, 44), (64, 32, 72, 123), (96, 64, 63, 66)])
def test_leading_channels_zero_decoders(c, cout, h, w, setting):
    g = torch.Generator().manual_seed(c + 5)
    a0, wt = torch.randn(1, c, h, w, generator=g), he_normal_conv_weight(cout, c, 5, 7)
    up = lambda t: F.interpolate(t.double(), scale_factor=2, mode="bilinear", align_corners=False)      # noqa: E731
    for scale in (1e-4, 1e-5, 1e-6, 1e-7):
        a = _leading_zero(a0, c, scale)
        ref, bound = F.conv2d(up(a), wt.double(), padding=2), F.conv2d(up(a.abs()), wt.double().abs(), padding=2)
        e = (_up2x(a, None, wt, "f16x2") - ref).abs()
        assert (e <= 6e-7 * bound).all(), (scale, (e / bound).max())


@pytest.mark.parametrize("c1,c2,cout,h,w,k", TCONVS)
def test_leading_channels_zero_transposed(c1, c2, cout, h, w, k, setting):
    g = torch.Generator().manual_seed(c1 + 5)
    x0, wt = torch.randn(1, c1 + c2, h, w, generator=g), torch.randn(c1 + c2, cout, k, k, generator=g) * (8.0 / ((c1 + c2) * k * k)) ** 0.5
    for scale in (1e-4, 1e-5, 1e-6, 1e-7):
        x = _leading_zero(x0, c1, scale)
        ref, bound = _tconv_ref(x, wt, k)
        e = (_tconv(x, c1, wt, k, "f16x2") - ref).abs()
        assert (e <= 4e-7 * bound).all(), (scale, (e / bound).max())


@pytest.mark.parametrize("cin,cout,k,stride,h,w,c1", SHAPES)
def test_channels_of_many_sizes(cin, cout, k, stride, h, w, c1, setting):
    """Channels of 1 ... 2^8 and of 1 ... 2^30, growing and falling, which end the contraction in two terms at a chunk in the middle.  Where a few
    channels make up the sums, all roundings of a chain are at their size: three terms are up to 7.4e-7 of sum |x||w| from fp64, 1.1e-6 of the
    norm.  So: no further than these, or 4e-7 as above; of the norm, with one rounding more at the size of the sum, where the two sets of
    sums meet, and the chains of the one-launch form, which three terms of growing channels keep to 0.9e-7: 1.4 times."""
    g = torch.Generator().manual_seed(cin + 11)
    x0, wt = torch.randn(1, cin, h, w, generator=g), he_normal_conv_weight(cout, cin, k, 7)
    for top in (8.0, 30.0):
        for order in (torch.arange(cin), torch.arange(cin).flip(0), torch.randperm(cin, generator=g)):
            x = x0 * (2.0 ** (top * order / cin)).view(1, -1, 1, 1)
            ref = F.conv2d(x.double(), wt.double(), stride=stride, padding=k // 2)
            bound = F.conv2d(x.double().abs(), wt.double().abs(), stride=stride, padding=k // 2)
            e, e3 = ((_conv(x, wt, k, stride, mode, c1) - ref).abs() for mode in ("f16x2", "bf16x3"))
            assert (e / bound).max() <= max(4e-7, (e3 / bound).max()) and e.norm() <= 1.4 * e3.norm(), (top, (e / bound).max(), e.norm() / e3.norm())


def _graph_us(f):
    """us of a call, the least of eight replays of twenty."""
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        f()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            for _ in range(20):
                f()
    graph.replay()
    best = float("inf")
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 50.0)
    return best


@pytest.mark.parametrize("what", ["channels", "pixels", "filter"])
def test_decoders_that_do_not_fit_take_about_as_long_as_in_three_terms(what, setting):
    """256->128 at 33x44: 47, 65 and 65 us against 42; as two contractions, the second on the fp32 instruction, 120."""
    c, cout, h, w = 256, 128, 33, 44
    g = torch.Generator().manual_seed(3)
    a, wt = torch.randn(1, c, h, w, generator=g), he_normal_conv_weight(cout, c, 5, 7)
    if what == "channels":
        a = a * (2.0 ** (8.0 * torch.arange(c) / c)).view(1, -1, 1, 1)
    elif what == "pixels":
        a[:, :, 1::2] *= 2.0 ** -28
    else:
        wt[3] *= 1e-12
    ts_up, ts = TileMask(1, 2 * h, 2 * w, DEV), TileMask(1, 2 * h, 2 * w, DEV)
    ops.build_mask_tiles(None, None, 1, h, w, _lib.FOOT_UP2X, 0, 0, 0, ts_up)
    ops.build_mask_tiles(ts_up, None, 1, 2 * h, 2 * w, _lib.FOOT_CONV, 5, 1, 2, ts)
    out, filt, x = ops.new_nhwc(1, cout, 2 * h, 2 * w, DEV), _filt(wt), _dev(a)
    us = {}
    for mode in ("bf16x3", "f16x2"):
        ops.f32_matmul = mode
        us[mode] = _graph_us(lambda: ops.upconv2x_masked(x, None, x, None, filt, ts, out))
    assert us["f16x2"] < 2.0 * us["bf16x3"], us
