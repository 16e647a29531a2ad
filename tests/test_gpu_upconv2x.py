"""The decoder conv at the resolution of its inputs (mie_upconv2x_masked / _refresh) against the oracle: 5x5 conv over the
up-sampled sum.  Sizes: planes of border only, below / at / just above a block of 8 and a border strip of 32, several samples;
borders are what the combined filters can get wrong, so every pixel is compared."""
import pytest
import torch

from maskedincrementeval_amd import _lib, ops
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.synthetic import gaussian_delta, he_normal_conv_weight
from oracle import incr_oracle as io
from tolerances import BF16_RTOL, FP32_ATOL, FP32_RTOL, bf16_atol

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(t, dtype=torch.float32):
    return ops.as_nhwc(t.to(DEV).to(dtype).contiguous(memory_format=torch.channels_last))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,cout,h,w", [(1, 64, 32, 2, 2), (1, 64, 32, 2, 5), (2, 64, 64, 7, 2), (1, 64, 32, 3, 34), (1, 64, 64, 35, 3), (1, 64, 96, 8, 8), (1, 128, 64, 9, 16),
                                          (1, 256, 128, 12, 20), (2, 64, 32, 33, 44), (1, 256, 128, 33, 44), (1, 128, 64, 66, 88),
                                          (3, 64, 32, 80, 120), (1, 512, 32, 5, 3), (4, 256, 128, 60, 80)])
def test_decoder_conv_at_input_resolution(n, c, cout, h, w, dtype):
    bf = dtype == torch.bfloat16
    q = (lambda t: t.to(torch.bfloat16).float()) if bf else (lambda t: t)
    tol = (lambda ref: dict(rtol=BF16_RTOL, atol=bf16_atol(ref, 2.0))) if bf else (lambda ref: dict(rtol=FP32_RTOL, atol=FP32_ATOL))
    wt = he_normal_conv_weight(cout, c, 5, 9)
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    assert ops.upconv2x_takes(torch.empty((n, c, h, w), dtype=dtype), cout, 5, 1, 2, filt) or c == 64 or h * w < 300
    H, W = 2 * h, 2 * w
    ts_up, ts = TileMask(n, H, W, DEV), TileMask(n, H, W, DEV)
    out = ops.new_nhwc(n, cout, H, W, DEV, dtype)
    r0 = gaussian_delta(n, cout, H, W, 1.0, 1.0, seed=3)[0]
    res, res_ref = _dev(r0).clone(), r0.clone()
    # dense, sparse (stale tiles), nothing at all, one input only, fused epilogue with an addend
    for step, (da, db, two, act, add) in enumerate([(1.0, 1.0, True, _lib.ACT_NONE, False), (0.03, 0.05, True, _lib.ACT_RELU, False),
                                                    (0.0, 0.0, True, _lib.ACT_NONE, False), (0.2, 0.0, False, _lib.ACT_LEAKY_RELU, True)]):
        def one(d, seed):
            if d == 0.0:
                return torch.zeros(n, c, h, w), torch.zeros(n, 1, h, w, dtype=torch.uint8)
            return gaussian_delta(n, c, h, w, d, 0.5, seed=seed)
        (a, ma), (b, mb) = one(da, 100 + step), one(db, 200 + step)
        a, b = q(a), q(b)
        ref = io.conv_incr(io.interp_incr(a + b if two else a), wt, 1, 2)
        dma, dmb = ma.to(DEV), mb.to(DEV)
        ops.build_mask_tiles(dma, dmb if two else None, n, h, w, _lib.FOOT_UP2X, 0, 0, 0, ts_up)
        ops.build_mask_tiles(ts_up, None, n, H, W, _lib.FOOT_CONV, 5, 1, 2, ts)
        extra = q(gaussian_delta(n, cout, H, W, 1.0, 0.3, seed=7)[0] * ts.pixmask.cpu().float()) if add else None
        poison = lambda t, m: torch.where(m.bool().expand_as(t), t, torch.full_like(t, float("nan")))
        ops.upconv2x_masked(_dev(poison(a, ma), dtype), dma, _dev(poison(b, mb), dtype) if two else None, dmb if two else None, filt, ts,
                            out, None if act == _lib.ACT_NONE else res, act, 0.1, addend=None if extra is None else _dev(extra, dtype))
        got = out.float().cpu()
        z = ref if extra is None else ref + extra
        if act == _lib.ACT_NONE:
            want = z
        else:
            op = torch.relu if act == _lib.ACT_RELU else (lambda t: torch.nn.functional.leaky_relu(t, 0.1))
            want = op(res_ref + z) - op(res_ref)
            res_ref = res_ref + z
            assert torch.allclose(res.cpu(), res_ref, rtol=FP32_RTOL, atol=bf16_atol(ref, 2.0) if bf else FP32_ATOL)
        assert torch.isfinite(got).all()
        assert torch.allclose(got, want, **tol(want)), "step %d max|diff| %.3e of %.3e" % (step, (got - want).abs().max(), want.abs().max())
        assert torch.count_nonzero(got * (1 - ts.pixmask.cpu().float())) == 0
    # the dense twin
    full, dense = TileMask(n, H, W, DEV), ops.new_nhwc(n, cout, H, W, DEV, dtype)
    ops.build_mask_tiles(None, None, n, H, W, _lib.FOOT_CONV, 1, 1, 0, full)
    a, b = q(gaussian_delta(n, c, h, w, 1.0, 0.5, seed=11)[0]), q(gaussian_delta(n, c, h, w, 1.0, 0.5, seed=12)[0])
    bias = torch.linspace(-1, 1, cout)
    ops.upconv2x_refresh(_dev(a, dtype), _dev(b, dtype), filt, bias.to(DEV), full, dense, res, _lib.ACT_RELU)
    pre = io.conv_incr(io.interp_incr(a + b), wt, 1, 2) + bias.view(1, -1, 1, 1)
    assert torch.allclose(res.cpu(), pre, rtol=FP32_RTOL, atol=bf16_atol(pre, 2.0) if bf else 2 * FP32_ATOL)
    assert torch.allclose(dense.float().cpu(), torch.relu(pre), **tol(pre))


@pytest.mark.parametrize("kind", ["white", "smooth"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,cout,h,w", [(1, 256, 128, 33, 44), (1, 128, 64, 66, 88), (2, 128, 64, 25, 35), (1, 64, 32, 132, 176), (4, 256, 128, 30, 40)])
def test_error_against_fp64_beside_the_list_driven_form(n, c, cout, h, w, dtype, kind):
    """The two forms of a decoder layer next to the layer in fp64, over the fp32 weights.
    bf16: each rounds the sum of its inputs (up-sampled or not), its weights (combined or not) and its output to 8 bits, a
    relative error of 1.66e-3 rms each (a mantissa spread evenly over its octave), sqrt(3) of that = 2.87e-3 where the
    products are independent: 3.0e-3 allowed, and 4 % more than the list-driven form on white inputs (whose blend of
    independent pixels spreads the mantissas more evenly: 2.5-3 % measured).  On smooth inputs this form is the closer one:
    its taps' combined weights share less of their roundings (the list-driven form's then add up: 2.75-3.34e-3 measured).
    fp32: the order of the sums and the accumulators are what differs; no more error than the list-driven form's."""
    g = torch.Generator().manual_seed(c + h)
    a, b = (torch.randn(n, c, h, w, generator=g) for _ in range(2))
    if kind == "smooth":
        a, b = (torch.nn.functional.avg_pool2d(t, 5, 1, 2) * 4.0 + 1.0 for t in (a, b))
    wt = he_normal_conv_weight(cout, c, 5, 9)
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    da, db = _dev(a, dtype), _dev(b, dtype)
    # fp64 on the GPU as 25 matrix products over shifted planes of the up-sampled sum
    up = torch.nn.functional.interpolate(da.double() + db.double(), scale_factor=2, mode="bilinear", align_corners=False)
    up = torch.nn.functional.pad(up, (2, 2, 2, 2)).permute(0, 2, 3, 1).contiguous()
    H, W = 2 * h, 2 * w
    ref = sum(up[:, y:y + H, x:x + W].reshape(-1, c) @ filt.plain[:, y, x].double() for y in range(5) for x in range(5))
    ref = ref.view(n, H, W, cout).permute(0, 3, 1, 2)
    ts = TileMask(n, H, W, DEV)
    ops.build_mask_tiles(None, None, n, H, W, _lib.FOOT_CONV, 1, 1, 0, ts)
    err = []
    for form in (lambda out: ops.upconv_masked(da, None, db, None, filt, 5, 2, ts, out),
                 lambda out: ops.upconv2x_masked(da, None, db, None, filt, ts, out)):
        out = ops.new_nhwc(n, cout, H, W, DEV, dtype)
        form(out)
        err.append(((out.double() - ref).norm() / ref.norm()).item())
    print("%s %s %dx%dx%d %d->%d: list-driven %.3e, here %.3e" % (dtype, kind, n, h, w, c, cout, *err))
    if dtype == torch.bfloat16:
        assert err[1] < 3.0e-3 and err[1] <= (1.04 if kind == "white" else 1.0) * err[0], err
    else:
        assert err[1] <= err[0], err


@pytest.mark.parametrize("n,h,w", [(3, 100, 118), (1, 182, 183), (2, 129, 145), (2, 10, 2100), (5, 80, 84)])
def test_fused_tail_at_input_resolution(n, h, w):
    # mie_upconv2x_pred_masked: the last decoder (64 -> 32, bf16) with the 1x1 prediction over its increment and a second
    # delta.  Away from the border the conv runs at the resolution of its inputs, in items of 2 x 4 tiles: tile grids whose
    # inner part is and is not a multiple of an item, last tiles of 2 .. 8 rows, two rows of inner tiles only; NaN in every
    # inactive input pixel; dense, sparse, empty and one-input steps (stale tiles).
    bf = torch.bfloat16
    c, cout, H, W = 64, 32, 2 * h, 2 * w
    q = lambda t: t.to(bf).float()
    wt = he_normal_conv_weight(cout, c, 5, 9)
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    pw = q(torch.randn(cout, generator=torch.Generator().manual_seed(4)) * 0.3)
    pred_w = torch.stack((pw, -0.5 * pw)).contiguous().to(DEV)
    assert ops.upconv_pred_takes(c, cout, 5, 1, 2, filt, bf, _lib.tile_capacity(n, H, W), _lib.ACT_RELU)
    ts_up, ts_dec, ts = (TileMask(n, H, W, DEV) for _ in range(3))
    out = ops.new_nhwc(n, 1, H, W, DEV, bf)
    res_ref, pres_ref = gaussian_delta(n, cout, H, W, 1.0, 1.0, seed=3)[0], gaussian_delta(n, 1, H, W, 1.0, 1.0, seed=5)[0]
    res, pres = _dev(res_ref).clone(), _dev(pres_ref).clone()
    poison = lambda t, m: torch.where(m.bool().expand_as(t), t, torch.full_like(t, float("nan")))
    for step, (da, db, ds, two) in enumerate([(1.0, 1.0, 1.0, True), (0.02, 0.01, 0.1, True), (0.0, 0.0, 0.0, True), (0.05, 0.0, 0.3, False)]):
        def one(ch, hh, ww, d, seed):
            if d == 0.0:
                return torch.zeros(n, ch, hh, ww), torch.zeros(n, 1, hh, ww, dtype=torch.uint8)
            return gaussian_delta(n, ch, hh, ww, d, 0.5, seed=seed)
        (a, ma), (b, mb), (sk, ms) = one(c, h, w, da, 100 + step), one(c, h, w, db, 200 + step), one(cout, H, W, ds, 300 + step)
        a, b, sk = q(a), q(b), q(sk)
        dma, dmb, dms = ma.to(DEV), mb.to(DEV), ms.to(DEV)
        ops.build_mask_tiles(dma, dmb if two else None, n, h, w, _lib.FOOT_UP2X, 0, 0, 0, ts_up)
        ops.build_mask_tiles(ts_up, None, n, H, W, _lib.FOOT_CONV, 5, 1, 2, ts_dec)
        ops.build_mask_tiles(ts_dec, dms, n, H, W, _lib.FOOT_CONV, 1, 1, 0, ts)
        ops.upconv_pred_masked(_dev(poison(a, ma), bf), dma, _dev(poison(b, mb), bf) if two else None, dmb if two else None, filt, ts,
                               res, _lib.ACT_RELU, 0.0, _dev(poison(sk, ms), bf), dms, pred_w, pres, _lib.ACT_SIGMOID, 0.0, out,
                               dense_plane=True)
        conv = io.conv_incr(io.interp_incr(a + b if two else a), wt, 1, 2)
        got_res = res.cpu()
        assert torch.allclose(got_res, res_ref + conv, rtol=BF16_RTOL, atol=bf16_atol(conv, 2.0)), "step %d reservoir %.3e" % (
            step, (got_res - res_ref - conv).abs().max())
        # the tail from the decoder's own sums: what is left is fp32 rounding and y's rounding to bf16, which the kernel does
        y = q(torch.relu(got_res) - torch.relu(res_ref))
        z = (y * pw.view(1, -1, 1, 1) - 0.5 * sk * pw.view(1, -1, 1, 1)).sum(1, keepdim=True)
        want = torch.sigmoid(pres_ref + z) - torch.sigmoid(pres_ref)
        live = ts.pixmask.cpu().float()
        assert torch.allclose(pres.cpu(), pres_ref + z, rtol=1e-5, atol=1e-5), "step %d: %.3e" % (step, (pres.cpu() - pres_ref - z).abs().max())
        assert torch.allclose(out.float().cpu(), want * live, rtol=2 ** -8, atol=1e-5), "step %d: %.3e" % (
            step, (out.float().cpu() - want * live).abs().max())
        assert torch.count_nonzero(out.float().cpu() * (1 - live)) == 0
        res_ref, pres_ref = got_res, pres.cpu()


@pytest.mark.parametrize("kind", ["white", "smooth"])
@pytest.mark.parametrize("n,h,w", [(3, 100, 118), (1, 182, 183), (2, 129, 145)])
def test_fused_tail_error_against_fp64_beside_the_one_tile_form(n, h, w, kind):
    """The two forms of the fused tail (mie_upconv2x_pred_masked, mie_upconv_pred_masked) next to the decoder and the prediction in
    fp64, over the fp32 weights of the decoder.  Each rounds the sum of its inputs (up-sampled or not) and its weights (combined
    or not) to 8 bits before the sums, and the activation increment to 8 bits behind them; the accumulators are fp32 in both.  On
    smooth inputs, as layers see them, this form is the closer one (the decoder's sums 0.64 - 0.67 of the one-tile form's error, the
    prediction's 0.79 - 0.86, its delta 0.83 - 0.93); on white noise the blend of independent pixels spreads the one-tile form's
    mantissas more evenly, as in test_error_against_fp64_beside_the_list_driven_form: 1.01 - 1.03, 1.04 allowed."""
    bf = torch.bfloat16
    c, cout, H, W = 64, 32, 2 * h, 2 * w
    g = torch.Generator().manual_seed(h)
    a, b = (torch.randn(n, c, h, w, generator=g) for _ in range(2))
    if kind == "smooth":
        a, b = (torch.nn.functional.avg_pool2d(t, 5, 1, 2) * 4.0 + 1.0 for t in (a, b))
    skip = torch.randn(n, cout, H, W, generator=g)
    wt = he_normal_conv_weight(cout, c, 5, 9)
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    pred_w = (torch.randn(2, cout, generator=g) * 0.3).to(DEV)
    da, db, ds = _dev(a, bf), _dev(b, bf), _dev(skip, bf)
    ts = TileMask(n, H, W, DEV)
    ops.build_mask_tiles(None, None, n, H, W, _lib.FOOT_CONV, 1, 1, 0, ts)
    r0, p0 = (torch.randn(n, k, H, W, generator=g) for k in (cout, 1))
    up = torch.nn.functional.interpolate(da.double() + db.double(), scale_factor=2, mode="bilinear", align_corners=False)
    up = torch.nn.functional.pad(up, (2, 2, 2, 2)).permute(0, 2, 3, 1).contiguous()
    conv = sum(up[:, y:y + H, x:x + W].reshape(-1, c) @ filt.plain[:, y, x].double() for y in range(5) for x in range(5)).view(n, H, W, cout)
    r = r0.to(DEV).double().permute(0, 2, 3, 1)
    y = torch.relu(r + conv) - torch.relu(r)
    z = (y * pred_w[0].double() + ds.double().permute(0, 2, 3, 1) * pred_w[1].double()).sum(3)
    p = p0.to(DEV).double()[:, 0]
    delta = torch.sigmoid(p + z) - torch.sigmoid(p)
    err = []
    for dense in (False, True):
        res, pres, out = _dev(r0).clone(), _dev(p0).clone(), ops.new_nhwc(n, 1, H, W, DEV, bf)
        assert ops.upconv_pred_takes(c, cout, 5, 1, 2, filt, bf, ts.capacity, _lib.ACT_RELU)
        ops.upconv_pred_masked(da, None, db, None, filt, ts, res, _lib.ACT_RELU, 0.0, ds, None, pred_w, pres, _lib.ACT_SIGMOID, 0.0, out,
                               dense_plane=dense)
        rel = lambda got, want: ((got - want).norm() / want.norm()).item()
        err.append((rel(res.double().permute(0, 2, 3, 1) - r, conv), rel(pres.double()[:, 0] - p, z), rel(out.double()[:, 0], delta)))
    print("%s %dx%dx%d: decoder / prediction sums, delta: one tile %.3e %.3e %.3e, here %.3e %.3e %.3e" % (kind, n, h, w, *err[0], *err[1]))
    assert err[1][0] < 3.0e-3, err      # (three roundings of 1.66e-3 rms; the prediction's sums cancel, more or less, by chance)
    for one, here in zip(*err):
        assert here <= (1.04 if kind == "white" else 1.0) * one, err


@pytest.mark.parametrize("n,h,w", [(3, 100, 118), (1, 150, 170), (8, 35, 67), (2, 20, 801)])
def test_decoder_conv_of_many_items(n, h, w):
    # 128 -> 64 channels in bf16 from three items of 8 x 16 positions a workgroup on: the persistent kernel makes all but the
    # border's positions (the step with an addend stays with the other form).  Planes whose last item is and is not
    # filled.
    test_decoder_conv_at_input_resolution(n, 128, 64, h, w, torch.bfloat16)


@pytest.mark.parametrize("form", ["blocks", "list"])
@pytest.mark.parametrize("n,c,cout,h,w,dtype", [(1, 128, 64, 9, 16, torch.bfloat16), (1, 128, 64, 150, 170, torch.bfloat16), (8, 128, 64, 35, 67, torch.bfloat16),
                                                (1, 64, 32, 20, 24, torch.bfloat16), (1, 64, 32, 182, 183, torch.bfloat16), (1, 128, 64, 33, 20, torch.float32)])
def test_pixels_outside_the_mask_keep_their_reservoir(n, c, cout, h, w, dtype, form):
    # The contract of every matrix-core conv: at a pixel of an active tile that lies outside the output pixel mask the delta is
    # zero and the reservoir is not touched -- also where it holds an infinity or a NaN, whose increment would be NaN.  Planes
    # that the blocks, the persistent kernel of 128 -> 64 channels and the one of 64 -> 32 (list-driven, from 2048 tiles) take.
    H, W = 2 * h, 2 * w
    filt = ops.ConvFilter(he_normal_conv_weight(cout, c, 5, 9).permute(1, 2, 3, 0).contiguous().to(DEV))
    ts_up, ts = TileMask(n, H, W, DEV), TileMask(n, H, W, DEV)
    out = ops.new_nhwc(n, cout, H, W, DEV, dtype)
    odd = torch.tensor([float("inf"), float("-inf"), float("nan")])
    for step, act in enumerate((None, _lib.ACT_NONE, _lib.ACT_RELU, _lib.ACT_LEAKY_RELU)):
        (a, ma), (b, mb) = (gaussian_delta(n, c, h, w, d, 0.5, seed=40 + 10 * k + step) for k, d in enumerate((0.02, 0.05)))
        dma, dmb = ma.to(DEV), mb.to(DEV)
        ops.build_mask_tiles(dma, dmb, n, h, w, _lib.FOOT_UP2X, 0, 0, 0, ts_up)
        ops.build_mask_tiles(ts_up, None, n, H, W, _lib.FOOT_CONV, 5, 1, 2, ts)
        off = ~ts.pixmask.cpu().bool().expand(n, cout, H, W)
        r0 = gaussian_delta(n, cout, H, W, 1.0, 1.0, seed=3)[0]
        r0[off] = odd[torch.arange(int(off.sum())) % 3]
        res = None if act is None else _dev(r0).clone()
        args = (_dev(a, dtype), dma, _dev(b, dtype), dmb, filt)
        if form == "blocks":
            ops.upconv2x_masked(*args, ts, out, res, act or _lib.ACT_NONE, 0.1)
        else:
            ops.upconv_masked(*args, 5, 2, ts, out, res, act or _lib.ACT_NONE, 0.1)
        got = out.float().cpu()
        assert torch.isfinite(got).all() and torch.count_nonzero(got[off]) == 0, "step %d: %d not finite" % (step, (~torch.isfinite(got)).sum())
        assert torch.count_nonzero(got[~off]) > 0
        if res is not None:
            bits = lambda t: t.contiguous().view(torch.int32)
            assert torch.equal(bits(res.cpu())[off], bits(r0)[off])


# fp32, 64 or 96 channels, more workgroups than two to a CU: the four phases in one workgroup.  Blocks and strips
# cut off at both sides, one row of blocks, planes of strips only (which stay with the other form), slabs, samples.
@pytest.mark.parametrize("n,c,cout,h,w", [(1, 64, 32, 100, 140), (2, 96, 64, 40, 41), (1, 64, 32, 3, 1200), (1, 64, 32, 1200, 3),
                                          (1, 64, 32, 2, 2200), (9, 64, 96, 17, 10)])
def test_decoder_conv_of_few_channels_on_many_blocks(n, c, cout, h, w):
    assert _lib.lib().mie_f16x2_takes_upconv2x(n, h, w, c, cout) == (h > 2)
    test_decoder_conv_at_input_resolution(n, c, cout, h, w, torch.float32)
    if n == 1 and h > 2 and c == 64:
        test_pixels_outside_the_mask_keep_their_reservoir(n, c, cout, h, w, torch.float32, "blocks")


# bf16, 64 channels, more such workgroups than CUs
@pytest.mark.parametrize("n,c,cout,h,w", [(2, 64, 32, 100, 140), (1, 64, 96, 75, 74), (5, 64, 32, 34, 90), (1, 64, 32, 2100, 3), (1, 64, 32, 3, 2100)])
def test_decoder_conv_of_one_chunk_on_many_blocks(n, c, cout, h, w):
    assert _lib.lib().mie_all_phases_upconv2x(n, h, w, c, cout, _lib.DTYPE_BF16)
    test_decoder_conv_at_input_resolution(n, c, cout, h, w, torch.bfloat16)
    test_pixels_outside_the_mask_keep_their_reservoir(n, c, cout, h, w, torch.bfloat16, "blocks")


# ... whose layers a network does not take there: upconv_masked holds a + b in 32 bits up to the blend, this form rounds it to bf16
@pytest.mark.parametrize("n,cout,h,w", [(2, 32, 100, 140), (1, 96, 75, 74), (8, 32, 240, 320)])
def test_decoders_of_one_chunk_keep_the_sum_of_their_inputs_in_32_bits(n, cout, h, w):
    filt = ops.ConvFilter(torch.zeros(64, 5, 5, cout, device=DEV))
    for refresh in (False, True):
        assert not ops.upconv2x_takes(torch.empty((n, 64, h, w), dtype=torch.bfloat16), cout, 5, 1, 2, filt, refresh)
