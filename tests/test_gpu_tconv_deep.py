"""The 3x3 stride-2 transposed conv on planes of few blocks in one launch (csrc/mie_conv_deep.hip) against fp64."""
import pytest
import torch
import torch.nn.functional as F

from maskedincrementeval_amd import _lib, ops
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.synthetic import gaussian_delta

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(t):
    return ops.as_nhwc(t.to(DEV).contiguous(memory_format=torch.channels_last))


# chunks of 32 channels: fewer than the eight waves, as many, more, no multiple; planes of one pixel, of part of the rows of a
# workgroup, cut off at both edges; the last shapes of two rows a workgroup, of four in one round and in two, and the first beyond
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c1,c2,cout,h,w", [
    (1, 128, 0, 32, 1, 1), (2, 64, 64, 32, 5, 9), (1, 576, 0, 32, 17, 10), (1, 256, 256, 256, 16, 15), (1, 192, 64, 512, 13, 16),
    (1, 512, 512, 64, 7, 6), (1, 128, 128, 128, 31, 32), (1, 128, 64, 128, 33, 31), (1, 64, 64, 64, 63, 64), (1, 128, 0, 64, 65, 64), (1, 64, 0, 64, 16, 16)])
def test_transposed_conv_in_one_launch(n, c1, c2, cout, h, w, dtype):
    bf, cin = dtype == torch.bfloat16, c1 + c2
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    wt = q(torch.randn(cin, cout, 3, 3, generator=torch.Generator().manual_seed(cin + cout)) * (2.0 / (9 * cin)) ** 0.5)
    filt = ops.ConvFilter(wt.permute(0, 2, 3, 1).contiguous().to(DEV))
    ho, wo = 2 * h, 2 * w
    ts, blocks, out = TileMask(n, ho, wo, DEV), TileMask(n, h, w, DEV), ops.new_nhwc(n, cout, ho, wo, DEV, dtype)
    ref = torch.randn(n, cout, ho, wo, generator=torch.Generator().manual_seed(5)).double()
    res, tol = _dev(ref.float()), torch.zeros_like(ref)
    up = lambda x, f: F.conv_transpose2d(x.double(), f.double(), stride=2, padding=1, output_padding=1)
    for step, dens in enumerate((0.3, 0.03, 1.0)):
        parts, masks = [], []
        for i, c in enumerate((c1, c2)):
            d, m = gaussian_delta(n, c, h, w, dens / (1 + i), 0.5, seed=700 + 10 * step + i) if c else (torch.zeros(n, 0, h, w), torch.zeros(n, 1, h, w, dtype=torch.uint8))
            parts.append(q(d))
            masks.append(m)
        d, m = torch.cat(parts, 1), masks[0] | masks[1]
        xs = [_dev(torch.where(k.bool(), p, torch.full((), float("nan")))).to(dtype) if p.shape[1] else None for p, k in zip(parts, masks)]
        ms = [k.to(DEV) if p.shape[1] else None for p, k in zip(parts, masks)]
        ops.build_mask_tiles(ms[0], ms[1], n, h, w, _lib.FOOT_TCONV, 3, 2, 1, ts)
        ops.build_mask_tiles(ts, None, n, ho, wo, _lib.FOOT_CONV, 2, 2, 0, blocks)
        live = up(m.float(), torch.ones(1, 1, 3, 3)) > 0
        add = q(gaussian_delta(n, cout, ho, wo, 1.0, 0.3, seed=800 + step)[0]) * live
        sums, bound = up(d, wt) + add.double(), up(d.abs(), wt.abs()) + add.double().abs()
        # as in test_gpu_conv_deep.py: three fp32 roundings of sum |x||w| and the reservoir's own, step upon step
        before, tol = tol, tol + 4e-7 * bound + 2.0 ** -23 * (ref.abs() + sums.abs())
        ops.tconv2x_masked(xs[0], ms[0], xs[1], ms[1], filt, 3, ts, blocks, out, res, _lib.ACT_RELU, 0.0, _dev(add).to(dtype))
        torch.cuda.synchronize()
        off = (res.cpu().double() - (ref + sums)).abs()
        assert (off <= tol).all(), (step, (off / tol.clamp(min=1e-30)).max())
        want, got = (ref + sums).clamp(min=0) - ref.clamp(min=0), out.cpu().double()
        assert ((got - want).abs() <= (before + tol) * (1 + 2.0 ** -8) + (2.0 ** -8 if bf else 0.0) * want.abs()).all(), step
        assert not got[~live.expand_as(got)].any()
        ref = ref + sums
    bias = torch.randn(cout, generator=torch.Generator().manual_seed(6))
    for t, hh, ww in ((ts, ho, wo), (blocks, h, w)):
        ops.build_mask_tiles(None, None, n, hh, ww, _lib.FOOT_CONV, 1, 1, 0, t)
    ops.tconv2x_refresh(_dev(d[:, :c1]).to(dtype), _dev(d[:, c1:]).to(dtype) if c2 else None, filt, bias.to(DEV), 3, ts, blocks, out, res)
    want = up(d, wt) + bias.double().view(1, -1, 1, 1)
    assert ((res.cpu().double() - want).abs() <= 4e-7 * bound + 2.0 ** -23 * want.abs()).all()


# fp32 of very many channels: split where there is a workspace that holds two parts, else one launch
def test_transposed_conv_of_very_many_channels():
    n, c1, c2, cout, h, w = 1, 768, 704, 32, 5, 9
    wt = torch.randn(c1 + c2, cout, 3, 3, generator=torch.Generator().manual_seed(2)) * (2.0 / (9 * (c1 + c2))) ** 0.5
    filt = ops.ConvFilter(wt.permute(0, 2, 3, 1).contiguous().to(DEV))
    ts, blocks = TileMask(n, 2 * h, 2 * w, DEV), TileMask(n, h, w, DEV)
    d, m = gaussian_delta(n, c1 + c2, h, w, 0.4, 0.5, seed=3)
    dm = m.to(DEV)
    up = lambda x, f: F.conv_transpose2d(x.double(), f.double(), stride=2, padding=1, output_padding=1)
    want, bound = up(d, wt), up(d.abs(), wt.abs())
    got = {}
    for name, ws in (("shared", None), ("own", torch.full((ops.SPLIT_WORKSPACE_BYTES // 4,), float("nan"), device=DEV)),
                     ("too small", torch.full((4 * h * w * cout,), float("nan"), device=DEV)), ("none", False)):
        ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_TCONV, 3, 2, 1, ts)
        ops.build_mask_tiles(ts, None, n, 2 * h, 2 * w, _lib.FOOT_CONV, 2, 2, 0, blocks)
        out, res = ops.new_nhwc(n, cout, 2 * h, 2 * w, DEV), ops.new_nhwc(n, cout, 2 * h, 2 * w, DEV)
        ops.tconv2x_masked(_dev(d[:, :c1]), dm, _dev(d[:, c1:]), dm, filt, 3, ts, blocks, out, res, workspace=ws)
        assert ((res.cpu().double() - want).abs() <= 4e-7 * bound).all(), name
        assert ws is None or ws is False or torch.isfinite(ws).any() == (name == "own")
        got[name] = res
    assert torch.equal(got["shared"], got["own"]) and torch.equal(got["too small"], got["none"])


# two more input channels in front (a part whose mask the wide parts' covers): every phase, planes cut off at both edges, two and four rows
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c1,c2,cout,h,w", [(1, 128, 0, 32, 1, 1), (2, 64, 64, 32, 5, 9), (1, 128, 128, 128, 31, 32), (1, 64, 64, 64, 63, 64),
                                              (1, 64, 0, 32, 13, 11), (2, 64, 64, 32, 100, 125), (1, 64, 0, 64, 150, 170), (1, 64, 0, 128, 150, 170)])
def test_transposed_conv_with_a_leading_part(n, c1, c2, cout, h, w, dtype):
    bf, cin = dtype == torch.bfloat16, c1 + c2
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    wt = q(torch.randn(2 + cin, cout, 3, 3, generator=torch.Generator().manual_seed(cin)) * (2.0 / (9 * cin)) ** 0.5)
    filt = ops.ConvFilter(wt.permute(0, 2, 3, 1).contiguous().to(DEV))
    ho, wo = 2 * h, 2 * w
    ts, blocks, out = TileMask(n, ho, wo, DEV), TileMask(n, h, w, DEV), ops.new_nhwc(n, cout, ho, wo, DEV, dtype)
    assert ops.tconv2x_takes_lead(2, c1, c2, cout, 3, dtype)
    up = lambda x, f: F.conv_transpose2d(x.double(), f.double(), stride=2, padding=1, output_padding=1)
    ref = torch.zeros(n, cout, ho, wo, dtype=torch.float64)
    res, tol = _dev(ref.float()), torch.zeros_like(ref)
    for step, dens in enumerate((0.2, 1.0)):
        d, m = gaussian_delta(n, cin, h, w, dens, 0.5, seed=900 + step)
        m0 = m if step else m * (torch.rand(m.shape, generator=torch.Generator().manual_seed(3)) < 0.5).to(m.dtype)
        d0 = q(torch.randn(n, 2, h, w, generator=torch.Generator().manual_seed(4 + step))) * m0
        d = torch.cat([d0, q(d)], 1)
        x = torch.where(torch.cat([m0.expand(-1, 2, -1, -1), m.expand(-1, cin, -1, -1)], 1).bool(), d, torch.full((), float("nan"))).to(dtype)
        dm, dm0 = m.to(DEV), m0.to(DEV)
        ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_TCONV, 3, 2, 1, ts)
        ops.build_mask_tiles(ts, None, n, ho, wo, _lib.FOOT_CONV, 2, 2, 0, blocks)
        ops.tconv2x_masked(_dev(x[:, 2:2 + c1]), dm, _dev(x[:, 2 + c1:]) if c2 else None, dm if c2 else None, filt.rows(2, 2 + cin), 3, ts, blocks,
                           out, res, lead=(_dev(x[:, :2]), dm0 if step == 0 else None, filt.rows(0, 2)))
        torch.cuda.synchronize()
        sums, bound = up(d, wt), up(d.abs(), wt.abs())
        tol = tol + 4e-7 * bound + 2.0 ** -23 * (ref.abs() + sums.abs())
        ref = ref + sums
        assert ((res.cpu().double() - ref).abs() <= tol).all(), step
        got = out.cpu().double()
        assert ((got - sums).abs() <= 2 * tol + (2.0 ** -8 if bf else 0.0) * sums.abs()).all(), step
    with pytest.raises(ValueError):
        ops.tconv2x_masked(_dev(x[:, 2:2 + c1]), dm, _dev(x[:, 2 + c1:]) if c2 else None, dm if c2 else None, filt.rows(2, 2 + cin), 3, ts, blocks,
                           out, res, lead=(_dev(x[:, :1]), dm0, filt.rows(0, 1)))


def test_where_a_leading_part_goes_along():
    assert not ops.tconv2x_takes_lead(2, 96, 0, 64, 3, torch.float32) and not ops.tconv2x_takes_lead(2, 128, 0, 64, 5, torch.float32)
    assert not ops.tconv2x_takes_lead(3, 128, 0, 64, 3, torch.bfloat16) and not ops.tconv2x_takes_lead(2, 128, 0, 48, 3, torch.bfloat16)
