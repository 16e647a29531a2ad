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


# chunks of 32 channels: fewer, as many and more than the 8 waves, 1, 2 or 4 of them a chunk, of one input or two; planes of one
# pixel, of less than two rows or columns of a tile, of whole tiles; the last shapes at which two rows a workgroup (256), four
# (256 / 512) and the form itself are taken, and the first beyond
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c1,c2,cout,h,w,pad", [
    (1, 64, 0, 32, 1, 1, 1), (2, 64, 64, 64, 3, 2, 1), (1, 192, 0, 32, 5, 9, 1), (1, 256, 128, 96, 13, 11, 0), (1, 320, 0, 32, 9, 7, 2),
    (1, 512, 0, 64, 16, 17, 1), (3, 256, 64, 32, 12, 8, 3), (1, 128, 0, 256, 16, 16, 1), (1, 64, 0, 256, 16, 24, 1),
    (1, 64, 64, 512, 16, 16, 1), (1, 64, 0, 512, 16, 24, 1), (2, 64, 0, 512, 16, 16, 1), (1, 128, 0, 512, 24, 24, 1)])
def test_whole_contraction_in_a_workgroup(n, c1, c2, cout, h, w, pad, dtype):
    cin, bf = c1 + c2, dtype == torch.bfloat16
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    wt = q(he_normal_conv_weight(cout, cin, 3, 21))
    filt = ops.ConvFilter(wt.permute(1, 2, 3, 0).contiguous().to(DEV))
    ho, wo = ops.conv_out_size(h, w, 3, 1, pad)
    ts = TileMask(n, ho, wo, DEV)
    tiles = ts.capacity
    takes = _lib.lib().mie_conv_needs_no_workspace(3, 1, c1, c2, cout, tiles, _lib.DTYPE_BF16 if bf else _lib.DTYPE_F32_BF16X3)
    assert takes == (2 * tiles * (cout // 16) <= (512 if bf else 256))
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
        live = F.max_pool2d(F.pad(m.float(), (pad,) * 4), 3, 1) > 0
        add = q(gaussian_delta(n, cout, ho, wo, 1.0, 0.3, seed=400 + step)[0]) * live if step else None
        dm = m.to(DEV)
        x = torch.where(m.bool(), d, torch.full((), float("nan")))       # what an inactive pixel holds is not read
        x1, x2 = _dev(x[:, :c1]).to(dtype), _dev(x[:, c1:]).to(dtype) if c2 else None
        ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_CONV, 3, 1, pad, ts)
        sums = F.conv2d(d.double(), wt.double(), padding=pad) + (0 if add is None else add.double())
        bound = F.conv2d(d.double().abs(), wt.double().abs(), padding=pad) + (0 if add is None else add.double().abs())
        # three fp32 roundings of sum |x||w|, as for the other forms, and the reservoir's own, step upon step
        before, tol = tol, tol + 4e-7 * bound + 2.0 ** -23 * (ref.abs() + sums.abs())
        for i, ws in enumerate((None, split)):
            ops.conv_masked(x1, dm, x2, None if x2 is None else dm, filt, 3, 1, pad, ts, outs[i], ress[i], _lib.ACT_RELU, 0.0,
                            _lib.PATH_AUTO, None if add is None else _dev(add).to(dtype), workspace=ws)
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
        ops.conv_refresh(_dev(d[:, :c1]).to(dtype), _dev(d[:, c1:]).to(dtype) if c2 else None, filt, bias.to(DEV), 3, 1, pad, every, y, res)
        want = F.conv2d(d.double(), wt.double(), bias.double(), padding=pad)
        assert ((res.cpu().double() - want).abs() <= 4e-7 * bound + 2.0 ** -23 * want.abs()).all()
