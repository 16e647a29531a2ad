"""The stacked gates conv of a ConvGRU with the gate math as its epilogue (mie_conv_gru_masked) against fp64, beside the two calls."""
import pytest
import torch
import torch.nn.functional as F

from maskedincrementeval_amd import _lib, ops
from maskedincrementeval_amd.evflownet_incr import ConvGRUIncr
from maskedincrementeval_amd.masked_types import TileMask
from maskedincrementeval_amd.synthetic import gaussian_delta, he_normal_conv_weight

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(t):
    return ops.as_nhwc(t.to(DEV).contiguous(memory_format=torch.channels_last))


# planes of one pixel, of part of a tile, of a workgroup's 2, 4 and 8 rows and the last shapes at which each is taken; then slabs
# of 32, 64 and 128 columns, of tiles cut off at both edges; filters with more rows than the input has channels
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,cin,more,hid,h,w", [
    (1, 64, 0, 16, 1, 1), (2, 64, 64, 16, 3, 2), (1, 192, 16, 48, 13, 11), (1, 512, 512, 128, 16, 16), (1, 64, 0, 256, 16, 17),
    (1, 64, 64, 32, 64, 64), (1, 128, 0, 64, 31, 64), (1, 64, 0, 64, 41, 57), (1, 64, 64, 16, 90, 93), (1, 64, 0, 32, 90, 93),
    (1, 128, 0, 32, 155, 160), (1, 64, 0, 64, 90, 93), (2, 64, 0, 64, 117, 113)])
def test_gates_conv_and_gru_in_one(n, cin, more, hid, h, w, dtype):
    bf = dtype == torch.bfloat16
    q = (lambda t: t.to(dtype).float()) if bf else (lambda t: t)
    assert ops.conv_gru_takes(cin, cin + more, hid, dtype)
    wt = q(he_normal_conv_weight(2 * hid, cin + more, 3, 31))
    order = ops.gru_interleave_index(hid)
    assert torch.equal(order.sort().values, torch.arange(2 * hid))
    cell = ConvGRUIncr(cin, hid, 3)
    for gate, part in ((cell.update_gate, wt[:hid]), (cell.out_gate, wt[hid:])):
        gate.weight = torch.nn.Parameter(part)
    assert torch.equal(cell._stacked_filter(True).plain, wt[order].permute(1, 2, 3, 0))
    filt, stacked = (ops.ConvFilter(t.permute(1, 2, 3, 0).contiguous().to(DEV)) for t in (wt[order], wt))
    gen = torch.Generator().manual_seed(6)
    ref = torch.randn(n, 2 * hid, h, w, generator=gen).double()           # pre-activations: update | candidate
    tol = torch.zeros_like(ref)
    forms = [[_dev(r.float()) for r in ref.split(hid, 1)] for _ in range(2)]
    outs = [ops.new_nhwc(n, hid, h, w, DEV, dtype).zero_() for _ in range(2)]       # (tiles neither active nor stale aren't written)
    both = ops.new_nhwc(n, 2 * hid, h, w, DEV, dtype)
    ts = TileMask(n, h, w, DEV)
    state = lambda r: r[:, :hid].sigmoid() * r[:, hid:].tanh()
    for step, dens in enumerate((0.3, 0.02, 1.0)):
        d, m = gaussian_delta(n, cin, h, w, dens, 0.5, seed=500 + step)
        d = q(d)
        x = _dev(torch.where(m.bool(), d, torch.full((), float("nan")))).to(dtype)      # what an inactive pixel holds is not read
        dm = m.to(DEV)
        live = F.max_pool2d(F.pad(m.float(), (1,) * 4), 3, 1) > 0
        ops.build_mask_tiles(dm, None, n, h, w, _lib.FOOT_CONV, 3, 1, 1, ts)
        sums, bound = (F.conv2d(t, v[:, :cin], padding=1) for t, v in ((d.double(), wt.double()), (d.double().abs(), wt.double().abs())))
        # as in test_gpu_conv_deep.py: fp32 roundings of sum |x||w| and the reservoir's own, step upon step
        before, ref, was = ref, ref + sums, tol
        tol = tol + 4e-7 * bound + 2.0 ** -23 * (ref.abs() + sums.abs())
        want = state(ref) - state(before)
        # sigmoid and tanh carry errors of their arguments with slopes of at most 1/4 and 1; their own errors and the product's
        # roundings are some 2^-24 of values below 2 (16 of them); bf16: the result's rounding
        err = was + tol
        tol_h = 0.25 * err[:, :hid] + err[:, hid:] + 16 * 2.0 ** -24 * 2 + (2.0 ** -8 * want.abs() if bf else 0)
        ops.conv_gru_incr(x, dm, filt, ts, *forms[0], outs[0])
        ops.conv_masked(x, dm, None, None, stacked, 3, 1, 1, ts, both)
        ops.convgru_gates_incr(both, *forms[1], outs[1], ts)
        torch.cuda.synchronize()
        got = torch.cat([r.cpu().double() for r in forms[0]], 1)
        assert ((got - ref).abs() <= tol).all(), (step, ((got - ref).abs() / tol.clamp(min=1e-30)).max())
        h_d = outs[0].cpu().double()
        assert ((h_d - want).abs() <= tol_h).all(), (step, ((h_d - want).abs() / tol_h).max())
        assert not h_d[~live.expand_as(h_d)].any()                         # (stale tiles and pixels off the mask too)
        if not bf:        # (the two calls round bf16 gates in between)
            errs = [(torch.cat(f, 1).cpu().double() - ref).abs().max().item() for f in forms]
            assert errs[0] <= 2 * errs[1] + 1e-7, errs
            assert ((outs[1].cpu().double() - want).abs() <= tol_h).all()


def test_what_it_refuses():
    filt = ops.ConvFilter(torch.randn(64, 3, 3, 64, device=DEV))
    for cin, hid, dt in ((64, 24, torch.float32), (48, 32, torch.float32), (32, 32, torch.bfloat16)):
        assert not ops.conv_gru_takes(cin, 64, hid, dt)
    x, ts = ops.new_nhwc(1, 64, 8, 8, DEV).zero_(), TileMask(1, 8, 8, DEV)
    m = torch.ones(1, 1, 8, 8, dtype=torch.uint8, device=DEV)
    ops.build_mask_tiles(m, None, 1, 8, 8, _lib.FOOT_CONV, 3, 1, 1, ts)
    u, c, dh = (ops.new_nhwc(1, 32, 8, 8, DEV).zero_() for _ in range(3))
    with pytest.raises(Exception, match="distinct"):
        ops.conv_gru_incr(x, m, filt, ts, u, u, dh)
    with pytest.raises(ValueError):
        ops.conv_gru_incr(x, m, filt, ts, u, c, dh[:, :16])
    for wrong in (TileMask(2, 8, 8, DEV), TileMask(1, 8, 16, DEV)):
        with pytest.raises(ValueError, match="tile set"):
            ops.conv_gru_incr(x, m, filt, wrong, u, c, dh)
    with pytest.raises(ValueError, match="columns"):
        ops.conv_gru_incr(x, m, ops.ConvFilter(torch.randn(64, 3, 3, 65, device=DEV)), ts, u, c, dh)
    plain, mc = filt.for_dtype(torch.float32, False)
    assert _lib.lib().mie_conv_gru_masked(x.data_ptr(), m.data_ptr(), 64, 8, 8, plain.data_ptr(), mc.data_ptr(), 64, 32, ts.ref,
                                          u.data_ptr(), c.data_ptr(), dh.data_ptr(), _lib.DTYPE_F32, None) == -2
