"""Sizes at which the tile loops, the launch rules and the result-store rules of the GPU kernels change: one voxel less and
more than a tile, one workgroup's tiles, the first second round of the persistent loops, and the size limit between
cached and streaming stores.  Expected values come from the CPU oracle or from the unfused ops that it pins."""
import pytest
import torch

import oracle
from conftest import cpu_gen, rand_cl3d, rand_dw_weight
from kerops_amd.ops.addition import AddStats, AddStatsBackward
from kerops_amd.ops.avgpool import AvgPoolCeilStats, AvgPoolCeilStatsBackward
from kerops_amd.ops.bnrelu import ApplyBNReLU, ApplyBNReLUBackward
from kerops_amd.ops.conv import DWConv, DWConvBackward, DWConvStats, DWConvWGRAD
from kerops_amd.ops.fused import DWSepBlock
from kerops_amd.ops.linear import (ApplyBNReLULinearAdd, ApplyBNReLULinearBackward, LinBReLULinAdd,
                                   LinBReLULinBackward, ReLULinearAdd, ReLULinearBackward)
from kerops_amd.ops.quantization import DequantUint8Window, QuantInt8Sym, QuantUint8Window
from kerops_amd.ops.stats import Stats, StatsBackward
from kerops_amd.settings import stream_table

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
CHANNELS = [(16, 16), (16, 32), (32, 16), (16, 128), (128, 16), (32, 64), (64, 64), (64, 128), (128, 128)]


def bits(t):
    return t.contiguous().view(torch.int16)


def flat(g, v, c):
    return rand_cl3d(g, 1, c, v, 1, 1)


def matrix(g, cin, cout):
    return (torch.randn(cin, cout, generator=g) / cin ** 0.5).half()


@pytest.mark.parametrize('cin,cout', CHANNELS)
@pytest.mark.parametrize('v', [1, 63, 65, 127, 129, 255, 257])
def test_relu_linear_backward_tile_edges(cin, cout, v):
    g = cpu_gen(v * 1000 + cin + cout)
    x, grad, w = flat(g, v, cin), flat(g, v, cout), matrix(g, cin, cout)
    dx, dw = ReLULinearBackward(x.to(DEV), grad.to(DEV), w.to(DEV), out_dtype=torch.float32)
    ref_dx, ref_dw = oracle.relu_linear_bwd(x, grad, w)
    # fp32 sums of at most 128 products against fp64, then one rounding to fp16
    assert (dx.cpu().float() - ref_dx.float()).abs().max() <= 2.0 ** -9 * max(1.0, ref_dx.abs().max().item())
    # fp32 sums of at most 257 products: 257 * 2^-24
    assert ((dw.cpu().double() - ref_dw).norm() / ref_dw.norm()).item() < 257 * 2.0 ** -24


# (input channels, output channels) -> voxels of a tile, workgroups from half a million voxels on, matrix instructions that
# one accumulator of the weight gradient takes per tile
LINEAR_TILES = {(16, 16): (128, 768, 1), (16, 32): (128, 512, 1), (32, 16): (128, 512, 1), (32, 32): (64, 768, 0.5),
                (16, 64): (128, 512, 2), (64, 16): (64, 512, 1), (32, 64): (64, 512, 1), (64, 64): (64, 512, 2),
                (16, 128): (64, 768, 2), (64, 128): (64, 512, 2), (128, 128): (64, 512, 4)}


@pytest.mark.parametrize('cin,cout', LINEAR_TILES)
def test_relu_linear_backward_many_tiles(cin, cout):
    # every workgroup runs two tiles, some a third, ragged one
    tile, workgroups, _ = LINEAR_TILES[cin, cout]
    v = 2 * workgroups * tile + 3 * tile // 2 + 5
    g = cpu_gen(cin + 3 * cout)
    x, grad, w = flat(g, v, cin), flat(g, v, cout), matrix(g, cin, cout)
    dx, dw = ReLULinearBackward(x.to(DEV), grad.to(DEV), w.to(DEV), out_dtype=torch.float32)
    ref_dx, ref_dw = oracle.relu_linear_bwd(x, grad, w)
    # fp32 sums of at most 128 products against fp64, then one rounding to fp16
    assert (dx.cpu().float() - ref_dx.float()).abs().max() <= 2.0 ** -9 * max(1.0, ref_dx.abs().max().item())
    # one voxel too many, missing or counted twice shifts dw by about 1 / sqrt(v), 4e-3 and more
    assert ((dw.cpu().double() - ref_dw).norm() / ref_dw.norm()).item() < 2.0 ** -20


# A rounding to fp32 leaves 0.42 * 2^-24 of its value (rms over the values of a binade).  Inputs ~ N(0, 1): a running sum of
# n equal parts that is rounded r times a part ends with a relative error of 0.42 * 2^-24 * sqrt(r (n + 1) / 2).
@pytest.mark.parametrize('cin,cout', LINEAR_TILES)
def test_weight_gradient_error_of_large_volumes(cin, cout):
    v = 900037
    tile, workgroups, per_tile = LINEAR_TILES[cin, cout]
    gen = torch.Generator(DEV).manual_seed(cin + cout)
    x = torch.randn(v, cin, device=DEV, generator=gen).half()
    grad = torch.randn(v, cout, device=DEV, generator=gen).half()
    w = matrix(cpu_gen(), cin, cout).to(DEV)
    _, dw = ReLULinearBackward(x.view(1, v, 1, 1, cin).permute(0, 4, 1, 2, 3), grad.view(1, v, 1, 1, cout).permute(0, 4, 1, 2, 3),
                               w, out_dtype=torch.float32)
    ref = torch.relu(x).double().t().contiguous() @ grad.double()
    error = ((dw.double() - ref).norm() / ref.norm()).item()
    tiles = v / tile / workgroups
    if (cin, cout) == (128, 128):  # a chain of four instructions per tile, one addition per tile
        parts = 2 * (4 + 1) / 2 + (tiles + 1) / 2
    else:                          # chains over the tiles, each rounded twice per instruction
        parts = 2 * (tiles * per_tile + 1) / 2
    parts += 2                     # the row of the workgroup, the result
    # a fifth above the expectation: the scatter over the results (256 of them at 16 -> 16), the downward part of the roundings
    assert error < 1.2 * 0.42 * 2.0 ** -24 * parts ** 0.5, (error, parts)


@pytest.mark.parametrize('cin,cout', [(16, 16), (64, 64), (128, 32), (128, 128)])
def test_scale_and_shift_gradient_error_of_large_volumes(cin, cout):
    v = 900037
    gen = torch.Generator(DEV).manual_seed(cin - cout)
    x = torch.randn(v, cin, device=DEV, generator=gen).half().view(1, v, 1, 1, cin).permute(0, 4, 1, 2, 3)
    grad = torch.randn(v, cout, device=DEV, generator=gen).half().view(1, v, 1, 1, cout).permute(0, 4, 1, 2, 3)
    w = matrix(cpu_gen(), cin, cout).to(DEV)
    scale, shift = torch.rand(cin, device=DEV, generator=gen) + 0.5, torch.randn(cin, device=DEV, generator=gen) * 0.3
    gz, _ = ReLULinearBackward(ApplyBNReLU(x, scale, shift), grad, w)
    _, dscale, _, _ = ApplyBNReLULinearBackward(x, scale, shift, grad, w)
    xl, gl = (t.permute(0, 2, 3, 4, 1).reshape(v, cin) for t in (x, gz))
    ref = (xl.double() * gl.double() * (xl.float() * scale > -shift)).sum(0)
    # chains of at most 8 values, two additions of lanes, the row, the result; 16 results: a factor of 1.5 for their scatter
    parts = (8 + 1) / 2 + 2 + 2
    assert ((dscale.double() - ref).norm() / ref.norm()).item() < 1.5 * 0.42 * 2.0 ** -24 * parts ** 0.5


# (131109 voxels: a second tile for one workgroup at least of every channel pair, a ragged last tile)
@pytest.mark.parametrize('cin,cout', CHANNELS)
@pytest.mark.parametrize('v', [1, 63, 65, 127, 129, 257, 131109])
def test_bnrelu_linear_backward_equals_its_parts(cin, cout, v):
    g = cpu_gen(v * 7 + cin + cout)
    x, grad, w = flat(g, v, cin), flat(g, v, cout), matrix(g, cin, cout).to(DEV)
    scale, shift = torch.randn(cin, generator=g), torch.randn(cin, generator=g) * 0.3
    scale[0], shift[1] = 0.0, 0.0
    xd, gd, sd, bd = x.to(DEV), grad.to(DEV), scale.to(DEV), shift.to(DEV)
    z = ApplyBNReLU(xd, sd, bd)
    gz, dw_ref = ReLULinearBackward(z, gd, w)
    dx_ref, _, _ = ApplyBNReLUBackward(xd, sd, bd, gz)
    dx, dscale, dshift, dw = ApplyBNReLULinearBackward(xd, sd, bd, gd, w)
    assert torch.equal(bits(dx), bits(dx_ref))
    # the same fp32 products in another order of rows, rounded once to fp16: neighbouring values at most
    assert (dw.float() - dw_ref.float()).abs().max().item() <= 2.0 ** -10 * dw_ref.abs().max().item()
    _, ref_scale, ref_shift = oracle.bnrelu_bwd(x, scale, shift, gz.cpu())
    # each result goes through at most 2^9 dependent fp32 additions (a thread's rows, lanes, wavefronts; the rows of the
    # workgroups are added in fp64): 2^9 * 2^-24 of the summed magnitudes
    gzf = gz.float()
    size = gzf.abs().sum((0, 2, 3, 4)).max().item() + (gzf * xd.float()).abs().sum((0, 2, 3, 4)).max().item()
    for got, ref in ((dscale, ref_scale), (dshift, ref_shift)):
        assert got.dtype == torch.float32 and got.shape == (cin,)
        assert (got.cpu().double() - ref).abs().max().item() <= 2.0 ** -15 * size + 1e-30


def same_special(a, b):
    """The same NaNs, infinities of the same sign, and the same values elsewhere (a NaN's own bits are not specified)."""
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and torch.equal(torch.where(nan, 0, a), torch.where(nan, 0, b))


# channel pairs of every split of the weight gradient, two workgroups at least
@pytest.mark.parametrize('cin,cout', [(16, 16), (32, 32), (16, 64), (64, 64), (128, 32), (128, 128)])
@pytest.mark.parametrize('where', ['x', 'scale', 'shift', 'grad'])
def test_bnrelu_linear_backward_of_special_values_equals_its_parts(cin, cout, where):
    v = 700
    g = cpu_gen(cin + cout)
    x, grad, w = flat(g, v, cin), flat(g, v, cout), matrix(g, cin, cout).to(DEV)
    scale, shift = torch.rand(cin, generator=g) + 0.5, torch.randn(cin, generator=g) * 0.3
    scale[5], shift[6] = -0.75, 0.0
    inf, nan = float('inf'), float('nan')
    if where == 'x':  # one per channel, in different workgroups
        for ch, (row, value) in enumerate([(3, inf), (300, -inf), (690, nan), (4, 65504.0), (301, -65504.0), (5, 6e-8), (6, -0.0)]):
            x[0, ch, row] = value
    elif where == 'scale':
        scale[:5] = torch.tensor([inf, -inf, nan, 3e38, 1e-45])
    elif where == 'shift':
        shift[:5] = torch.tensor([inf, -inf, nan, 3e38, -0.0])
    else:
        for ch, (row, value) in enumerate([(3, inf), (300, -inf), (690, nan), (4, 65504.0), (301, 6e-8)]):
            grad[0, ch, row] = value
    xd, gd, sd, bd = x.to(DEV), grad.to(DEV), scale.to(DEV), shift.to(DEV)
    z = ApplyBNReLU(xd, sd, bd)
    gz, dw_ref = ReLULinearBackward(z, gd, w)
    dx_ref, dscale_ref, dshift_ref = ApplyBNReLUBackward(xd, sd, bd, gz)
    dx, dscale, dshift, dw = ApplyBNReLULinearBackward(xd, sd, bd, gd, w)
    assert same_special(dx, dx_ref)
    for got, ref, size in ((dw, dw_ref, None), (dscale, dscale_ref, xd.float() * gz.float()), (dshift, dshift_ref, gz.float())):
        got, ref = got.double(), ref.double()
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        usual = torch.isfinite(ref)
        assert torch.equal(torch.isinf(got), torch.isinf(ref)) and torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
        # dw: neighbouring fp16 values; the sums: fp32 additions of the summed magnitudes, 2^9 in a row at most
        if size is None:
            bound = 2.0 ** -10 * ref.abs() + 2.0 ** -14
        else:
            bound = 2.0 ** -15 * size.double().abs().nan_to_num(0.0, 0.0, 0.0).sum((0, 2, 3, 4)) + 1e-30
        assert ((got - ref).abs() <= bound)[usual].all()


# 2 or 3 workgroups of 128 voxels per compute unit: 65536 or 98304 voxels a round
@pytest.mark.parametrize('cin,cout', CHANNELS)
@pytest.mark.parametrize('v', [1, 31, 33, 127, 129, 65569, 98400])
def test_pointwise_residual_tiles_and_rounds(cin, cout, v):
    g = cpu_gen(v + cin * cout)
    x, add, w = flat(g, v, cin), flat(g, v, cout), matrix(g, cin, cout)
    scale, shift = torch.rand(cin, generator=g) + 0.5, torch.randn(cin, generator=g) * 0.3
    out = ReLULinearAdd(x.to(DEV), w.to(DEV), add.to(DEV)).cpu()
    ref = oracle.pointwise(x, w, add=add, relu_in=True)
    # fp16(product) may be a neighbour of the oracle's, then one more rounding of the sum
    assert (out.float() - ref.float()).abs().max() <= 2.0 ** -9 * max(1.0, ref.abs().max().item())
    fused = ApplyBNReLULinearAdd(x.to(DEV), scale.to(DEV), shift.to(DEV), w.to(DEV), add.to(DEV))
    z = ApplyBNReLU(x.to(DEV), scale.to(DEV), shift.to(DEV))
    assert torch.equal(bits(fused), bits(ReLULinearAdd(z, w.to(DEV), add.to(DEV))))


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16, torch.float32])
def test_quantiser_store_rule(dtype):
    # results up to 96 MiB are stored plainly, larger ones with the streaming hint: the same values on both sides
    limit = 96 << 20
    back = limit // dtype.itemsize
    gen = torch.Generator(DEV).manual_seed(5)
    for n in (limit, limit + 8):
        x = torch.randn(n, device=DEV, generator=gen).to(dtype)
        q = QuantUint8Window(x, 2.5)
        for lo, hi in ((0, 4099), (n - 4099, n)):
            assert torch.equal(q[lo:hi].cpu(), oracle.quant_u8_window(x[lo:hi].cpu(), 2.5))
        half = QuantUint8Window(x[:n // 2].clone(), 2.5)
        assert torch.equal(q[:n // 2], half)
    for n in (back, back + 8):
        part = q[:n].clone()
        out = DequantUint8Window(part, dtype, 2.5)
        assert torch.equal(out[:n // 2], DequantUint8Window(part[:n // 2].clone(), dtype, 2.5))
        assert torch.equal(out[n - 4099:].cpu(), oracle.dequant_u8_window(part[n - 4099:].cpu(), dtype, 2.5))


# few patches (chunks of H without crossing), shares that cross patches, odd extents, one plane, two channel slabs
@pytest.mark.parametrize('shape', [(1, 8, 64, 64, 32), (2, 32, 13, 24, 40), (1, 128, 34, 21, 19), (1, 16, 1, 33, 37),
                                   (3, 64, 47, 17, 9), (1, 64, 96, 9, 9)])
def test_built_in_split_of_the_march(shape):
    n, c, h, w, d = shape
    g = cpu_gen(sum(shape))
    x, grad = rand_cl3d(g, n, c, h, w, d).to(DEV), rand_cl3d(g, n, c, h, w, d).to(DEV)
    _, wk = rand_dw_weight(g, c)
    wd = wk.to(DEV)
    # one workgroup per patch, no chunks: the same output and input gradient bit for bit
    y = DWConv(x, wd)
    assert torch.equal(bits(y), bits(DWConv(x, wd, H_chunk=h)))
    ys, mean, sqmean = DWConvStats(x, wd)
    assert torch.equal(bits(ys), bits(y))
    rmean, rsq = oracle.stats(y.cpu())
    assert torch.allclose(mean.cpu().double(), rmean, rtol=1e-5, atol=1e-6)
    assert torch.allclose(sqmean.cpu().double(), rsq, rtol=1e-5, atol=1e-6)
    dx, gw = DWConvBackward(x, grad, wd, out_dtype=torch.float32)
    assert torch.equal(bits(dx), bits(DWConvBackward(x, grad, wd, H_chunk=h)[0]))
    ref = oracle.dwconv_wgrad(x.cpu(), grad.cpu())
    for got in (gw, DWConvWGRAD(x, grad, out_dtype=torch.float32)):
        # fp32 sums of at most a few thousand products a workgroup, then fp64: the bound of the weight-gradient tests
        assert ((got.cpu().double() - ref).norm() / ref.norm()).item() < 1e-5


# backward: 32769 voxels at 64 channels, 65553 at 32: a second tile for one workgroup of 512; 131109: a second or ragged third
# tile at every channel count, forward and backward
@pytest.mark.parametrize('c', [16, 32, 64])
@pytest.mark.parametrize('v', [1, 31, 33, 63, 65, 32769, 65553, 131109])
def test_inverted_bottleneck_tiles_and_rounds(c, v):
    g = cpu_gen(c + v)
    x, add, grad = flat(g, v, c), flat(g, v, c), flat(g, v, c)
    up, down, bias = matrix(g, c, 2 * c), matrix(g, 2 * c, c), (torch.randn(2 * c, generator=g) * 0.3).half()
    dev = [t.to(DEV) for t in (x, up, down, bias, add, grad)]
    out = LinBReLULinAdd(*dev[:5]).cpu()
    ref = oracle.lin_brelu_lin_add(x, up, down, bias, add)
    # two products and two sums, each rounded to fp16: a hidden value may be a neighbour of the oracle's
    assert (out.float() - ref.float()).abs().max() <= 2.0 ** -8 * max(1.0, ref.abs().max().item())
    got = LinBReLULinBackward(dev[0], dev[5], dev[1], dev[2], dev[3], out_dtype=torch.float32)
    want = oracle.lin_brelu_lin_bwd(x, grad, up, down, bias)
    for a, b in zip(got, want):
        # the ReLU's mask can differ where a pre-activation rounds to the other side of zero (one in about 2^11 within
        # a rounding of it), and a hidden value by one rounding
        err = ((a.cpu().double() - b.double()).norm() / max(b.double().norm().item(), 1e-30)).item()
        assert err < 2.0 ** -5 if v < 1000 else err < 2.0 ** -8, err


def test_inverted_bottleneck_of_a_large_volume_is_that_of_its_parts():
    # 2.6 M voxels of 32 channels, many tiles per workgroup: every voxel's result is its own, so the parts give the same bits
    c, v = 32, (5 << 19) + 33
    gen = torch.Generator(DEV).manual_seed(9)
    x, add = (torch.randn(1, v, 1, 1, c, device=DEV, generator=gen).half().permute(0, 4, 1, 2, 3) for _ in range(2))
    g = cpu_gen(9)
    up, down, bias = (t.to(DEV) for t in (matrix(g, c, 2 * c), matrix(g, 2 * c, c), (torch.randn(2 * c, generator=g) * 0.3).half()))
    out = LinBReLULinAdd(x, up, down, bias, add)
    cut = 1 << 20
    for part in (slice(0, cut), slice(cut, v)):
        assert torch.equal(bits(out[:, :, part]), bits(LinBReLULinAdd(x[:, :, part], up, down, bias, add[:, :, part])))
    tail = slice(v - 5000, v)
    ref = oracle.lin_brelu_lin_add(*(t.cpu() for t in (x[:, :, tail], up, down, bias, add[:, :, tail])))
    assert (out[:, :, tail].cpu().float() - ref.float()).abs().max() <= 2.0 ** -8 * max(1.0, ref.abs().max().item())


# either side of the volumes at which the workgroups per compute unit change: every voxel's result is its own, so one part
# of the volume gives the same bits as the whole
@pytest.mark.parametrize('c, line', [(16, 140000), (16, 500000), (64, 180000)])
def test_inverted_bottleneck_either_side_of_a_volume_line(c, line):
    g = cpu_gen(c)
    x, add = flat(g, line + 1, c), flat(g, line + 1, c)
    up, down, bias = matrix(g, c, 2 * c), matrix(g, 2 * c, c), (torch.randn(2 * c, generator=g) * 0.3).half()
    dev = [t.to(DEV) for t in (x, up, down, bias, add)]
    out = LinBReLULinAdd(*dev)
    below = LinBReLULinAdd(dev[0][:, :, :line - 1], *dev[1:4], dev[4][:, :, :line - 1])
    assert torch.equal(bits(out[:, :, :line - 1]), bits(below))
    tail = slice(line - 2000, line + 1)
    ref = oracle.lin_brelu_lin_add(x[:, :, tail], up, down, bias, add[:, :, tail])
    assert (out[:, :, tail].cpu().float() - ref.float()).abs().max() <= 2.0 ** -8 * max(1.0, ref.abs().max().item())


# either side of the volumes at which the pointwise ops change their number of workgroups, or wait for their stores
@pytest.mark.parametrize('cin,cout,line', [(16, 16, 6000000), (16, 32, 12000000), (16, 64, 3000000), (32, 64, 6000000), (32, 16, 700000), (64, 32, 3000000),
                                           (64, 64, 3000000), (128, 16, 1500000), (128, 32, 700000), (32, 32, 2000000), (32, 128, 700000), (64, 128, 6000000)])
def test_pointwise_ops_either_side_of_a_volume_line(cin, cout, line):
    gen = torch.Generator(DEV).manual_seed(cin + cout)
    x, add = (torch.randn(1, line, 1, 1, c, device=DEV, generator=gen, dtype=torch.float16).permute(0, 4, 1, 2, 3) for c in (cin, cout))
    mix = (torch.randn(cin, cout, device=DEV, generator=gen) / cin ** 0.5).half()
    scale, shift = torch.rand(cin, device=DEV, generator=gen) + 0.5, torch.randn(cin, device=DEV, generator=gen)
    part = slice(0, line - 1)
    low_x, low_add = x[:, :, part], add[:, :, part]
    # every voxel's result is its own
    for whole, below in ((ReLULinearAdd(x, mix, add), ReLULinearAdd(low_x, mix, low_add)),
                         (ApplyBNReLULinearAdd(x, scale, shift, mix, add), ApplyBNReLULinearAdd(low_x, scale, shift, mix, low_add)),
                         (ReLULinearBackward(x, add, mix)[0], ReLULinearBackward(low_x, low_add, mix)[0])):
        assert torch.equal(whole[:, :, part], below)
    tail = slice(line - 2000, line)
    ref = oracle.pointwise(x[:, :, tail].cpu(), mix.cpu(), add=add[:, :, tail].cpu(), relu_in=True)
    got = ReLULinearAdd(x, mix, add)[:, :, tail].cpu()
    assert (got.float() - ref.float()).abs().max() <= 2.0 ** -8 * max(1.0, ref.abs().max().item())


# the pooling backward in output order (8, 16 and, from 24 MiB on, 32 channels): single rows and voxels, runs of a wavefront
# that end inside a row, many rounds of one workgroup, both sides of the 32-channel line
@pytest.mark.parametrize('c,shape', [(8, (1, 1, 1, 1)), (8, (2, 3, 5, 7)), (8, (1, 2, 1, 65)), (8, (1, 9, 8, 64)), (16, (1, 1, 6, 31)),
                                     (16, (3, 4, 5, 33)), (16, (1, 6, 7, 128)), (32, (1, 71, 73, 75)), (32, (1, 71, 73, 76)),
                                     (32, (1, 64, 64, 96)), (32, (1, 64, 64, 95))])
@pytest.mark.parametrize('knobs', [{}, dict(blocks=1, segment=1), dict(blocks=3, segment=2, num_warps=8)])
def test_pool_backward_rows(c, shape, knobs):
    n, h, w, d = shape
    if knobs and n * h * w * d > 100000:
        knobs = dict(knobs, blocks=knobs['blocks'] * 40)
    g = cpu_gen(h * w + d)
    small = (n, c, (h + 1) // 2, (w + 1) // 2, (d + 1) // 2)
    grad, pooled = rand_cl3d(g, *small), rand_cl3d(g, *small)
    mg, sg = torch.randn(c, generator=g), torch.randn(c, generator=g)
    dx = AvgPoolCeilStatsBackward(*(t.to(DEV) for t in (grad, mg, sg, pooled)), (n, c, h, w, d), **knobs)
    # the same operations in the same order
    assert torch.equal(bits(dx.cpu()), bits(oracle.avgpool_ceil_stats_bwd(grad, mg, sg, pooled, (n, c, h, w, d))))


# either side of the sizes at which the built-in launch shapes of the pooling backward and its order change: rows of
# 128 voxels, whose results the kernel in input order redistributes, and of 127
@pytest.mark.parametrize('c,mib', [(c, mib) for c in (8, 16, 32) for mib in (6, 24, 64, 192)] + [(8, 512), (16, 512), (8, 1024), (16, 1024)])
@pytest.mark.parametrize('d', [127, 128])
def test_pool_backward_either_side_of_a_size_line(c, mib, d):
    gen = torch.Generator(DEV).manual_seed(c + mib)
    w = 256
    line = (mib << 20) // (2 * c * w * d)
    for h in (line, line + 1):
        small = (1, -(-h // 2), w // 2, 64)
        grad, pooled = (torch.randn(*small, c, device=DEV, generator=gen, dtype=torch.float16).permute(0, 4, 1, 2, 3) for _ in range(2))
        mg, sg = (torch.randn(c, device=DEV, generator=gen) for _ in range(2))
        args = (grad, mg, sg, pooled, (1, c, h, w, d))
        # every element is the same whatever the shape
        assert torch.equal(AvgPoolCeilStatsBackward(*args), AvgPoolCeilStatsBackward(*args, blocks=2000, num_warps=8, segment=1))
        part = 2 * min(4, h // 2)  # the last rows against the oracle: whole windows, and the rest of an odd height
        lo = h - h % 2 - part
        ref_args = [t[:, :, lo // 2:].cpu() for t in (grad, pooled)]
        count = grad.numel() // c
        # (the oracle takes its mean over the part's windows)
        scale = ref_args[0].numel() // c / count
        ref = oracle.avgpool_ceil_stats_bwd(ref_args[0], mg.cpu() * scale, sg.cpu() * scale, ref_args[1], (1, c, h - lo, w, d))
        got = AvgPoolCeilStatsBackward(*args)[:, :, lo:].cpu()
        # a rounding to fp16, of up to 2^-11, of either
        assert ((got.float() - ref.float()).norm() / ref.float().norm()).item() < 2.0 ** -10


# one voxel to either side of the sizes at which the built-in launch shapes of the stream ops change
@pytest.mark.parametrize('mib', [3, 14, 20, 32, 40, 56, 112, 160, 192, 256, 384, 512, 1280, 1536])
@pytest.mark.parametrize('off', [-1, 1])
def test_stream_ops_either_side_of_a_size_line(mib, off, monkeypatch):
    c = 64
    monkeypatch.setattr(stream_table, '_table', {})  # the library's shapes, at every size
    v = (mib << 20) // (2 * c) + off
    gen = torch.Generator(DEV).manual_seed(mib)
    x, y = (torch.randn(1, v, 1, 1, c, device=DEV, generator=gen).half().permute(0, 4, 1, 2, 3) for _ in range(2))
    scale, shift = torch.rand(c, device=DEV, generator=gen) + 0.5, torch.randn(c, device=DEV, generator=gen)
    one = dict(blocks=64, num_warps=4, segment=1)  # a shape of its own: every element is the same whatever the shape
    peak = torch.full((1,), 5.0, device=DEV)
    q = QuantUint8Window(x, 3.0)
    pooled, pmean, psq = AvgPoolCeilStats(x)
    z, zmean, zsq = AddStats(x, y)
    dx, dscale, dshift = ApplyBNReLUBackward(x, scale, shift, y)
    for got, ref in ((q, QuantUint8Window(x, 3.0, **one)),
                     (DequantUint8Window(q, torch.float16, 3.0), DequantUint8Window(q, torch.float16, 3.0, **one)),
                     (QuantInt8Sym(x, peak)[0], QuantInt8Sym(x, peak, **one)[0]),
                     (ApplyBNReLU(x, scale, shift), ApplyBNReLU(x, scale, shift, **one)),
                     (dx, ApplyBNReLUBackward(x, scale, shift, y, **one)[0]),
                     (z, AddStats(x, y, **one)[0]),
                     (StatsBackward(x, scale, shift), StatsBackward(x, scale, shift, **one)),
                     (AddStatsBackward(x, scale, shift, y), AddStatsBackward(x, scale, shift, y, **one)),
                     (pooled, AvgPoolCeilStats(x, **one)[0]),
                     (AvgPoolCeilStatsBackward(pooled, scale, shift, pooled, tuple(x.shape)),
                      AvgPoolCeilStatsBackward(pooled, scale, shift, pooled, tuple(x.shape), **one))):
        assert torch.equal(got, ref)

    def rows(t):
        return t.permute(0, 2, 3, 4, 1).double().view(-1, c)

    def sums(t):
        return t.mean(0), (t * t).mean(0)

    # the statistics are those of the averages ahead of their rounding to fp16
    averages = torch.cat([rows(x)[:v // 2 * 2].view(-1, 2, c).mean(1), rows(x)[v // 2 * 2:]])
    active = torch.where(dx == 0, 0.0, y.double())  # (scale > 0: the gradient is zero where the ReLU is, or y itself)
    dscale_ref, dshift_ref = ((active * t).sum((0, 2, 3, 4)) for t in (x.double(), 1.0))
    for got, ref in ((Stats(x), sums(rows(x))), ((zmean, zsq), sums(rows(z))), ((pmean, psq), sums(averages)),
                     ((dscale, dshift), (dscale_ref, dshift_ref))):
        # fp32 sums of a workgroup's values (chains of at most a few hundred, error below 2^-24 times their root), fp64
        # from there; means of N(0, 1) values over v voxels are 1 / sqrt(v) in size
        for a, b in zip(got, ref):
            assert ((a.double() - b).norm() / b.norm()).item() < 1e-5


# marches of 3 to 8 plane steps and more: every remainder of the groups of four, one and several segments of a workgroup, at
# both ends of the volume and inside it
@pytest.mark.parametrize('c,w,d', [(8, 9, 67), (16, 9, 33), (32, 17, 17), (64, 9, 9), (128, 9, 9)])
@pytest.mark.parametrize('h_chunk', [1, 2, 3, 4, 5, 6, 7, -2, -6])
def test_depthwise_marches_of_any_length(c, w, d, h_chunk):
    g = cpu_gen(c + h_chunk)
    n, h = 2, 13
    x, grad = rand_cl3d(g, n, c, h, w, d).to(DEV), rand_cl3d(g, n, c, h, w, d).to(DEV)
    wt = rand_dw_weight(g, c)[1].to(DEV)
    # a chunk of the whole height, which the oracle tests pin: an output does not depend on the march that computes it
    assert torch.equal(bits(DWConv(x, wt, H_chunk=h_chunk)), bits(DWConv(x, wt, H_chunk=h)))
    dx, gw = DWConvBackward(x, grad, wt, H_chunk=h_chunk, out_dtype=torch.float32)
    dx_ref, gw_ref = DWConvBackward(x, grad, wt, H_chunk=h, out_dtype=torch.float32)
    assert torch.equal(bits(dx), bits(dx_ref))
    # fp32 sums of a few thousand products in another order
    assert ((gw - gw_ref).norm() / gw_ref.norm()).item() < 1e-5


def channel_sums(*terms):
    """Sums over the voxels in 64 bits, a part of the tensors at a time; terms: (function, tensors ...)."""
    out = []
    for f, *ts in terms:
        parts = zip(*(t.permute(0, 2, 3, 4, 1).reshape(-1, t.shape[1]).split(1 << 18) for t in ts))
        out.append(sum(f(*(p.double() for p in part)).sum(0) for part in parts))
    return out


# Zero-mean values, whose sums are small against their terms: the error of a channel sum against 64 bits, over the size of the
# sums.  Rounding a sum to fp32 is at most 2^-25 to 2^-24 of it, evenly spread: 2^-24 / sqrt(3) = 3.4e-8 in the mean square.
# Sums of fp16 values (mean, dshift) have no other error: the few of a step of the walk are nearly exact.  Products
# (dscale) are rounded as a step adds them, four in a row: sqrt(1 + (1 + 2 + 3 + 4) / 4) times as much, 6.4e-8.  10 % for
# the spread of 64 to 128 channels.
@pytest.mark.parametrize('c,shape', [(64, (1, 86, 86, 88)), (128, (1, 136, 136, 128)), (8, (1, 123, 125, 123)), (64, (1, 236, 236, 228))])
def test_channel_sums_of_the_built_in_shapes_have_no_chains(c, shape):
    gen = torch.Generator(DEV).manual_seed(c)
    n, h, w, d = shape
    x, y = (torch.randn(n, h, w, d, c, device=DEV, generator=gen, dtype=torch.float16).permute(0, 4, 1, 2, 3) for _ in range(2))
    scale, shift = torch.rand(c, device=DEV, generator=gen) + 0.5, torch.randn(c, device=DEV, generator=gen) * 0.1
    one, ten_percent = 2.0 ** -24 / 3 ** 0.5, 1.1

    def check(got, total, bound):
        assert ((got.double() - total).norm() / total.norm()).item() < bound * one * ten_percent

    v = x.numel() // c
    z, mean, _ = AddStats(x, y)
    check(mean, channel_sums((lambda t: t, z))[0] / v, 1.0)
    del z
    dx, dscale, dshift = ApplyBNReLUBackward(x, scale, shift, y)
    on = (dx != 0) | (y == 0)  # (scale > 0: the gradient is zero where the ReLU is, or y itself)
    for got, total, bound in zip((dscale, dshift), channel_sums((lambda t, g, m: t * g * m, x, y, on), (lambda g, m: g * m, y, on)),
                                 ((1 + 10 / 4) ** 0.5, 1.0)):
        check(got, total, bound)
    # (Stats and the pooling have shapes in the table for the largest tensors, whose workgroups hand over fp32 sums)
    if x.numel() * 2 >= stream_table.SMALL_BYTES:
        return
    check(Stats(x)[0], channel_sums((lambda t: t, x))[0] / v, 1.0)
    pmean = AvgPoolCeilStats(x)[1]
    # (all windows of a voxel's sample have 8, 4, 2 or 1 voxels: a voxel counts with one over that number)
    weight = torch.ones(h, w, d, device=DEV, dtype=torch.float64)
    for axis, e in enumerate((h, w, d)):
        edge = torch.full((e,), 0.5, device=DEV, dtype=torch.float64)
        if e % 2:
            edge[-1] = 1.0
        weight *= edge.view([-1 if a == axis else 1 for a in range(3)])
    weight = weight.expand(1, 1, h, w, d)
    windows = n * -(-h // 2) * -(-w // 2) * -(-d // 2)
    check(pmean, channel_sums((lambda t, k: t * k, x, weight))[0] / windows, 1.0)


# the same for the convolution with statistics where half a round of workgroups marches over twice the rows (and, the last, where
# a full round does).  A lane's sums over a march are fp32 here: 20 % for them and the spread
@pytest.mark.parametrize('c,shape', [(16, (1, 58, 58, 60)), (32, (1, 54, 54, 56)), (64, (1, 44, 42, 44)), (128, (1, 34, 34, 36)), (64, (1, 18, 16, 20))])
def test_sums_of_the_convolution_with_statistics(c, shape):
    one, errors = 2.0 ** -24 / 3 ** 0.5, []
    for seed in range(8):
        gen = torch.Generator(DEV).manual_seed(seed)
        x = torch.randn(*shape, c, device=DEV, generator=gen, dtype=torch.float16).permute(0, 4, 1, 2, 3)
        y, mean, sqmean = DWConvStats(x, (torch.randn(3, 3, 3, c, device=DEV, generator=gen) / 27 ** 0.5).half())
        total, squares = (t * c / x.numel() for t in channel_sums((lambda t: t, y), (lambda t: t * t, y)))
        errors.append(((mean.double() - total).norm() / total.norm()).square().item())
        assert ((sqmean.double() - squares).norm() / squares.norm()).item() < 1e-6
    assert (sum(errors) / len(errors)) ** 0.5 < 1.2 * one


def test_channel_sums_that_are_not_finite():
    c, v = 64, 80000  # (9.8 MiB: rows of pairs)
    gen = torch.Generator(DEV).manual_seed(3)
    x = torch.randn(1, v, 1, 1, c, device=DEV, generator=gen).half().permute(0, 4, 1, 2, 3)
    x[0, 1, 5], x[0, 2, 7], x[0, 3, 9], x[0, 3, 11] = float('inf'), float('nan'), float('-inf'), float('-inf')
    inf, nan = float('inf'), float('nan')
    one, zero = torch.ones(c, device=DEV), torch.zeros(c, device=DEV)
    for mean, sqmean in (Stats(x), AddStats(x, torch.zeros_like(x))[1:], AvgPoolCeilStats(x)[1:]):
        assert mean[1] == inf and sqmean[1] == inf and mean[3] == -inf and sqmean[3] == inf
        assert mean[2].isnan() and sqmean[2].isnan()
        assert mean[4:].isfinite().all() and sqmean[4:].isfinite().all() and mean[0].isfinite()
    _, dscale, dshift = ApplyBNReLUBackward(torch.ones_like(x), one, zero, x)
    for got in (dscale, dshift):
        assert torch.equal(got[1:4].nan_to_num(7.0), torch.tensor([inf, nan, -inf], device=DEV).nan_to_num(7.0)) and got[4:].isfinite().all()


# planes of just under 2^31 elements (the largest accepted): the byte offsets of the buffer accesses go up to 2^32 - 16
@pytest.mark.parametrize('c,w,d', [(8, 16383, 16384), (64, 5793, 5792)])
def test_depthwise_planes_up_to_four_gigabytes(c, w, d):
    gen = torch.Generator(DEV).manual_seed(c)
    x = torch.randn(1, 1, w, d, c, device=DEV, generator=gen, dtype=torch.float16).permute(0, 4, 1, 2, 3)
    taps = (torch.randn(3, 3, 3, c, device=DEV, generator=gen) / 27 ** 0.5).half()
    rows = 40
    half = 2 ** 31 // (2 * c * d)  # the row of W with the voxel at byte 2^31
    # an output depends on its neighbours alone: the rows of a narrower plane around the place, without its edge rows
    parts = [(0, rows, 0, rows - 1), (half - rows // 2, half + rows // 2, 1, rows - 1), (w - rows, w, 1, rows)]
    y, _, _ = DWConvStats(x, taps)
    assert torch.equal(y, DWConv(x, taps))
    dx, gw = DWConvBackward(x, x, taps, out_dtype=torch.float32)
    for a, b, first, last in parts:
        sub = x[:, :, :, a:b].contiguous(memory_format=torch.channels_last_3d)
        for whole, part in ((y, DWConv(sub, taps)), (dx, DWConvBackward(sub, sub, taps)[0])):
            assert torch.equal(bits(whole[:, :, :, a + first:a + last]), bits(part[:, :, :, first:last]))
    del y, dx
    # the centre tap's gradient of x with itself is a sum of squares: all of the plane, or a part of it is missing
    flat_x = x.permute(0, 2, 3, 4, 1).reshape(-1, c)
    square = sum(t.double().square().sum(0) for t in flat_x.split(1 << 22))
    assert ((gw[1, 1, 1] - square).abs() <= 1e-4 * square).all()


def test_fused_block_planes_up_to_four_gigabytes():
    w, d = 4095, 4096
    gen = torch.Generator(DEV).manual_seed(1)
    x = torch.randn(1, 1, w, d, 64, device=DEV, generator=gen, dtype=torch.float16).permute(0, 4, 1, 2, 3)
    taps = (torch.randn(3, 3, 3, 64, device=DEV, generator=gen) / 27 ** 0.5).half()
    scale, shift = torch.rand(64, device=DEV, generator=gen) + 0.5, torch.randn(64, device=DEV, generator=gen) * 0.1
    mix = (torch.randn(64, 128, device=DEV, generator=gen) / 8).half()
    y, peak = DWSepBlock(x, taps, scale, shift, mix)
    assert peak.item() == max(t.abs().amax().item() for t in y.permute(0, 2, 3, 4, 1).reshape(-1, 128).split(1 << 22))
    for a, b, first, last in ((0, 40, 0, 39), (2028, 2068, 1, 39), (w - 40, w, 1, 40)):
        part, _ = DWSepBlock(x[:, :, :, a:b].contiguous(memory_format=torch.channels_last_3d), taps, scale, shift, mix)
        assert torch.equal(bits(y[:, :, :, a + first:a + last]), bits(part[:, :, :, first:last]))


def test_pool_backward_rows_up_to_four_gigabytes():
    n, c, h, w, d = 1, 8, 650, 650, 635
    gen = torch.Generator(DEV).manual_seed(2)
    grad, pooled = (torch.randn(n, h // 2, w // 2, (d + 1) // 2, c, device=DEV, generator=gen, dtype=torch.float16) for _ in range(2))
    mg, sg = torch.randn(c, device=DEV, generator=gen) * 1e7, torch.randn(c, device=DEV, generator=gen) * 1e7
    m = torch.tensor(float(pooled.numel() // c), device=DEV)
    dx = AvgPoolCeilStatsBackward(grad.permute(0, 4, 1, 2, 3), mg, sg, pooled.permute(0, 4, 1, 2, 3), (n, c, h, w, d))
    out = dx.permute(0, 2, 3, 4, 1)
    taps = torch.full(((d + 1) // 2,), 8.0, device=DEV)
    taps[-1] = 4.0
    for a in (*range(0, 325, 40), 162, 163, 324):  # (byte 2^31 is in the rows of 162)
        g, o = grad[0, a].float(), pooled[0, a].float()
        ref = ((g + mg / m + 2.0 * o * sg / m) / taps[:, None]).half().repeat_interleave(2, 0).repeat_interleave(2, 1)[:, :d]
        for row in (2 * a, 2 * a + 1):
            assert torch.equal(bits(out[0, row]), bits(ref))
