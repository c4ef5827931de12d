"""Exact's products of four activations a workgroup (exact_quad_kernel), bit
for bit the oracle's nibble4 and nibble kernels (internal/cq/kernel.go:170-183,
239-374): every group size it takes at both widths, activation counts with
and without a rest of four, blocks that do not fill a workgroup, padded
inputs, several views, and values that are not finite."""

import numpy as np
import pytest

from go_whistle_amd import cq, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, np.float32).reshape(-1), np.asarray(b, np.float32).reshape(-1)
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


@pytest.mark.parametrize("bits,group", [(4, 16), (4, 32), (4, 64), (4, 128), (4, 256), (2, 32), (2, 64), (2, 128), (2, 256)])
@pytest.mark.parametrize("out,inp,rows", [(700, 300, 212), (700, 300, 213), (64, 130, 643), (1050, 256, 130),  # some below its line
                                          (700, 300, 300), (700, 300, 333), (64, 130, 2400), (64, 130, 3603), (1050, 256, 210)])
def test_exact_quads(bits, group, out, inp, rows):
    import torch

    g = synth.rng(out + inp + rows + bits + group)
    p = synth.random_packed(g, out, inp, group, bits)
    m, o = cq.New(p).Exact(), orc.OMatrix.new(p)
    x = (g.standard_normal((rows, inp)) * 2).astype(np.float32)
    y = torch.full((rows, out), 5.0, device="cuda")
    m.gemm_dev(y, torch.from_numpy(x).cuda(), rows)
    torch.cuda.synchronize()
    assert same(y.cpu().numpy(), o.gemm(x.reshape(-1), rows, orc.NIBBLE4))


@pytest.mark.parametrize("bits,group,out,inp,rows", [
    # either side of the work from which the four-activation kernel runs: 4 bits
    # in whole fours and with a rest, 2 bits with a rest, long inputs, blocks
    # that leave wavefronts of a tile idle
    (4, 128, 512, 500, 199), (4, 128, 512, 500, 200), (4, 128, 512, 500, 297), (4, 128, 512, 500, 298),
    (2, 64, 512, 300, 300), (2, 64, 512, 300, 301), (2, 64, 512, 300, 445), (2, 64, 512, 300, 446),
    (4, 32, 70, 1000, 716), (4, 32, 70, 1000, 720), (2, 256, 300, 1600, 284), (2, 256, 300, 1600, 288)])
def test_exact_either_side_of_the_line(bits, group, out, inp, rows):
    test_exact_quads(bits, group, out, inp, rows)


def test_views_and_special_values():
    import torch

    g = synth.rng(31)
    rows = 166
    p = synth.random_packed(g, 1200, 512, 128, 4, sigma=0.05)
    m, o = cq.New(p), orc.OMatrix.new(p)
    views = [(37, 900), (900, 901), (1000, 1200)]
    x = (g.standard_normal((rows, 512)) * 2).astype(np.float32)
    x[1, 5], x[2, 130], x[165, 511], x[7] = np.nan, np.inf, -np.inf, 0
    ms = [m.Rows(*v).Exact() for v in views]
    ys = [torch.full((rows, v[1] - v[0]), 5.0, device="cuda") for v in views]
    cq.gemms_dev(ms, ys, torch.from_numpy(x).cuda(), rows)
    torch.cuda.synchronize()
    for y, v in zip(ys, views):
        assert same(y.cpu().numpy(), o.rows(*v).gemm(x.reshape(-1), rows, orc.NIBBLE4))
