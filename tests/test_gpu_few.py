"""Products of few rows (lut_few_kernel), bit for bit the oracle's lut GEMM
(internal/cq/lut.go:158-313): one set of 32 rows and several, one to sixteen
groups, padded inputs, several matrices on one input, views that start
mid-block, NaN and Inf inputs, and the sizes either side of the rule."""

import numpy as np
import pytest

from go_whistle_amd import cq, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, np.float32).reshape(-1), np.asarray(b, np.float32).reshape(-1)
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


def check(ps, views, rows, x):
    import torch

    ms = [cq.New(p) if v is None else cq.New(p).Rows(*v) for p, v in zip(ps, views)]
    os_ = [orc.OMatrix.new(p) if v is None else orc.OMatrix.new(p).rows(*v) for p, v in zip(ps, views)]
    ys = [torch.full((rows, m.Out()), 7.0, device="cuda") for m in ms]
    cq.gemms_dev(ms, ys, torch.from_numpy(x).cuda(), rows)
    torch.cuda.synchronize()
    for y, o in zip(ys, os_):
        assert same(y.cpu().numpy(), o.gemm(x.reshape(-1), rows, orc.LUT))


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("outs,inp,rows", [((4, 4, 16), 2048, 3), ((1,), 2000, 5), ((32,), 512, 700), ((33,), 512, 130),
                                           ((40, 56), 500, 41), ((128,), 512, 1024), ((128,), 512, 1025),
                                           ((512,), 128, 256), ((300, 212), 100, 9), ((64,), 1024, 2), ((24,), 2048, 600)])
def test_few_rows(bits, outs, inp, rows):
    g = synth.rng(sum(outs) + inp + rows + bits)
    ps = [synth.random_packed(g, o, inp, 128, bits, sigma=0.05) for o in outs]
    for p in ps:
        p.Codebook = ps[0].Codebook
    x = (g.standard_normal((rows, inp)) * 2).astype(np.float32)
    x[0, : inp // 2] = 0
    check(ps, [None] * len(ps), rows, x)


@pytest.mark.parametrize("bits", [2, 4])
def test_few_views_and_special_values(bits):
    g = synth.rng(90 + bits)
    p = synth.random_packed(g, 200, 640, 128, bits, sigma=0.05)
    p.Norms = p.Norms.copy()
    p.Norms[:8] = 0  # a zero norm
    x = (g.standard_normal((6, 640)) * 2).astype(np.float32)
    x[1] = 0
    x[2, 5], x[3, 130], x[4, 639] = np.nan, np.inf, -np.inf
    check([p, p, p], [(50, 71), (0, 7), (190, 200)], 6, x)
