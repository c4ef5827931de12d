"""The 4-bit table form's split of its table entries into three int8
products and a residual (ResidLevels, csrc/cq_internal.hpp): the residual's
bound over codebooks made to be hard for it (on the CPU), and the products
over such codebooks, and over codebooks the split does not take, bit for bit
the oracle's lut GEMM (internal/cq/lut.go:158-313)."""

import numpy as np
import pytest

from go_whistle_amd import cq, synth
from oracle import binding as orc

KINDS = ["normal", "ties127", "ties8", "one", "symmetric"]


def codebook(kind, g):
    """16 levels: ties127 and ties8 put every level of a plane half way
    between two integers (the largest rounding error), one has a single
    level that is not zero."""
    if kind == "ties127":
        c = (g.integers(-127, 127, 16) + 0.5) / 127
    elif kind == "ties8":
        c = (2 * g.integers(-8 * 127, 8 * 127, 16) + 1) / (16 * 127)
    elif kind == "one":
        c = np.zeros(16)
    else:
        c = g.standard_normal(16)
        if kind == "symmetric":
            c[8:] = -c[:8]
    c = np.asarray(c, np.float32) * np.float32(0.05)
    c[0] = np.float32(0.05) if kind != "normal" else c[0]
    return np.sort(c)


@pytest.mark.parametrize("kind", KINDS)
def test_residual_bound(kind):
    # |e| <= 4/2 + 8/2 + 4 + 8/2 + 1/2 < 15 by the levels' and planes'
    # roundings; E2M3 holds the integers to 16
    g = synth.rng(KINDS.index(kind))
    for _ in range(50):
        cb = codebook(kind, g)
        cm = np.abs(cb).max()
        gam = cb.astype(np.float64) / float(cm)
        c1, c2 = np.rint(127 * gam), np.rint(8 * gam)
        c3 = np.rint(8 * (127 * gam - c1))
        x = g.uniform(-1, 1, 2048).astype(np.float32)
        x[:2] = 1, -1
        x[2:500] = (g.integers(-64, 64, 498) + 0.5) * 127 / 8191  # A1's ties
        x = x * (np.float32(8191) / np.float32(cm * np.abs(x).max()))
        v = np.rint(cb[:, None] * x)
        al = x * cm
        a1 = np.rint(al * np.float32(1 / 127))
        a2, a3 = np.rint((al - 127 * a1) * np.float32(0.125)), np.rint(a1 * np.float32(0.125))
        e = v - a1 * c1[:, None] - a2 * c2[:, None] - a3 * c3[:, None]
        assert np.abs(e).max() <= 15 and np.abs(a1).max() <= 65 and max(np.abs(a2).max(), np.abs(a3).max()) <= 8
        assert max(np.abs(c1).max(), np.abs(c2).max(), np.abs(c3).max()) <= 127


def same(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def product(p, rows, x):
    import torch

    m = cq.New(p)
    y = torch.full((rows, p.Out), float("nan"), device="cuda")
    m.gemm_dev(y, torch.from_numpy(x).cuda(), rows)
    torch.cuda.synchronize()
    return m.gemm_path(rows), y.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("out,inp,rows", [(2048, 256, 130), (2080, 200, 1888)])  # a block, and slabs of four
@pytest.mark.parametrize("kind", KINDS)
def test_hard_codebooks(kind, out, inp, rows):
    g = synth.rng(out + KINDS.index(kind))
    p = synth.random_packed(g, out, inp, 128, 4, sigma=0.05)
    p.Codebook = codebook(kind, g)
    x = (g.standard_normal((rows, inp)) * 2).astype(np.float32)
    x[3] = 0
    x[5, :] = 0
    x[5, 7] = 3  # one value: every rotated value at the bound
    path, y = product(p, rows, x)
    assert path == "lut-mfma-tab"
    assert same(y.reshape(-1), orc.OMatrix.new(p).gemm(x.reshape(-1), rows, orc.LUT))


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.0, 2.0 ** -70, 2.0 ** 70])
def test_codebooks_outside_the_split(scale):
    # products of such codebooks run the other forms
    g = synth.rng(77)
    p = synth.random_packed(g, 2048, 256, 128, 4, sigma=0.05)
    p.Codebook = (p.Codebook * np.float32(scale)).astype(np.float32)
    rows = 200
    x = g.standard_normal((rows, 256)).astype(np.float32)
    path, y = product(p, rows, x)
    assert path != "lut-mfma-tab"
    assert same(y.reshape(-1), orc.OMatrix.new(p).gemm(x.reshape(-1), rows, orc.LUT))
