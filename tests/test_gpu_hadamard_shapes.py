"""HadamardMLP's two forms over the shapes they branch on: factors of 16 and 32
(a wavefront a row, one and two tiles of 16 a factor) and others (a workgroup a
row), widths cut inside a float4, ranks that are no multiple of 8, rows off a
16-byte line, few rows and many; within 1e-5 of the float64 form
(internal/needle/hadamard_test.go:152-191). A row's bits are the same in every
call."""

import numpy as np
import pytest

from go_whistle_amd import needle
from oracle import hadamard_ref as hr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb,rank,dim,rows,offset", [
    (16, 16, 8, 256, 7, 0), (16, 32, 16, 512, 5, 0), (32, 16, 8, 512, 4, 0), (32, 32, 32, 1024, 3, 0), (24, 32, 16, 768, 5, 0),
    (16, 32, 8, 500, 6, 0), (16, 32, 8, 511, 3, 0), (16, 32, 5, 512, 3, 0), (16, 32, 8, 512, 3, 1), (17, 3, 1, 40, 9, 0),
    (1, 1, 1, 1, 2, 0), (64, 16, 8, 1000, 2, 0), (5, 40, 2, 200, 3, 0),
    (17, 3, 1, 40, 2049, 0), (24, 32, 16, 768, 2050, 0), (16, 32, 5, 511, 2049, 0), (16, 32, 8, 512, 2500, 1)])
def test_shapes(na, nb, rank, dim, rows, offset):
    import torch

    g = np.random.default_rng(na * 100 + nb + rank + dim + offset)
    w = hr.random_weights(g, na, nb, rank, dim)
    x = (g.standard_normal((rows, dim)) * 1.5).astype(np.float32)
    z = torch.full((rows * dim + 4,), float("nan"), device="cuda")
    xd = torch.zeros(rows * dim + 4, device="cuda")[offset:offset + rows * dim].copy_(torch.from_numpy(x.ravel()))
    needle.HadamardMLP(w).forward_dev(z[offset:], xd, rows)
    torch.cuda.synchronize()
    got = z.cpu().numpy()
    want = hr.forward(w, x, rows)
    y = got[offset:offset + rows * dim].reshape(rows, dim).astype(np.float64)
    assert np.max(np.abs(y - want)) <= 1e-5 * max(1.0, np.max(np.abs(want)))
    assert np.isnan(got[:offset]).all() and np.isnan(got[offset + rows * dim:]).all()  # nothing past the rows


def test_nan_and_inf_stay_in_their_rows():
    import torch

    g = np.random.default_rng(5)
    w = hr.random_weights(g, 16, 32, 8, 512)
    x = g.standard_normal((4, 512)).astype(np.float32)
    x[1, 3], x[2, 9] = np.nan, np.inf
    out = torch.zeros(4, 512, device="cuda")
    needle.HadamardMLP(w).forward_dev(out, torch.from_numpy(x).cuda(), 4)
    torch.cuda.synchronize()
    y = out.cpu().numpy()
    for r in (0, 3):
        want = hr.forward(w, x[r:r + 1], 1)[0]
        assert np.max(np.abs(y[r] - want)) <= 1e-5 * max(1.0, np.max(np.abs(want)))
    assert np.isnan(y[1]).all() and not np.isfinite(y[2]).any()


@pytest.mark.parametrize("na,nb,rank,dim", [(16, 16, 8, 256), (16, 32, 8, 511), (32, 16, 5, 512), (32, 32, 16, 1024),
                                            (24, 32, 16, 768), (17, 3, 1, 40), (40, 5, 3, 200)])
def test_rows_do_not_depend_on_the_call(na, nb, rank, dim):
    # a row's bits are the same alone, in a long call and off a 16-byte line,
    # and with weights off it
    import torch

    g = np.random.default_rng(na + nb + rank + dim)
    w = hr.random_weights(g, na, nb, rank, dim)
    m = needle.HadamardMLP(w)
    rows, few = 2100, 6
    x = torch.from_numpy(g.standard_normal((rows, dim)).astype(np.float32)).cuda()
    z = lambda n: torch.zeros(n + 4, device="cuda")[1:n + 1]
    many, some, off = torch.zeros(rows, dim, device="cuda"), torch.zeros(few, dim, device="cuda"), z(few * dim)
    m.forward_dev(many, x, rows)
    m.forward_dev(some, x, few)
    m.forward_dev(off, z(few * dim).copy_(x[:few].reshape(-1)), few)
    bits = lambda t: t.reshape(-1)[:few * dim].view(torch.int32)
    assert torch.equal(bits(many), bits(some)) and torch.equal(bits(some), bits(off))
