"""RMSUnit rows of any width, and the mHC heads and lane mix over the lane
counts and widths their kernels branch on (2 and 4 lanes by DPP, others by the
generic loop; widths of whole float4s and not, wider than a pass), bit for
bit the oracle (internal/needle/norm.go:68-81, mhc.go:204-299)."""

import numpy as np
import pytest

from go_whistle_amd import needle
from oracle import binding as orc

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, np.float32).ravel(), np.asarray(b, np.float32).ravel()
    return a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32))


def _t(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


@pytest.mark.parametrize("dim", [1, 3, 4, 63, 67, 130, 256, 500, 1000, 2048, 2051, 4095, 4096, 4100])
def test_rms_unit_widths(dim):
    import torch

    rows = 3
    x = (np.random.default_rng(dim).standard_normal((rows, dim)) * 3).astype(np.float32)
    x[1] = 0
    y = torch.full((rows, dim), 9.0, device="cuda")
    needle.rms_unit_dev(y, _t(x), rows, dim)
    torch.cuda.synchronize()
    assert same(y.cpu().numpy(), orc.rms_unit(x, rows, dim))


@pytest.mark.parametrize("dim,rows", [(1, 16), (1, 17), (5, 80), (5, 81), (64, 1024), (64, 1025), (255, 4081), (256, 4096),
                                      (256, 4097), (257, 4200), (512, 9), (1025, 5), (2049, 5)])
def test_rms_unit_row_counts(dim, rows):
    # either side of the rows that a wavefront a row takes, and of the widths
    # at which a thread's values double
    import torch

    x = (np.random.default_rng(dim + rows).standard_normal((rows, dim)) * 3).astype(np.float32)
    y = torch.full((rows, dim), 9.0, device="cuda")
    needle.rms_unit_dev(y, _t(x), rows, dim)
    torch.cuda.synchronize()
    assert same(y.cpu().numpy(), orc.rms_unit(x, rows, dim))


@pytest.mark.parametrize("lanes", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("dim,offset", [(512, 0), (512, 1), (1540, 0), (5, 0), (70, 0), (4, 0)])
def test_heads_and_mix(lanes, dim, offset):
    # offset 1: the stream and outputs start one float past a 16-byte line
    import torch

    rows = 5
    g = np.random.default_rng(100 * lanes + dim + offset)
    f = lambda *s: g.standard_normal(s).astype(np.float32)
    pre, post, res = f(rows, lanes), f(rows, lanes), f(rows, lanes * lanes) * 3
    stream, block_out, aff = f(rows, lanes, dim), f(rows, dim), f(3 + 4 * lanes + lanes * lanes)
    z = lambda n: torch.zeros(n + 4, device="cuda")[offset:offset + n]
    put = lambda a: z(a.size).copy_(_t(a.ravel()))
    hp, hq, hr = (torch.zeros(rows * k, device="cuda") for k in (lanes, lanes, lanes * lanes))
    st, u, out, bo = put(stream), z(rows * dim), z(rows * lanes * dim), put(block_out)
    needle.mhc_heads_dev(hp, hq, hr, u, _t(pre), _t(post), _t(res), st, rows, lanes, dim, _t(aff))
    needle.mhc_mix_dev(out, st, hr, hq, bo, u, rows, lanes, dim)
    torch.cuda.synchronize()
    ohp, ohq, ohr, ou = orc.mhc_heads(pre, post, res, stream, rows, lanes, dim, aff)
    for got, want in ((hp, ohp), (hq, ohq), (hr, ohr), (u, ou), (out, orc.mhc_mix(stream, ohr, ohq, block_out, ou, rows, lanes, dim))):
        assert same(got.cpu().numpy(), want)


@pytest.mark.parametrize("lanes,dim,rows", [(4, 512, 256), (4, 512, 257), (4, 512, 769), (4, 64, 768), (4, 64, 769), (3, 70, 900),
                                            (5, 128, 900), (8, 500, 150), (8, 5, 3000), (3, 1024, 600), (1, 512, 1100)])
def test_mix_output_lanes(lanes, dim, rows):
    # one, two and all output lanes a workgroup, a last one short of its two
    import torch

    g = np.random.default_rng(lanes + dim + rows)
    f = lambda *s: g.standard_normal(s).astype(np.float32)
    stream, hr, hq, block_out, u = f(rows, lanes, dim), f(rows, lanes, lanes), f(rows, lanes), f(rows, dim), f(rows, dim)
    out = torch.full((rows, lanes, dim), 9.0, device="cuda")
    needle.mhc_mix_dev(out, _t(stream), _t(hr), _t(hq), _t(block_out), _t(u), rows, lanes, dim)
    torch.cuda.synchronize()
    assert same(out.cpu().numpy(), orc.mhc_mix(stream, hr, hq, block_out, u, rows, lanes, dim))
