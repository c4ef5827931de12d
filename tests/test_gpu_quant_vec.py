"""QuantizeRows and fakeQuant over the widths and alignments their kernels
branch on (16 lanes a chunk, 64 lanes with 1 to 8 float4s, the generic form
past them and off the alignment), bit for bit the oracle
(internal/needle/int8.go:36-75), special values included."""

import numpy as np
import pytest

from go_whistle_amd import needle
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [4, 12, 48, 64, 68, 256, 260, 512, 516, 1024, 1500, 2048, 2052, 30, 65])
@pytest.mark.parametrize("chunks,offset", [(1, 0), (37, 0), (37, 1)])
def test_quantize_and_fake_quant(width, chunks, offset):
    import torch

    g = np.random.default_rng(width * 10 + chunks + offset)
    x = (g.standard_normal((chunks, width)) ** 3).astype(np.float32)
    if chunks > 4:
        x[1] = 0
        x[2, 0], x[3, width - 1], x[4, width // 2] = np.nan, np.inf, -0.0
    n = x.size
    xd = torch.zeros(n + 4, device="cuda")[offset:offset + n].copy_(torch.from_numpy(x.ravel()))
    q = torch.full((n + 4,), 99, dtype=torch.int8, device="cuda")
    s = torch.full((chunks + 1,), 7.0, device="cuda")
    d = torch.full((n + 4,), 7.0, device="cuda")
    needle.quantize_rows_dev(q[offset:], s, xd, chunks, width, width)
    needle.fake_quant_dev(d[offset:], xd, chunks, width, width)
    needle.fake_quant_dev(xd, xd, chunks, width, width)  # in place
    torch.cuda.synchronize()
    wq, ws = orc.quantize_rows(x.ravel(), width, width)
    wf = orc.fake_quant(x.ravel(), width, width)
    bits = lambda a: np.asarray(a, np.float32).ravel().view(np.uint32)
    assert np.array_equal(q.cpu().numpy()[offset:offset + n], wq.ravel())
    assert (q.cpu().numpy()[:offset] == 99).all() and (q.cpu().numpy()[offset + n:] == 99).all()
    assert np.array_equal(bits(s.cpu().numpy()[:chunks]), bits(ws)) and s[chunks] == 7.0
    for got in (d.cpu().numpy()[offset:offset + n], xd.cpu().numpy()):
        nan = np.isnan(wf.ravel())
        assert np.array_equal(np.isnan(got), nan) and np.array_equal(bits(got[~nan]), bits(wf.ravel()[~nan]))
    assert (d.cpu().numpy()[offset + n:] == 7.0).all()
