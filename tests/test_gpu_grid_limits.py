"""Calls of more work than one launch's grid can hold (HIP refuses 2^32
work-items): their launches are split. Each call repeats a period of rows, and
every period's result is the first one's, bit for bit the oracle's."""

import numpy as np
import pytest

from go_whistle_amd import cq, needle, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu

PERIOD = 1024


def _repeat(base, n):
    """n rows of base, over and over, on the device."""
    import torch

    return torch.from_numpy(base).cuda().repeat(-(-n // len(base)), *[1] * (base.ndim - 1))[:n].contiguous()


def _same(got, base):
    """Every row of got is base's row at its place in the period."""
    import torch

    whole = len(got) // len(base)
    want, bits = torch.from_numpy(np.ascontiguousarray(base)).cuda(), {4: torch.int32, 1: torch.int8}[got.element_size()]
    want, got = want.view(bits), got.view(bits)
    return bool((got[:whole * len(base)].view(whole, *want.shape) == want).all()) and \
        torch.equal(got[whole * len(base):], want[:len(got) - whole * len(base)])


def test_few_rows_product():
    # one matrix row over one group: a wavefront an activation
    import torch

    rows = (1 << 26) + 5
    g = synth.rng(4)
    p = synth.random_packed(g, 1, 4, 128, 4, sigma=0.05)
    x = g.standard_normal((PERIOD, 4)).astype(np.float32)
    y = torch.full((rows, 1), 7.0, device="cuda")
    cq.gemms_dev([cq.New(p)], [y], _repeat(x, rows), rows)
    assert _same(y, orc.OMatrix.new(p).gemm(x.reshape(-1), PERIOD, orc.LUT).reshape(PERIOD, 1))


@pytest.mark.parametrize("width,chunks", [(4, (1 << 28) + 5), (1, (1 << 26) + 5)])  # float4s, 16 lanes a chunk; the rest, 64
def test_quantise_rows_and_fake_quant(width, chunks):
    import torch

    x = (np.random.default_rng(width).standard_normal((PERIOD, width)) ** 3).astype(np.float32)
    q, s = orc.quantize_rows(x.reshape(-1), width, width)
    xd = _repeat(x, chunks)
    qd, sd = torch.full((chunks, width), 99, dtype=torch.int8, device="cuda"), torch.full((chunks,), 9.0, device="cuda")
    needle.quantize_rows_dev(qd, sd, xd, chunks, width, width)
    assert _same(qd, q.reshape(PERIOD, width)) and _same(sd, s)
    del qd, sd
    needle.fake_quant_dev(xd, xd, chunks, width, width)
    want = q.reshape(PERIOD, width).astype(np.float32) * s[:, None]
    assert _same(xd, want.astype(np.float32))


def test_prompt_attention():
    # 17 pairs a stream in workgroups of 16 wavefronts: two a stream, the
    # second nearly empty, 2^32 threads where a wavefront a pair has 2^31
    import torch

    batch, t, qk, vd, nk = 1 << 21, 17, 16, 64, 4
    g = np.random.default_rng(17)
    kq, vq = (g.integers(-128, 128, (nk, w), dtype=np.int8) for w in (qk, vd))
    ks, vs = ((g.random((nk, 1)) * 0.05 + 1e-3).astype(np.float32) for _ in range(2))
    q = g.standard_normal((PERIOD, t * qk)).astype(np.float32)
    spans = np.tile(np.array([[0, 0, 0, nk]], np.int32), (PERIOD * t, 1))
    out = torch.full((batch, t * vd), 7.0, device="cuda")
    dev = lambda a: torch.from_numpy(a).cuda()
    needle.attend_int8_dev(out, _repeat(q, batch), t, 1, dev(kq), dev(ks), qk, qk, dev(vq), dev(vs), vd, vd,
                           _repeat(spans, batch * t), nk, 4.0, True, batch=batch, kv_stride=0, s_stride=0)
    want = orc.attend_int8_spans(q.reshape(-1), PERIOD * t, 1, kq.reshape(-1), ks.reshape(-1), qk, qk, vq.reshape(-1),
                                 vs.reshape(-1), vd, vd, nk, spans, np.float32(4.0), True, 1)
    assert _same(out, want.reshape(PERIOD, t * vd))


def test_rms_unit():
    import torch

    rows = (1 << 26) + 5
    x = np.random.default_rng(8).standard_normal((PERIOD, 1)).astype(np.float32)
    y = torch.full((rows, 1), 9.0, device="cuda")
    needle.rms_unit_dev(y, _repeat(x, rows), rows, 1)
    assert _same(y, orc.rms_unit(x, PERIOD, 1).reshape(PERIOD, 1))
