"""Int8 attention of spans that overlap: two spans of more keys together than
the cache has leave their output untouched in every kernel (its logits have no
more places), and the rows beside them are bit for bit the oracle's."""

import numpy as np
import pytest

from go_whistle_amd import needle, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,t,qk,vd", [
    (4, 1, 64, 64),     # all value rows resident
    (160, 1, 64, 64),   # the ring
    (160, 1, 48, 64),   # one wavefront's chain
    (160, 1, 64, 128),  # 128-code value heads
    (160, 1, 64, 96),   # any head width
    (8, 90, 48, 64),    # prompts over keys staged once
])
def test_overlapping_spans(batch, t, qk, vd):
    import torch

    g = synth.rng(batch + qk + vd)
    heads, nk = 4, 200
    kc, vc = heads * qk, heads * vd
    cols = max(kc, vc)
    kq, vq = (g.integers(-128, 128, size=(batch, nk * cols), dtype=np.int8) for _ in range(2))
    ks, vs = ((g.random((batch, nk * heads)) * 0.05 + 1e-4).astype(np.float32) for _ in range(2))
    q = g.standard_normal((batch, t, heads * qk)).astype(np.float32)
    spans = np.zeros((batch, t, 4), np.int32)
    flat = spans.reshape(-1, 4)
    flat[:] = [3, 90, 100, nk]
    bad = np.arange(len(flat)) % 3 == 1
    flat[bad] = [0, nk, 1, nk]
    flat[::7] = [10, 60, 40, 120]  # overlapping, within the places
    bad[::7] = False
    out = torch.full((batch, t, heads * vd), 7.0, device="cuda")
    dev = [torch.from_numpy(a).cuda() for a in (q, kq, ks, vq, vs, spans)]
    needle.attend_int8_dev(out, dev[0], t, heads, dev[1], dev[2], kc, qk, dev[3], dev[4], vc, vd, dev[5], nk, 8.0, True,
                           batch=batch, kv_stride=nk * cols, s_stride=nk * heads)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(got.reshape(len(flat), -1)[bad] == 7.0)
    for b in sorted({0, 1, batch // 2, batch - 1}):
        good = ~bad.reshape(batch, t)[b]
        want = orc.attend_int8_spans(q[b][good].reshape(-1), int(good.sum()), heads, kq[b][:nk * kc], ks[b], kc, qk,
                                     vq[b][:nk * vc], vs[b], vc, vd, nk, spans[b][good], np.float32(8.0), True, 1)
        assert np.array_equal(got[b][good].reshape(-1).view(np.uint32), want.reshape(-1).view(np.uint32)), b
