"""Int8 attention of many streams over the ring of key and value chunks, two
chunks of 32 keys a turn: every length from one key to past four chunks (odd
and even chunk counts, a last chunk of any size, fewer chunks than slots), in
one span and cut in two, with the int8 and the float query. Bit for bit
against the oracle."""

import numpy as np
import pytest

from go_whistle_amd import needle, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", [True, False])
@pytest.mark.parametrize("cut", [False, True])
def test_ring_turns_bit_exact(quant, cut):
    import torch

    g = synth.rng(7 + cut)
    batch, heads, hd, nk = 165, 4, 64, 300
    lengths = [*range(1, 162), 191, 193, 256, nk]
    spans = np.array([[0, n // 3, nk - (n - n // 3), nk] if cut else [0, 0, 0, n] for n in lengths], np.int32)
    kq, vq = (g.integers(-128, 128, size=(batch, nk * heads * hd), dtype=np.int8) for _ in range(2))
    ks, vs = ((g.random((batch, nk * heads)) * 0.05 + 1e-4).astype(np.float32) for _ in range(2))
    q = g.standard_normal((batch, heads * hd)).astype(np.float32)
    out = torch.zeros(batch, heads * hd, device="cuda")
    dev = [torch.from_numpy(a).cuda() for a in (q, kq, ks, vq, vs, spans)]
    needle.attend_int8_dev(out, dev[0], 1, heads, dev[1], dev[2], heads * hd, hd, dev[3], dev[4], heads * hd, hd, dev[5],
                           nk, 8.0, quant, batch=batch, kv_stride=nk * heads * hd, s_stride=nk * heads)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for b in range(batch):
        want = orc.attend_int8_spans(q[b], 1, heads, kq[b], ks[b], heads * hd, hd, vq[b], vs[b], heads * hd, hd, nk,
                                     spans[b:b + 1], np.float32(8.0), quant, 1)
        assert np.array_equal(got[b].view(np.uint32), want.view(np.uint32)), lengths[b]
