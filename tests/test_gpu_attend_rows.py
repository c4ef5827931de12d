"""Int8 attention of prompts (t > 1, more (row, head) pairs than stay
resident): several pairs a workgroup over keys and values staged once.
Bit for bit against the oracle at the edges of what the kernel splits by:
the pairs of a workgroup (4 to 16, with a last one that is not full, and fewer
where the LDS ends), the 32-key blocks and the four keys of a weight read, two spans in any order and
at any distance, empty spans and spans off the cache, RoPE of the query,
shared and paged caches, infinite scales; few keys, and key counts past its
LDS, go to the other kernels."""

import numpy as np
import pytest

import go_whistle_amd.decoder as dec
from go_whistle_amd import cq, synth
from go_whistle_amd._lib import check, lib
from oracle import binding as orc

pytestmark = pytest.mark.gpu


def _p(t):
    from ctypes import c_void_p

    return c_void_p(t.data_ptr())


def _spans(kind, g, batch, t, nk):
    sp = np.zeros((batch, t, 4), np.int32)
    for b in range(batch):
        for i in range(t):
            if kind == "causal":
                sp[b, i] = [0, 0, 0, max(0, nk - t + i + 1 - b)]
            else:  # two disjoint spans, either first; some empty, some off the cache
                c = np.sort(g.integers(0, nk + 1, size=4))
                sp[b, i] = [*c[:2], *c[2:]] if i % 2 else [*c[2:], *c[:2]]
                if i % 7 == 3:
                    sp[b, i] = [0, 0, 0, 0]
                if i % 7 == 5:
                    sp[b, i] = [0, 0, 3, nk + 1]
                if i % 7 == 6:
                    sp[b, i] = [c[0], c[0], c[1], c[2]]
    return sp


@pytest.mark.parametrize("batch,t,heads,kv_heads,qk,nk,quant,kind,form", [
    (4, 96, 8, 2, 48, 448, True, "causal", "plain"),
    (3, 37, 8, 2, 64, 130, True, "two", "plain"),
    (3, 37, 8, 8, 64, 131, False, "two", "plain"),
    (5, 27, 4, 1, 16, 33, True, "two", "rope"),
    (7, 19, 4, 4, 32, 64, True, "two", "shared"),
    (4, 33, 6, 3, 48, 97, False, "two", "paged"),
    (40, 2, 8, 2, 64, 100, True, "two", "paged"),
    (2, 200, 8, 4, 64, 3, True, "causal", "plain"),
    (130, 4, 8, 8, 64, 448, True, "causal", "plain"),   # four pairs a workgroup, too many of them
    (2, 80, 8, 2, 64, 900, True, "causal", "plain"),    # past the LDS
    (3, 40, 8, 2, 64, 70, True, "two", "inf"),
    # 16 wavefronts a workgroup, whole and with a last one of 4; cut to 14 by the
    # LDS, without and with a page table in it
    (4, 128, 8, 2, 48, 448, True, "two", "plain"),
    (13, 85, 4, 1, 64, 200, True, "two", "plain"),
    (16, 32, 8, 2, 64, 560, True, "two", "plain"),
    (16, 33, 8, 2, 64, 560, False, "two", "paged"),
    # few keys and pairs enough for the kernel, and either side of the fewest keys
    # it takes below that
    (128, 4, 8, 1, 48, 3, True, "two", "plain"),
    (256, 4, 8, 8, 64, 20, True, "two", "plain"),
    (5, 27, 4, 1, 16, 65, True, "two", "rope"),
    (5, 27, 4, 1, 16, 64, True, "two", "rope"),
    (7, 19, 4, 4, 32, 70, True, "two", "shared"),
    (3, 40, 8, 2, 64, 81, True, "two", "inf"),
])
def test_prompt_rows_bit_exact(batch, t, heads, kv_heads, qk, nk, quant, kind, form):
    import torch

    g = synth.rng(batch * 1000 + t)
    vd = 64
    caches = 3 if form == "shared" else batch
    rows = nk if form != "paged" else (nk + 15) // 16 * 16
    width = kv_heads * max(qk, vd)
    kq = g.integers(-128, 128, size=(caches, rows * width), dtype=np.int8)
    vq = g.integers(-128, 128, size=(caches, rows * width), dtype=np.int8)
    ks = (g.random((caches, rows * kv_heads)) * 0.05 + 1e-4).astype(np.float32)
    vs = (g.random((caches, rows * kv_heads)) * 0.05 + 1e-4).astype(np.float32)
    if form == "inf":
        vs[:, 5 * kv_heads] = np.inf
    q = g.standard_normal((batch, t, heads, qk)).astype(np.float32)
    spans = _spans(kind, g, batch, t, nk)
    scale = np.float32(np.sqrt(qk))
    idx = np.arange(batch, dtype=np.int32) % (caches + 1) if form == "shared" else np.arange(batch, dtype=np.int32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    out = torch.full((batch, t, heads, vd), 5.0, device="cuda")
    qd, kd, vd_, ksd, vsd, spd, idd = (dev(a) for a in (q, kq, vq, ks, vs, spans, idx))
    stream = cq._stream()
    tail = [_p(spd), nk, float(scale), int(quant), batch]
    head = [_p(out), 0, _p(qd), 0, t, heads]
    k_cols, v_cols = kv_heads * qk, kv_heads * vd
    cos = sin = qpos = None
    if form == "rope":
        cos, sin = dec.rope_tables(qk, nk + t, 1e4)
        qpos = g.integers(0, nk + t, size=batch * t).astype(np.int32)
        cd, sd, pd = dev(cos), dev(sin), dev(qpos)
    if form == "paged":
        np_ = rows // 16
        pages = g.permutation(batch * np_).astype(np.int32).reshape(batch, np_)
        # the pool: page pages[b, i] holds rows 16 i .. 16 i + 15 of stream b
        pool = [np.zeros((batch * np_ * 16, c), a.dtype) for a, c in ((kq, k_cols), (vq, v_cols), (ks, kv_heads), (vs, kv_heads))]
        for b in range(batch):
            for i in range(np_):
                for dst, src, c in zip(pool, (kq, vq, ks, vs), (k_cols, v_cols, kv_heads, kv_heads)):
                    dst[pages[b, i] * 16:pages[b, i] * 16 + 16] = src[b, i * 16 * c:(i + 1) * 16 * c].reshape(16, c)
        pk, pv, pks, pvs, pg = (dev(a) for a in (*pool, pages))
        check(lib().kv_attend_int8_paged_dev(*head, _p(pk), _p(pks), k_cols, qk, _p(pv), _p(pvs), v_cols, vd, *tail,
                                             None, None, None, _p(pg), np_, 16, batch * np_, stream))
    else:
        mid = [_p(kd), _p(ksd), k_cols, qk, _p(vd_), _p(vsd), v_cols, vd, rows * width, rows * kv_heads]
        if form == "rope":
            check(lib().kv_attend_int8_rope_dev(*head, *mid, *tail, _p(cd), _p(sd), _p(pd), stream))
        elif form == "shared":
            check(lib().kv_attend_int8_shared_dev(*head, *mid, *tail, _p(idd), caches, stream))
        else:
            check(lib().kv_attend_int8_dev(*head, *mid, *tail, stream))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for b in sorted(set([0, 1, batch // 2, batch - 1])):
        c = int(idx[b])
        if c >= caches:
            assert np.all(got[b] == 5.0)
            continue
        qb = q[b].reshape(-1)
        if form == "rope":
            qb = orc.rope(qb.copy(), heads, qk, cos, sin, qpos[b * t:(b + 1) * t])
        good = [i for i in range(t) if spans[b, i, 3] <= nk]
        qg = qb.reshape(t, heads * qk)[good].reshape(-1)
        want = orc.attend_int8_spans(qg, len(good), heads, kq[c][:rows * k_cols], ks[c], k_cols, qk, vq[c][:rows * v_cols],
                                     vs[c], v_cols, vd, nk, spans[b][good], scale, quant, 1)
        want = want.reshape(len(good), heads, vd)
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got[b][good]), nan)
        assert np.array_equal(got[b][good].view(np.uint32)[~nan], want.view(np.uint32)[~nan]), b
        for i in set(range(t)) - set(good):
            assert np.all(got[b, i] == 5.0)
