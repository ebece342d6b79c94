"""Decode attention (attn_decode_split_kernel, attn_combine_kernel) by itself,
through the library's internal entry, against float64: softmax attention of
one query per sequence over its paged keys, times the sigmoid gate
(qwen35.rs:1187-1210).

Bar per element, in units of sum_j p_j |v_j| (gated): a score is a dot product
of 128 terms summed in chains of 8 and four adds, scaled once, so with scores
of scale s its error is at most 13 roundings of sum |q k| / sqrt(128), about
7.2 s: 5.6e-6 s.  It moves e^(score - max) and the sum below it by as much
each; expf, the 32-key chains of P V and the merge add less than 8e-6.  2e-5 s
covers the sum.  At scale 1 the softmax spreads over all keys, so a split left
out or merged without its weight passes the bar 250 times over at every length
here (in float64)."""
import ctypes as C

import numpy as np
import pytest

from ouroboros_amd import _lib
from ouroboros_amd.device import DeviceBuffer

D, PAGE, KEYS, REC = 128, 64, 256, 132  # head width, keys a cache page and a split, floats a split's record


def entry(name, res, args):
    fn = getattr(_lib.lib(), name)
    fn.restype, fn.argtypes = res, args
    return fn


def ws_bytes(B, nh, max_ctx):
    return entry("_ZN4ouro20attn_decode_ws_bytesEmim", C.c_size_t, [C.c_size_t, C.c_int, C.c_size_t])(B, nh, max_ctx)


def test_splits_do_not_depend_on_the_context():
    """256 keys a split for every context length."""
    for ctx in (1, 64, 255, 256, 257, 300, 512, 513, 2048, 16384):
        assert ws_bytes(3, 4, ctx) == 3 * 4 * -(-ctx // KEYS) * REC * 4, ctx


def setup(seed, lens, nh, nkv, scale):
    rng = np.random.default_rng(seed)
    B, maxp = len(lens), -(-max(lens) // PAGE)
    pages = rng.permutation(B * maxp).astype(np.int32).reshape(B, maxp)
    f32 = lambda *s: rng.standard_normal(s).astype(np.float32)
    return dict(lens=np.array(lens, np.int32), pages=pages, q=np.float32(scale) * f32(B, nh, D), gate=f32(B, nh, D),
                kc=f32(B * maxp * PAGE, nkv, D), vc=f32(B * maxp * PAGE, nkv, D))


def run(t, nh, nkv, rows=None):
    """Output [B][nh][D] and the splits' records of the chosen sequences."""
    rows = list(range(len(t["lens"]))) if rows is None else rows
    lens, pages = t["lens"][rows], np.ascontiguousarray(t["pages"][rows])
    B, mx = len(rows), int(lens.max())
    dev = [DeviceBuffer.from_host(np.ascontiguousarray(a)) for a in (t["q"][rows], t["gate"][rows], t["kc"], t["vc"], pages, lens)]
    out = DeviceBuffer((B * nh * D,), np.float32)
    nsplit = -(-mx // KEYS)
    part = DeviceBuffer((ws_bytes(B, nh, mx) // 4,), np.float32)
    fn = entry("_ZN4ouro11attn_decodeEPKfS1_S1_S1_PKiiS3_miPfiiS4_Pv", C.c_int,
               [C.c_void_p] * 5 + [C.c_int, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_void_p])
    assert fn(dev[0].ptr, dev[1].ptr, dev[2].ptr, dev[3].ptr, dev[4].ptr, pages.shape[1], dev[5].ptr, B, mx, out.ptr, nh, nkv,
              part.ptr, None) == 0
    return out.download().reshape(B, nh, D), part.download().reshape(B, nh, nsplit, REC)


LENS = [(1,), (63, 64, 65, 2), (255, 256, 257), (300, 511, 512, 513), (2304, 127, 769, 1, 510)]


@pytest.mark.gpu
@pytest.mark.parametrize("lens", LENS, ids=str)
@pytest.mark.parametrize("nh,nkv", [(4, 1), (2, 2), (16, 2), (6, 2)])
@pytest.mark.parametrize("scale", [1.0, 30.0])  # 30: e^score alone would pass fp32's range
def test_against_float64(gpu, lens, nh, nkv, scale):
    t = setup(len(lens) + nh, lens, nh, nkv, scale)
    got, rec = run(t, nh, nkv)
    bar = 2e-5 * scale
    for b, n in enumerate(lens):
        j = np.arange(n)
        at = t["pages"][b, j // PAGE].astype(np.int64) * PAGE + j % PAGE
        for h in range(nh):
            k, v = (t[c][at, h // (nh // nkv)].astype(np.float64) for c in ("kc", "vc"))
            s = k @ t["q"][b, h].astype(np.float64) / np.sqrt(D)
            for i in range(0, n, KEYS):  # each split by itself
                e = np.exp(s[i:i + KEYS] - s[i:i + KEYS].max())
                r = rec[b, h, i // KEYS].astype(np.float64)
                assert abs(r[D] - s[i:i + KEYS].max()) <= bar
                assert abs(r[D + 1] - e.sum()) <= bar * e.sum()
                assert (np.abs(r[:D] - e @ v[i:i + KEYS]) <= bar * (e @ np.abs(v[i:i + KEYS]))).all()
            p = np.exp(s - s.max())
            p /= p.sum()
            g = 1.0 / (1.0 + np.exp(-t["gate"][b, h].astype(np.float64)))
            assert (np.abs(got[b, h] - g * (p @ v)) <= bar * g * (p @ np.abs(v))).all(), (n, h)


@pytest.mark.gpu
def test_a_sequence_alone_and_in_any_batch(gpu):
    """The same bits alone, in pairs with a longer or shorter one, and in a full batch."""
    lens = (510, 511, 512, 513, 64, 65, 255, 256, 257, 2304, 1)
    t = setup(5, lens, 8, 2, 1.0)
    whole, _ = run(t, 8, 2)
    for b in range(len(lens)):
        for rows in ([b], [b, lens.index(2304)], [b, lens.index(1)]):
            assert np.array_equal(run(t, 8, 2, rows)[0][0], whole[b]), (lens[b], rows)
