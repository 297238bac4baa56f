"""The large-grid attention kernel (attn_fwd_d64) where its 16-bit and fp32 matrix
paths meet: sequence ends inside a key tile and a query block, every mask form, and
operands that the 16-bit forms cannot hold; and the grids around its least size."""
import ctypes as C

import numpy as np
import pytest

from inferc_amd import graphs, lib as L, rt
from inferc_amd.rt import Tensor
from tests import ref64

pytestmark = pytest.mark.gpu
HD = 64


def _run(ctx, q, k, v, mask, fill, off=0):
    """Attention over [B, S, H]; off: element offset of the operands (unaligned rows)."""
    B, S, H = q.shape
    ts = []
    for a in (q, k, v):
        flat = np.zeros(a.size + off, np.float32)
        flat[off:] = a.reshape(-1)
        ts.append(Tensor.from_numpy(ctx, flat))
    out = Tensor.empty(ctx, (B, S, H))
    m = Tensor.from_numpy(ctx, mask.astype(np.uint8)) if mask is not None else None
    ms = (C.c_int64 * 4)(*rt.mask_strides(mask.shape)) if mask is not None else None
    L.check(ctx._lib.inferc_hip_fused_attention_f32(
        ctx.handle, B, S, H, HD, *(t.ptr + 4 * off for t in ts), m.ptr if m else None, ms,
        C.c_float(fill), out.ptr))
    return out.numpy()


def _ref(q, k, v, mask, fill, magnitude=False):
    """In 64 bits; magnitude: sum of the weights times |v| instead."""
    B, S, H = q.shape
    n = H // HD
    hd = lambda a: a.astype(np.float64).reshape(B, S, n, HD).transpose(0, 2, 1, 3)  # noqa: E731
    s = hd(q) @ hd(k).transpose(0, 1, 3, 2) / 8.0
    if mask is not None:
        s = np.where(np.broadcast_to(mask, s.shape), np.float64(np.float32(fill)), s)
    p = np.exp(s - s.max(-1, keepdims=True))
    o = (p / p.sum(-1, keepdims=True)) @ (np.abs(hd(v)) if magnitude else hd(v))
    return o.transpose(0, 2, 1, 3).reshape(B, S, H)


def _inputs(B, S, heads, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    return [(scale * rng.standard_normal((B, S, heads * HD))).astype(np.float32)
            for _ in range(3)]


def _close(got, ref, v):
    # a weight is off by the score's absolute error (64 products of N(0, 1) / 8 round at 2^-24
    # of their sum, at most 30 here) and two roundings; S weights average V
    assert np.isfinite(got).all()
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(v).max()


@pytest.mark.parametrize("S,B", [(1, 300), (31, 260), (40, 127), (64, 128), (33, 260), (128, 24), (129, 132), (160, 150),
                                 (255, 130), (300, 90)])
@pytest.mark.parametrize("form", ["none", "row", "full"])
def test_attention_tiles_masks_and_edges(ctx, S, B, form):
    heads = 1
    q, k, v = _inputs(B, S, heads, S + B)
    rng = np.random.default_rng(B)
    mask = None
    if form == "row":
        lens = rng.integers(1, S + 1, B)
        mask = (np.arange(S)[None, :] >= lens[:, None]).reshape(B, 1, 1, S)
        mask[1] = True  # every key masked
        mask[2, ..., 0] = True  # an early key masked
    elif form == "full":
        mask = rng.random((B, 1, S, S)) < 0.4
    for off in (0, 1):
        _close(_run(ctx, q, k, v, mask, graphs.FILL_MIN, off),
               _ref(q, k, v, mask, graphs.FILL_MIN), v)


# the large-grid kernel starts at 256 blocks of 128 queries (one a CU), at 128 for four key
# tiles and more: the last grid of the small-grid kernels and the first of it
@pytest.mark.parametrize("S,B", [(96, 255), (96, 256), (97, 127), (97, 128), (97, 255), (200, 63),
                                 (200, 64), (200, 127), (300, 42), (300, 43)])
@pytest.mark.parametrize("form", ["none", "row"])
def test_attention_grids_around_the_least_size(ctx, S, B, form):
    q, k, v = _inputs(B, S, 1, S * B)
    mask = None
    if form == "row":
        lens = np.random.default_rng(B).integers(1, S + 1, B)
        mask = (np.arange(S)[None, :] >= lens[:, None]).reshape(B, 1, 1, S)
    _close(_run(ctx, q, k, v, mask, graphs.FILL_MIN), _ref(q, k, v, mask, graphs.FILL_MIN), v)


@pytest.mark.parametrize("n", [896, 897, 1000, 1024, 1051])
def test_attention_tiles_causal_prefill(ctx, n):
    """A causal prefill of 16 heads: 112 blocks (small-grid kernel) at 896 tokens, 128 and
    more (the large-grid kernel's causal rule, tile skip and score masks) from 897. The
    queries and keys are large, so that a key more or less moves the logits by 1e-2."""
    cfg = dict(layers=1, hidden=1024, heads=16, ffn=128, vocab=200, max_pos=1051, eps=1e-5)
    w = graphs.gpt2_weights(cfg, 11)
    w[4] = (w[4] * np.float32(4)).astype(np.float32)  # QKV
    w[6] = (w[6] * np.float32(4)).astype(np.float32)  # out-projection
    ids = np.random.default_rng(n).integers(0, cfg["vocab"], n)
    dec = rt.Gpt2Decoder(ctx, cfg, w, max_t=cfg["max_pos"])
    got = dec.forward(ids)
    dec.close()
    ref = ref64.gpt2_logits(cfg, w, ids)
    assert np.abs(got - ref).max() <= 1e-4, float(np.abs(got - ref).max())


@pytest.mark.parametrize("S,B,heads", [(100, 26, 12), (200, 13, 12)])
@pytest.mark.parametrize("kind", ["tiny_v", "subnormal_v", "tiny_qk", "zero_v", "sharp",
                                  "late_max", "huge_v", "huge_masked", "soft_fill", "large_qk",
                                  "masked_large_v", "small_late_v", "mixed_v", "one_key"])
def test_attention_tiles_operand_ranges(ctx, S, B, heads, kind):
    q, k, v = _inputs(B, S, heads, len(kind))
    lens = np.random.default_rng(3).integers(max(1, S // 4), S + 1, B)
    lens[0] = S // 2
    mask = (np.arange(S)[None, :] >= lens[:, None]).reshape(B, 1, 1, S)
    fill = graphs.FILL_MIN
    if kind == "tiny_v":
        v *= np.float32(1e-9)
    elif kind == "subnormal_v":
        v *= np.float32(1e-39)
    elif kind == "tiny_qk":
        q *= np.float32(1e-5)
        k *= np.float32(1e-5)
    elif kind == "zero_v":
        v[:, :, 5] = 0.0
    elif kind == "sharp":
        q *= np.float32(3)
    elif kind == "late_max":  # scores rise along the keys: the running maximum moves
        k *= (0.2 + 2.0 * np.arange(S) / S).astype(np.float32)[None, :, None]
    elif kind == "huge_v":
        v[0, 0, 0] = 1e6
    elif kind == "huge_masked":  # beyond fp16 where every key is masked away
        assert mask[0, 0, 0, -1]
        v[0, -1] = 3e5
        k[0, -1] = -1e7
    elif kind == "soft_fill":  # masked keys keep a weight
        fill = -2.5
        mask = np.random.default_rng(4).random((B, 1, S, S)) < 0.4
    elif kind == "large_qk":  # small elements of q meet large ones of k
        q *= np.float32(1e-6)
        k *= np.float32(1e5)
    elif kind == "masked_large_v":  # the first keys are masked and large, the rest small
        mask[..., :40] = True
        lens = np.maximum(lens, 60)
        mask[..., 40:] = np.arange(40, S)[None, :] >= lens[:, None, None, None]
        v[:, 40:] *= np.float32(1e-12)
    elif kind == "small_late_v":  # the same, the first keys unmasked but without weight
        k[..., :40, :] = -50.0 * np.sign(q[:, :1])
        q[:] = np.abs(q) * np.sign(q[:, :1])
        k[:, 40:] *= np.float32(0.1)
        v[:, 40:] *= np.float32(1e-12)
    elif kind == "mixed_v":  # every dim spans many decades
        v *= np.float32(10.0) ** np.random.default_rng(6).uniform(-30, 10, v.shape).astype(np.float32)
    elif kind == "one_key":  # each query all but selects one key
        k[:] = 0.0
        for d in range(HD):
            k[:, d::HD, d::HD] = 60.0
        q[:] = 0.0
        pick = np.random.default_rng(7).integers(0, HD, (B, S, heads))
        np.put_along_axis(q.reshape(B, S, heads, HD), pick[..., None], np.float32(8.0), -1)
        v *= np.float32(10.0) ** np.random.default_rng(8).uniform(-20, 0, v.shape).astype(np.float32)
    got, ref = _run(ctx, q, k, v, mask, fill), _ref(q, k, v, mask, fill)
    assert np.isfinite(got).all()
    # Every output against its own terms, sum p |v|: the scores' rounding (64 products at
    # 2^-24 of their sum of magnitudes) is a relative error of the weights, as are the
    # rounding of S weights' sums; half a subnormal step where the terms are that small.
    d = lambda a: a.astype(np.float64).reshape(B, S, heads, HD).transpose(0, 2, 1, 3)  # noqa: E731
    scores = (np.abs(d(q)) @ np.abs(d(k)).transpose(0, 1, 3, 2)).max() / 8.0
    lim = 2.0 ** -23 * scores + S * 2.0 ** -24
    mag = _ref(q, k, v, mask, fill, magnitude=True)
    assert (np.abs(got - ref) <= lim * mag + 2.0 ** -149).all(), \
        float((np.abs(got - ref) / (mag + 1e-300)).max() / lim)


@pytest.mark.parametrize("S,B", [(120, 260), (180, 140)])
def test_attention_tiles_infinities_and_nan(ctx, S, B):
    q, k, v = _inputs(B, S, 1, 4)
    v[0, 3, 2], v[1, 5, 7], k[2, 4, 0], q[3, 9, 1] = np.inf, np.nan, np.nan, np.nan
    got = _run(ctx, q, k, v, None, graphs.FILL_MIN)
    assert np.isposinf(got[0, :, 2]).all() and np.isnan(got[1, :, 7]).all()
    assert np.isnan(got[2]).all() and np.isnan(got[3, 9]).all()
    clean = np.isfinite(got)
    clean[2] = False
    ref = _ref(q[4:], k[4:], v[4:], None, 0.0)
    _close(got[4:], ref, v[4:])
    assert clean[0].sum() == S * 63 and clean[1].sum() == S * 63 and clean[3].sum() == (S - 1) * 64
