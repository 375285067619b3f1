"""The f32 matrix-core attention kernels (head widths 64 / 128 / 256) at the
edges of their tiles: 16-key tiles, 4- and 8-row decode sets, 32- and 64-row
tiles, key splits. Reference: float64 on the same values; and the scalar
kernels they stand in for (RXW8_FORCE_GENERIC=1) for values that are not
ordinary numbers. Tolerance: f32 sums over at most 256 dims and 300 keys of
N(0, 1) values err by a few 2^-24 sqrt(terms), far below 1e-5 of the largest
output (observed 1e-6)."""
import numpy as np
import pytest

import oracle
from conftest import rel_err

pytestmark = pytest.mark.gpu


def rx():
    import rxla_amd
    return rxla_amd


def softmax_rows(q, k, v, scale, mask, vis):
    """float64: q [H, S, D], k / v [Hkv, K, D], mask [H, S, K] or None, vis [S]."""
    out = np.zeros(q.shape[:2] + v.shape[-1:])
    for h in range(q.shape[0]):
        kv = h // (q.shape[0] // k.shape[0])
        for i in range(q.shape[1]):
            n = vis[i]
            s = k[kv, :n].astype(np.float64) @ q[h, i].astype(np.float64) * scale
            if mask is not None:
                s = s + mask[h, i, :n]
            p = np.exp(s - s.max())
            out[h, i] = p @ v[kv, :n].astype(np.float64) / p.sum()
    return out


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv,sq,sk", [(2, 2, 1, 1), (8, 2, 1, 17), (8, 1, 1, 300), (4, 2, 4, 16),
                                          (3, 1, 3, 31), (6, 2, 11, 129), (4, 4, 65, 65),
                                          (5, 1, 13, 64), (8, 2, 40, 250)])
@pytest.mark.parametrize("splits", [0, 3])
def test_masked_attention_tiles(rt, monkeypatch, d, hq, hkv, sq, sk, splits):
    if splits:
        monkeypatch.setenv("RXW8_ATTN_F32_SPLITS", str(splits))
    rng = np.random.default_rng(d + hq * sk)
    q = rng.standard_normal((2, hq, sq, d)).astype(np.float32)
    k = rng.standard_normal((2, hkv, sk, d)).astype(np.float32)
    v = rng.standard_normal((2, hkv, sk, d)).astype(np.float32)
    mask = np.where(rng.random((2, 1, sq, sk)) < 0.3, -np.inf, rng.standard_normal((2, 1, sq, sk)))
    mask[..., 0] = 0.0
    mask = mask.astype(np.float32)
    low = np.finfo(np.float32).min
    mask[0, 0, sq // 2, :] = low  # every key at the type's lowest value: equal weights
    r = rx()
    for rg in ("4", "2"):
        monkeypatch.setenv("RXW8_ATTN_F32_RG", rg)
        got = r.gqa_attention(rt, rt.buffer(q), rt.buffer(k), rt.buffer(v), rt.buffer(mask)).to_numpy()
        plain = r.gqa_attention(rt, rt.buffer(q), rt.buffer(k), rt.buffer(v), None, 0.25).to_numpy()
        for b in range(2):
            m = np.broadcast_to(mask[b], (hq, sq, sk)).astype(np.float32)
            s32 = np.float32(1.0) / np.sqrt(np.float32(d))
            want = softmax_rows(q[b], k[b], v[b], s32, m, [sk] * sq)
            if b == 0:  # f32 scores absorb into the lowest value
                want[:, sq // 2] = np.repeat(v[0].astype(np.float64).mean(axis=1), hq // hkv, axis=0)
            assert rel_err(got[b], want) <= 1e-5
            assert rel_err(plain[b], softmax_rows(q[b], k[b], v[b], 0.25, None, [sk] * sq)) <= 1e-5


@pytest.mark.parametrize("d,cache", [(64, "bf16"), (128, "f32"), (256, "bf16"), (256, "f32"), (64, "f32")])
@pytest.mark.parametrize("hq,hkv", [(3, 3), (8, 2), (8, 1), (12, 1)])
@pytest.mark.parametrize("splits", [0, 1, 5])
def test_decode_lengths(rt, monkeypatch, d, cache, hq, hkv, splits):
    """Lengths around the tile, clamped ones, garbage past them, a mask."""
    if splits:
        monkeypatch.setenv("RXW8_ATTN_F32_SPLITS", str(splits))
    r = rx()
    rng = np.random.default_rng(d + hq)
    lmax, lens = 273, np.array([1, 16, 17, 0, 128, 400], np.int32)
    b = len(lens)
    q = rng.standard_normal((b, hq, d)).astype(np.float32)
    k = oracle.round_bf16(rng.standard_normal((b, hkv, lmax, d)).astype(np.float32))
    v = oracle.round_bf16(rng.standard_normal((b, hkv, lmax, d)).astype(np.float32))
    vis = np.clip(lens, 1, lmax)
    for i in range(b):
        k[i, :, vis[i]:] = np.nan
        v[i, :, vis[i]:] = np.inf
    mask = rng.standard_normal((b, hq, lmax)).astype(np.float32)
    bits = (lambda x: rt.buffer(oracle.bf16_bits(x), r.DType.BF16)) if cache == "bf16" else rt.buffer
    bufs = (rt.buffer(q), bits(k), bits(v), rt.buffer(lens))
    for m in (None, mask):
        mb = None if m is None else rt.buffer(m)
        got = r.grouped_query_attention(rt, *bufs, mask=mb).to_numpy()
        out = rt.zeros(q.shape, r.DType.F32)
        r.grouped_query_attention_noalloc(rt, *bufs, out, mask=mb)
        np.testing.assert_array_equal(out.to_numpy(), got)
        scale = np.float32(1.0) / np.sqrt(np.float32(d))
        for i in range(b):
            want = softmax_rows(q[i][:, None], k[i], v[i], scale, None if m is None else m[i][:, None], [vis[i]])
            assert rel_err(got[i], want[:, 0]) <= 1e-5


@pytest.mark.parametrize("d,hq,hkv", [(64, 4, 2), (256, 4, 1), (128, 6, 2), (256, 2, 2)])
@pytest.mark.parametrize("s", [2, 33, 70])
def test_prefill_ignores_what_a_row_cannot_see(rt, d, hq, hkv, s):
    """Rows at the ends of tiles, caches whose later rows are NaN: a row's
    result is that of its own keys alone."""
    r = rx()
    rng = np.random.default_rng(d + s)
    starts, lmax = np.array([0, 45], np.int32), 45 + s
    q = rng.standard_normal((2, s, hq, d)).astype(np.float32)
    k = oracle.round_bf16(rng.standard_normal((2, hkv, lmax, d)).astype(np.float32))
    v = oracle.round_bf16(rng.standard_normal((2, hkv, lmax, d)).astype(np.float32))
    k[0, :, s:], v[0, :, s:] = np.nan, np.nan
    bits = lambda x: rt.buffer(oracle.bf16_bits(x), r.DType.BF16)  # noqa: E731
    clean = r.grouped_query_attention_prefill(rt, rt.buffer(q), bits(k), bits(v), rt.buffer(starts)).to_numpy()
    scale = np.float32(1.0) / np.sqrt(np.float32(d))
    for b in range(2):
        want = softmax_rows(q[b].transpose(1, 0, 2), k[b], v[b], scale, None,
                            [starts[b] + i + 1 for i in range(s)])
        assert rel_err(clean[b].transpose(1, 0, 2), want) <= 1e-5
    # a key that only the last rows see may be anything: the earlier rows stand
    last = s - 1
    v[0, :, last], v[1, :, 45 + last] = np.nan, np.inf
    dirty = r.grouped_query_attention_prefill(rt, rt.buffer(q), bits(k), bits(v), rt.buffer(starts)).to_numpy()
    assert np.max(np.abs(dirty[:, :last] - clean[:, :last])) <= 1e-5
    assert not np.isfinite(dirty[:, last]).any()


@pytest.mark.parametrize("sq,hq", [(1, 2), (7, 4), (40, 4)])
def test_not_a_number_and_infinities_as_the_scalar_kernel(rt, monkeypatch, sq, hq):
    """Masked keys that hold NaN or infinities, infinite scores, rows without
    a key: where the scalar kernel gives numbers so do these, and the rest is
    the same kind of non-number."""
    r = rx()
    rng = np.random.default_rng(sq)
    d, sk = 128, 70
    q = rng.standard_normal((6, hq, sq, d)).astype(np.float32)
    k = rng.standard_normal((6, 2, sk, d)).astype(np.float32)
    v = rng.standard_normal((6, 2, sk, d)).astype(np.float32)
    mask = np.zeros((6, 1, sq, sk), np.float32)
    mask[:, :, :, 40:] = -np.inf
    k[0, 0, 50, 3] = np.nan      # a masked key: the score is NaN all the same
    v[1, 1, 60, :5] = np.inf     # 0 x inf
    q[2], k[2, 0, 69] = np.abs(q[2]), 3e38  # the sum overflows in any order, the mask gives NaN
    mask[3, 0, sq - 1] = -np.inf  # a row that sees nothing
    q[4, 0, 0, 0] = np.inf
    mask[5] = np.finfo(np.float32).min
    bufs = [rt.buffer(x) for x in (q, k, v, mask)]
    got = r.gqa_attention(rt, *bufs).to_numpy()
    monkeypatch.setenv("RXW8_FORCE_GENERIC", "1")
    want = r.gqa_attention(rt, *bufs).to_numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.max(np.abs(got[ok] - want[ok])) <= 2e-5


def same_non_numbers(got, want):
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(got[np.isinf(got)], want[np.isinf(want)])
    ok = np.isfinite(want)
    assert np.max(np.abs(got[ok] - want[ok])) <= 2e-5


@pytest.mark.parametrize("sk", [1, 16, 70])
@pytest.mark.parametrize("d,sq,hq", [(64, 1, 4), (128, 4, 4), (256, 40, 2), (128, 40, 4)])
def test_infinite_value_of_the_last_key(rt, monkeypatch, d, sq, hq, sk):
    """The last key's row stands in for the rows that a 16-key tile has past
    it, with weight 0: an infinity there reaches the outputs as itself, as in
    the scalar kernel, and not as 0 x inf."""
    r = rx()
    rng = np.random.default_rng(sk + d)
    q = rng.standard_normal((2, hq, sq, d)).astype(np.float32)
    k = rng.standard_normal((2, 2, sk, d)).astype(np.float32)
    v = rng.standard_normal((2, 2, sk, d)).astype(np.float32)
    v[0, 1, sk - 1, :3], v[1, 0, sk - 1, d - 2:] = np.inf, -np.inf
    bufs = [rt.buffer(x) for x in (q, k, v, rng.standard_normal((2, 1, sq, sk)).astype(np.float32))]
    for rg in ("4", "2"):
        monkeypatch.setenv("RXW8_ATTN_F32_RG", rg)
        for mask in (bufs[3], None):
            got = r.gqa_attention(rt, *bufs[:3], mask).to_numpy()
            with monkeypatch.context() as m:
                m.setenv("RXW8_FORCE_GENERIC", "1")
                want = r.gqa_attention(rt, *bufs[:3], mask).to_numpy()
            assert np.isinf(want).any() and not np.isnan(want).any()
            same_non_numbers(got, want)


@pytest.mark.parametrize("d,cache", [(64, "bf16"), (256, "bf16"), (128, "f32")])
@pytest.mark.parametrize("hq", [2, 16])
def test_infinite_value_of_the_last_key_in_decode(rt, monkeypatch, d, cache, hq):
    r = rx()
    rng = np.random.default_rng(d + hq)
    lens = np.array([1, 16, 33, 70], np.int32)
    q = rng.standard_normal((4, hq, d)).astype(np.float32)
    k = oracle.round_bf16(rng.standard_normal((4, 1, 80, d)).astype(np.float32))
    v = oracle.round_bf16(rng.standard_normal((4, 1, 80, d)).astype(np.float32))
    for i in range(4):
        v[i, 0, lens[i] - 1, :3] = np.inf
    bits = (lambda x: rt.buffer(oracle.bf16_bits(x), r.DType.BF16)) if cache == "bf16" else rt.buffer
    bufs = (rt.buffer(q), bits(k), bits(v), rt.buffer(lens))
    got = r.grouped_query_attention(rt, *bufs).to_numpy()
    monkeypatch.setenv("RXW8_FORCE_GENERIC", "1")
    want = r.grouped_query_attention(rt, *bufs).to_numpy()
    assert np.isposinf(want[:, :, :3]).all() and np.isfinite(want[:, :, 3:]).all()
    same_non_numbers(got, want)


def captured(own, call):
    """The graph of call() on a stream of its own that stays the runtime's
    (call has run eagerly there first)."""
    import torch
    stream = torch.cuda.Stream()
    own.synchronize()
    own.set_stream(stream.cuda_stream)
    call()
    own.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream, capture_error_mode="thread_local"):
        call()
    return g, stream


@pytest.mark.parametrize("kind", ["decode", "decode-noalloc", "decode-d128", "masked", "prefill"])
def test_captured_calls_replay_beside_larger_ones(rt, kind):
    """A captured call gives the bits of the eager one (and the no-allocation
    decode call those of the other), at every replay, also with larger calls
    between and beside the replays: a captured call's split workspace is
    neither moved nor used by them. decode-d128 is the bf16 flash kernel, whose
    workspace the f32 kernels leave alone."""
    import torch
    r = rx()
    own = r.Runtime(0)
    rng = np.random.default_rng(3)
    d, dt = (128, r.DType.BF16) if kind == "decode-d128" else (256, r.DType.F32)
    f = lambda *shape: rng.standard_normal(shape).astype(np.float32)  # noqa: E731
    buf = lambda x: own.buffer(oracle.bf16_bits(x), dt) if dt == r.DType.BF16 else own.buffer(x)  # noqa: E731
    if kind == "masked":
        bufs = [own.buffer(x) for x in (f(1, 4, 20, 256), f(1, 2, 600, 256), f(1, 2, 600, 256), f(1, 1, 20, 600))]
        out = own.zeros((1, 4, 20, 256), r.DType.F32)
        call = lambda: r.gqa_attention(own, *bufs, out=out)  # noqa: E731
    elif kind == "prefill":
        kv = [own.buffer(oracle.bf16_bits(f(1, 2, 700, 64)), r.DType.BF16) for _ in range(2)]
        bufs = [own.buffer(f(1, 9, 8, 64)), *kv, own.buffer(np.array([600], np.int32))]
        out = own.zeros((1, 9, 8, 64), r.DType.F32)
        call = lambda: r.grouped_query_attention_prefill(own, *bufs, out=out)  # noqa: E731
    else:
        bufs = [own.buffer(f(2, 8, d)), buf(f(2, 2, 700, d)), buf(f(2, 2, 700, d)),
                own.buffer(np.array([700, 333], np.int32))]
        out = own.zeros((2, 8, d), r.DType.F32)
        fn = r.grouped_query_attention_noalloc if kind == "decode-noalloc" else r.grouped_query_attention
        call = lambda: fn(own, *bufs, out=out)  # noqa: E731
    if kind == "decode-noalloc":
        eager = r.grouped_query_attention(own, *bufs).to_numpy()
    else:
        call()
        eager = out.to_numpy()
    g, stream = captured(own, call)
    big = [own.buffer(x) for x in (f(8, 64, 256), f(8, 8, 2048, 256), f(8, 8, 2048, 256))]
    big_lens, big_out = own.buffer(np.full(8, 2048, np.int32)), own.zeros((8, 64, 256), r.DType.F32)
    prompt = [own.buffer(x) for x in (f(1, 16, 70, 128), f(1, 2, 4000, 128), f(1, 2, 4000, 128))]
    own.synchronize()
    own.set_stream(None)  # eager calls on a stream of their own from here on
    want = r.grouped_query_attention(own, *big, big_lens).to_numpy()
    for _ in range(4):
        out.copy_from(np.full(out.shape, 7.0, np.float32))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            g.replay()
            g.replay()
        if kind != "decode-d128":  # beside the replays
            r.grouped_query_attention(own, *big, big_lens, out=big_out)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.to_numpy(), eager)
        r.grouped_query_attention(own, *big, big_lens, out=big_out)
        r.gqa_attention(own, *prompt, None)
        np.testing.assert_array_equal(big_out.to_numpy(), want)
