"""GPU parity for causal GQA attention over a ragged batch of prefill tokens (config C4's attention: 16 q heads,
2 kv heads, head_dim 256, 16-token pages, a prefix shared by the sessions).

Each token (session s, position p) is compared with the oracle's dense softmax attention (reference.cpp:492-527)
over its session's K/V rows 0..p, times sigmoid(gate): within 1e-5 relative to sum|p||v| (fp16 matrix-core products of split
hi / lo operands, fp32 accumulation),
and the Q8 output equal to the quantization of the fp32 output it wrote.
"""
import ctypes

import numpy as np
import pytest

import halo_amd as H
import oracle_py as O
from test_gpu_attn import build, gather, outlier_kv, outlier_q

pytestmark = pytest.mark.gpu
D = 256


@pytest.mark.parametrize("S,prefix,segs,max_context", [
    (1, 0, [(0, 0, 100)], 256),
    (4, 512, [(0, 512, 37), (1, 512, 130), (2, 512, 1), (3, 512, 69), (0, 549, 8)], 512 + 256),
    (1, 0, [(0, 0, 64), (0, 64, 33)], 128),
])
def test_attn_prefill(dev, S, prefix, segs, max_context):
    run_case(dev, S, prefix, segs, max_context)


@pytest.mark.parametrize("qk,v", [(0.1, 1e-3), (2.0, 50.0)])
def test_attn_prefill_operand_magnitudes(dev, qk, v):
    """Small and large operands (q and K scaled by qk, V by v): the split-fp16 products keep the 1e-5 bar relative
    to sum |p| |v| with no absolute slack (V of 1e-3 is below the range whose lo halves an unscaled split keeps normal; the
    split paths scale their operands by powers of two, which covers |V| from about 1e-4 to 255)."""
    run_case(dev, 1, 0, [(0, 0, 70)], 128, qk, v, abs_tol=0.0)


def test_attn_prefill_outlier_channels(dev):
    """|q|, |K| and |V| far above 255 in single channels, the V outliers only on the page of positions 32-47 (the
    second 32-key chunk): query rows and K chunks take smaller power-of-two scales, and the V scale drops at that chunk
    (the accumulators of the rows that saw the first chunk are rescaled); same 1e-5 bar, outputs finite."""
    run_case(dev, 1, 0, [(0, 0, 90)], 128, outliers=True)


def run_case(dev, S, prefix, segs, max_context, qk=1.0, v=1.0, abs_tol=1e-6, outliers=False):
    Hq, Hkv = 16, 2
    rng = np.random.default_rng(S + prefix + len(segs))
    tweak = (lambda k_, v_, p_: outlier_kv(k_, v_, v_pages=[int(p_[0, 2])])) if outliers else None
    desc, g, kp, vp, pages, _ = build(dev, rng, S, Hkv, prefix, [max_context - prefix] * S, max_context, qk, v,
                                      tweak=tweak)
    seg_arr = (H.PrefillSegment * len(segs))()
    first = 0
    toks = []
    for i, (s, start, n) in enumerate(segs):
        seg_arr[i] = H.PrefillSegment(s, start, n, first)
        toks += [(s, start + j) for j in range(n)]
        first += n
    T = len(toks)
    q = (qk * rng.normal(0, 1, (T, Hq, D))).astype(np.float32)
    if outliers:
        outlier_q(q)
    gate = rng.normal(0, 1, (T, Hq, D)).astype(np.float32)
    gq, gg = dev.to_device(q), dev.to_device(gate)
    go = dev.array((T, Hq, D), np.float32)
    goq, gos = dev.array((T, Hq * D), np.int8), dev.array((T, Hq * D // 32), np.float32)
    nbytes = H.lib().halo_op_attn_prefill_workspace_bytes(seg_arr, len(segs))
    ws = dev.array(nbytes, np.uint8)
    dev.op("attn_prefill", ctypes.byref(desc),
           seg_arr, len(segs), gq.ptr, gg.ptr, go.ptr, goq.ptr, gos.ptr, Hq, ws.ptr, nbytes)
    got = go.download()
    assert np.isfinite(got).all()
    o = O.oracle()
    G = Hq // Hkv
    for ti, (s, p) in enumerate(toks):
        n = p + 1
        for h in range(Hq):
            K = np.ascontiguousarray(gather(kp, pages[s], n, h // G))
            V = np.ascontiguousarray(gather(vp, pages[s], n, h // G))
            oh = np.zeros(D, np.float32)
            o.or_attention_head(np.ascontiguousarray(q[ti, h]), K, V, n, D, D, oh)
            sg = 1 / (1 + np.exp(-gate[ti, h].astype(np.float64)))
            sc = K.astype(np.float64) @ q[ti, h] / 16.0
            pr = np.exp(sc - sc.max())
            pr /= pr.sum()
            mag = (pr @ np.abs(V)) * sg
            assert np.all(np.abs(got[ti, h] - oh * sg) <= 1e-5 * mag + abs_tol), f"token {ti} (s {s}, p {p}) head {h}"
    xq, xs = O.quantize(got.reshape(T, Hq * D))
    assert np.array_equal(goq.download(), xq)
    assert np.array_equal(gos.download().view(np.uint32), xs.view(np.uint32))


@pytest.mark.parametrize("segs", [
    [(0, 0, 7), (0, 7, 1), (0, 8, 8), (0, 16, 9)],  # 8-token tiles: below, at and past one
    [(0, 0, 33)],
])
def test_attn_prefill_tile_edges(dev, segs):
    run_case(dev, 1, 0, segs, 64)


def test_attn_prefill_tile_shapes_bitwise(dev):
    """A 2300-token prompt takes 16-token tiles, the same prompt in calls of 512 tokens 8-token ones (the output dims split
    over two waves): a query's operations are the same in both, so the outputs are equal bit for bit; and tokens at
    the edges of tiles and chunks match softmax attention in 64 bits within 1e-5 of sum |p| |v|."""
    Hq, Hkv, T = 16, 2, 2300
    rng = np.random.default_rng(11)
    desc, g, kp, vp, pages, _ = build(dev, rng, 1, Hkv, 0, [T], 2304, 2.0, 1.0)
    q = (2.0 * rng.normal(0, 1, (T, Hq, D))).astype(np.float32)
    gate = rng.normal(0, 1, (T, Hq, D)).astype(np.float32)
    gq, gg = dev.to_device(q), dev.to_device(gate)

    def run(pieces):
        go = dev.array((T, Hq, D), np.float32).fill(0)
        for start, n in pieces:
            seg = (H.PrefillSegment * 1)(H.PrefillSegment(0, start, n, start))
            nbytes = H.lib().halo_op_attn_prefill_workspace_bytes(seg, 1)
            ws = dev.array(nbytes, np.uint8)
            dev.op("attn_prefill", ctypes.byref(desc), seg, 1, gq.ptr, gg.ptr, go.ptr, None, None, Hq, ws.ptr, nbytes)
            dev.sync()
        return go.download()

    whole = run([(0, T)])
    assert np.array_equal(whole.view(np.uint32), run([(k, min(512, T - k)) for k in range(0, T, 512)]).view(np.uint32))
    for p in (0, 3, 15, 16, 31, 32, 33, 511, 1087, 1088, T - 2, T - 1):
        for h in (0, 7, 8, 15):
            K = gather(kp, pages[0], p + 1, h // 8).astype(np.float64)
            V = gather(vp, pages[0], p + 1, h // 8).astype(np.float64)
            s = K @ q[p, h].astype(np.float64) / 16.0
            pr = np.exp(s - s.max())
            pr /= pr.sum()
            sg = 1 / (1 + np.exp(-gate[p, h].astype(np.float64)))
            assert np.all(np.abs(whole[p, h] - pr @ V * sg) <= 1e-5 * (pr @ np.abs(V)) * sg + 1e-7), f"token {p} head {h}"


def reference(q, gate, kp, vp, pages_s, p, h):
    """One query's output in 64 bits and the magnitude of its terms, sum |p| |v| times the gate."""
    K = gather(kp, pages_s, p + 1, h // 8).astype(np.float64)
    V = gather(vp, pages_s, p + 1, h // 8).astype(np.float64)
    sc = K @ q.astype(np.float64) / 16.0
    pr = np.exp(sc - sc.max())
    pr /= pr.sum()
    sg = 1 / (1 + np.exp(-gate.astype(np.float64)))
    return pr @ V * sg, pr @ np.abs(V) * sg


def prefill(dev, desc, segs, gq, gg, T, Hq):
    """halo_op_attn_prefill over segs [(session, start, length)], tokens in order; o fp32."""
    arr, first = (H.PrefillSegment * len(segs))(), 0
    for i, (s, start, n) in enumerate(segs):
        arr[i] = H.PrefillSegment(s, start, n, first)
        first += n
    assert first == T
    go = dev.array((T, Hq, D), np.float32).fill(0)
    nbytes = H.lib().halo_op_attn_prefill_workspace_bytes(arr, len(segs))
    ws = dev.array(nbytes, np.uint8)
    dev.op("attn_prefill", ctypes.byref(desc), arr, len(segs), gq.ptr, gg.ptr, go.ptr, None, None, Hq, ws.ptr, nbytes)
    return go.download()


@pytest.mark.parametrize("T", [600, 1100, 2304])
def test_attn_prefill_any_split_bitwise(dev, T):
    """A prompt whole and in pieces whose tiles start at other tokens (a query then shares its wave and its 32-key
    chunks' tiles with other queries, and the pieces take either tile size): a query's bits are its own."""
    Hq, Hkv = 16, 2
    rng = np.random.default_rng(T)
    desc, g, *_ = build(dev, rng, 1, Hkv, 0, [T], T, 2.0, 1.0)
    q = (2.0 * rng.normal(0, 1, (T, Hq, D))).astype(np.float32)
    gate = rng.normal(0, 1, (T, Hq, D)).astype(np.float32)

    def run(pieces):
        out = []
        for a, n in pieces:
            gq, gg = dev.to_device(q[a : a + n]), dev.to_device(gate[a : a + n])
            out.append(prefill(dev, desc, [(0, a, n)], gq, gg, n, Hq))
        return np.concatenate(out).view(np.uint32)

    whole = run([(0, T)])
    for pieces in ([(0, 66), (66, 1), (67, T - 67)], [(0, 5), (5, 258), (263, T - 263)]):
        assert np.array_equal(whole, run(pieces)), pieces


@pytest.mark.parametrize("T", [300, 2400])  # 8-token tiles, 16-token tiles
@pytest.mark.parametrize("bits", [8, 20])
def test_attn_prefill_dominant_key(dev, T, bits):
    """The first key takes the weight (2^bits above every other one) and its V is zero, so the output is made of small
    probabilities alone. The other keys' scores are equal and V is positive, so that their rounding errors add up instead
    of averaging out. A probability is split at 2^14 times its size against the row's largest: its low half is within
    2^-25, 2^-39 of the largest, here at most 2^(bits + 1.5 - 39) of a probability (5.4e-6), under the 1e-5 bar."""
    dominant_key_case(dev, T, bits)


def dominant_key_case(dev, T, bits, outlier=None):
    Hq, Hkv = 16, 2
    rng = np.random.default_rng(bits)

    def tweak(kp, vp, pages):
        kp[:] = 0
        kp[pages[0, 0], :, 0] = np.where(np.arange(D) % 3 == 0, -0.875, 0.875)
        vp[:] = rng.uniform(0.5, 1.5, vp.shape)
        vp[pages[0, 0], :, 0] = 0
        if outlier is not None:
            pos, value = outlier
            vp[pages[0, pos // 16], :, pos % 16, 77] = value

    desc, g, kp, vp, pages, _ = build(dev, rng, 1, Hkv, 0, [T], -(-T // 16) * 16, tweak=tweak)
    # q . k0 / 16 = 14 c: the first score is bits + (0 .. 1.5) base-2 units above the others, c in steps of 2^-10 (exact)
    c = np.round(1024 * (bits + 1.5 * rng.random((T, Hq, 1))) * np.log(2) / 14) / 1024
    q = (c * np.where(np.arange(D) % 3 == 0, -1.0, 1.0)).astype(np.float32)
    gate = rng.normal(0, 1, (T, Hq, D)).astype(np.float32)
    got = prefill(dev, desc, [(0, 0, T)], dev.to_device(q), dev.to_device(gate), T, Hq)
    assert np.isfinite(got).all()
    worst = 0.0
    for p in sorted({1, 31, 32, 63, 64, 100, T // 2, T - 2, T - 1} | set(rng.integers(1, T, 20).tolist())):
        for h in range(0, Hq, 3):
            want, mag = reference(q[p, h], gate[p, h], kp, vp, pages[0], p, h)
            worst = max(worst, float(np.max(np.abs(got[p, h] - want) / mag)))
    assert worst <= 1e-5, f"{worst:.3g} of sum |p| |v|"


@pytest.mark.parametrize("T", [300, 2400])  # 8-token tiles, 16-token tiles
@pytest.mark.parametrize("outlier", [(5, 1e6), (40, 1e6), (40, 1e4), (270, -1e6)])
def test_attn_prefill_value_outlier(dev, T, outlier):
    """One V far above the rest (position, value), in the first 32-key chunk, the second or a later one: V of the chunks
    after it is staged at its smaller scale (2^-5 for 1e6: V keeps 2^-20 of itself) and the accumulators before it are
    rescaled exactly, while the probabilities, 2^8 below the first key's, keep their bits; the 1e-5 bar in every dim."""
    dominant_key_case(dev, T, 8, outlier)


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_attn_prefill_nonfinite_value(dev, value):
    """An infinite or NaN V makes its own dim of the queries that see its chunk non-finite, and nothing else."""
    Hq, Hkv, T, pos = 16, 2, 200, 70
    rng = np.random.default_rng(3)
    tweak = lambda kp, vp, pages: vp[pages[0, pos // 16]].__setitem__((slice(None), pos % 16, 9), value)  # noqa: E731
    desc, g, kp, vp, pages, _ = build(dev, rng, 1, Hkv, 0, [T], 208, tweak=tweak)
    q, gate = (rng.normal(0, 1, (T, Hq, D)).astype(np.float32) for _ in range(2))
    got = prefill(dev, desc, [(0, 0, T)], dev.to_device(q), dev.to_device(gate), T, Hq)
    others = np.arange(D) != 9
    assert np.isfinite(got[..., others]).all() and np.isfinite(got[:64]).all()
    assert not np.isfinite(got[pos:, :, 9]).any()
    vp[pages[0, pos // 16], :, pos % 16, 9] = 0
    for p in (63, 69, 70, 95, 96, T - 1):
        want, mag = reference(q[p, 3], gate[p, 3], kp, vp, pages[0], p, 3)
        assert np.all((np.abs(got[p, 3] - want) <= 1e-5 * mag + 1e-6)[others])


@pytest.mark.parametrize("qk,v,outliers", [(1.0, 1.0, False), (0.1, 1e-3, False), (2.0, 50.0, False), (1.0, 1.0, True)])
def test_attn_prefill_long_segments(dev, qk, v, outliers):
    """Ragged segments behind a shared prefix, long enough for 16-token tiles: plain, small and large operands, and outlier
    channels (V's on the page of positions 32 .. 47 of the prefix alone), as the short cases above, against 64 bits at
    tokens around tile, chunk and segment edges and at random ones; the Q8 output is the fp32 output's."""
    Hq, Hkv, prefix = 16, 2, 512
    segs = [(0, 512, 700), (1, 512, 1100), (2, 512, 1), (3, 512, 513)]
    rng = np.random.default_rng(int(10 * v) + outliers)
    tweak = (lambda k_, v_, p_: outlier_kv(k_, v_, v_pages=[int(p_[0, 2])])) if outliers else None
    desc, g, kp, vp, pages, _ = build(dev, rng, 4, Hkv, prefix, [1100] * 4, 1616, qk, v, tweak=tweak)
    T = sum(n for *_, n in segs)
    q = (qk * rng.normal(0, 1, (T, Hq, D))).astype(np.float32)
    if outliers:
        outlier_q(q)
    gate = rng.normal(0, 1, (T, Hq, D)).astype(np.float32)
    gq, gg = dev.to_device(q), dev.to_device(gate)
    arr, first = (H.PrefillSegment * 4)(), 0
    for i, (s, start, n) in enumerate(segs):
        arr[i] = H.PrefillSegment(s, start, n, first)
        first += n
    go, goq = dev.array((T, Hq, D), np.float32), dev.array((T, Hq * D), np.int8)
    gos = dev.array((T, Hq * D // 32), np.float32)
    nbytes = H.lib().halo_op_attn_prefill_workspace_bytes(arr, 4)
    ws = dev.array(nbytes, np.uint8)
    dev.op("attn_prefill", ctypes.byref(desc), arr, 4, gq.ptr, gg.ptr, go.ptr, goq.ptr, gos.ptr, Hq, ws.ptr, nbytes)
    got = go.download()
    assert np.isfinite(got).all()
    first = 0
    for s, start, n in segs:
        picks = {0, 1, 7, 8, 15, 16, 31, 32, n - 2, n - 1} | set(rng.integers(0, n, 12).tolist())
        for k in sorted(x for x in picks if 0 <= x < n):
            for h in range(Hq):
                want, mag = reference(q[first + k, h], gate[first + k, h], kp, vp, pages[s], start + k, h)
                assert np.all(np.abs(got[first + k, h] - want) <= 1e-5 * mag), f"session {s} position {start + k} head {h}"
        first += n
    xq, xs = O.quantize(got.reshape(T, Hq * D))
    assert np.array_equal(goq.download(), xq)
    assert np.array_equal(gos.download().view(np.uint32), xs.view(np.uint32))
