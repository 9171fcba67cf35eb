"""GPU parity of attention calls whose keys split over workgroups (few query
tiles and heads, several key tiles) and of their merge, against float64, at the
edges of tiles and chunks; an item alone equals the item in a batch, both in one
that splits and in one that runs the chunks in place, bit for bit."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_sessions import enc_layer
from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


def sdpa64(q, k, v, hq, hkv, hd, scale, causal, off):
    """float64 attention of one item, q [tq, hq*hd], k / v [tkv, hkv*hd]."""
    tq, tkv = q.shape[0], k.shape[0]
    out = np.zeros((tq, hq * hd))
    for h in range(hq):
        kh = slice((h // (hq // hkv)) * hd, (h // (hq // hkv) + 1) * hd)
        s = (q[:, h * hd:(h + 1) * hd].astype(np.float64) * scale) @ k[:, kh].astype(np.float64).T
        if causal:
            s[np.arange(tkv)[None] > off + np.arange(tq)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h * hd:(h + 1) * hd] = (p / p.sum(1, keepdims=True)) @ v[:, kh].astype(np.float64)
    return out


@pytest.mark.parametrize("hd,hq,hkv,tq,tkv,causal", [
    (64, 4, 4, 2, 321, False),     # fewest queries, five tiles and one key
    (64, 6, 6, 65, 640, False),    # a second query tile of one
    (64, 4, 2, 400, 400, True),    # unequal query tiles: one chunk and several
    (128, 16, 2, 130, 500, True),  # after a history of 370 positions
    (128, 2, 1, 64, 2000, False),  # many chunks
    (64, 3, 3, 33, 1281, True),    # later chunks masked for some queries
])
def test_key_splits_vs_float64(ctx, hd, hq, hkv, tq, tkv, causal):
    print(f"[case] attention key splits {hd} {hq}/{hkv} {tq}x{tkv} causal={causal}", flush=True)
    g = np.random.default_rng(tq + tkv)
    q = (3 * g.standard_normal((1, tq, hq * hd))).astype(np.float32)
    k = g.standard_normal((1, tkv, hkv * hd)).astype(np.float32)
    v = g.standard_normal((1, tkv, hkv * hd)).astype(np.float32)
    off = tkv - tq if causal else 0
    got = ctx.attn_f32(q, k, v, hq, hkv, causal=causal, q_offset=off)[0]
    want = sdpa64(q[0], k[0], v[0], hq, hkv, hd, hd ** -0.5, causal, off)
    # about 22 bits per product, f32 sums and exponentials: the bar of the undivided kernel's float64 comparison
    assert np.abs(got - want).max() <= 2e-5


# over workgroups in one launch, in place at both head_dims (768 query tiles and heads
# or more), and over workgroups in slices of the batch
@pytest.mark.parametrize("hd,hq,hkv,t,batch", [(64, 8, 8, 700, 2), (64, 8, 8, 700, 9), (128, 8, 2, 300, 3),
                                               (128, 16, 2, 300, 10), (64, 1, 1, 704, 60)])
def test_split_item_does_not_depend_on_the_batch(ctx, hd, hq, hkv, t, batch):
    print(f"[case] split attention batch {batch} == alone, hd {hd}", flush=True)
    g = np.random.default_rng(batch)
    q = g.standard_normal((batch, t, hq * hd)).astype(np.float32)
    k = g.standard_normal((batch, t, hkv * hd)).astype(np.float32)
    v = g.standard_normal((batch, t, hkv * hd)).astype(np.float32)
    for causal in (False, True):
        full = ctx.attn_f32(q, k, v, hq, hkv, causal=causal)
        for b in (0, batch - 1):
            assert np.array_equal(ctx.attn_f32(q[b], k[b], v[b], hq, hkv, causal=causal), full[b])


def test_non_finite_values_stay_in_their_rows(ctx):
    """A NaN in one value row reaches exactly the outputs that weigh it (all
    queries of its head and dimension), an unreachable key's nothing."""
    g = np.random.default_rng(1)
    t, H, hd = 640, 2, 64
    q, k, v = (g.standard_normal((1, t, H * hd)).astype(np.float32) for _ in range(3))
    v[0, 600, 5] = np.nan
    got = ctx.attn_f32(q, k, v, H, causal=False)[0]
    assert np.isnan(got[:, 5]).all() and np.isnan(got).sum() == t


class At:
    """A device buffer's pointer, `off` bytes in."""

    def __init__(self, buf, off):
        self.buf, self.ptr = buf, ctypes.c_void_p(buf.ptr.value + off)


def test_slices_of_a_batch_equal_its_items(ctx):
    """Few queries over many keys: more chunks than the partials' workspace holds."""
    g = np.random.default_rng(4)
    batch, tq, tkv, hd = 700, 3, 704, 64
    q = g.standard_normal((batch, tq, hd)).astype(np.float32)
    k = g.standard_normal((batch, tkv, hd)).astype(np.float32)
    v = g.standard_normal((batch, tkv, hd)).astype(np.float32)
    full = ctx.attn_f32(q, k, v, 1)
    for b in (0, 681, 682, 683, batch - 1):
        assert np.array_equal(ctx.attn_f32(q[b], k[b], v[b], 1), full[b])


@pytest.mark.parametrize("hd,h,t", [(64, 4, 321), (128, 2, 130)])
def test_values_off_16_bytes(ctx, hd, h, t):
    """v may start anywhere (q, k and out are 16-byte aligned)."""
    g = np.random.default_rng(hd)
    q, k, v = (g.standard_normal((t, h * hd)).astype(np.float32) for _ in range(3))
    want = ctx.attn_f32(q, k, v, h)
    d_q, d_k = (hip.DeviceBuffer.from_array(ctx, x) for x in (q, k))
    d_v = hip.DeviceBuffer.from_array(ctx, np.concatenate([np.full(1, 9.0, np.float32), v.reshape(-1)]))
    d_o = hip.DeviceBuffer(ctx, q.nbytes)
    ctx.attn_f32_dev(1, t, t, h, h, hd, d_q, d_k, At(d_v, 4), hd ** -0.5, False, 0, d_o)
    ctx.synchronize()
    assert np.array_equal(d_o.download(np.float32, q.size).reshape(q.shape), want)


def test_captured_split_without_its_workspace():
    """A capture on a context whose calls have not split their keys yet allocates
    nothing and replays the eager call's bits."""
    ctx = hip.HipContext(0)
    g = np.random.default_rng(11)
    wide = [hip.DeviceBuffer.from_array(ctx, g.standard_normal((800, 40 * 64)).astype(np.float32)) for _ in range(4)]
    ctx.attn_f32_dev(1, 800, 800, 40, 40, 64, *wide[:3], 0.125, False, 0, wide[3])  # 520 query tiles and heads: whole
    q, k, v = (g.standard_normal((1500, 8 * 64)).astype(np.float32) for _ in range(3))
    d = [hip.DeviceBuffer.from_array(ctx, x) for x in (q, k, v)]
    d_o = hip.DeviceBuffer(ctx, q.nbytes)
    graph = ctx.capture(lambda: ctx.attn_f32_dev(1, 1500, 1500, 8, 8, 64, *d, 0.125, False, 0, d_o))
    graph.launch()
    ctx.synchronize()
    first = d_o.download(np.float32, q.size)
    ctx.attn_f32_dev(1, 1500, 1500, 8, 8, 64, *d, 0.125, False, 0, d_o)  # eager: over workgroups
    ctx.synchronize()
    want = d_o.download(np.float32, q.size)
    assert np.array_equal(first, want)
    for _ in range(2):
        d_o.upload(np.zeros_like(q))
        graph.launch()
        ctx.synchronize()
        assert np.array_equal(d_o.download(np.float32, q.size), want)
    del graph
    ctx.close()


def test_captured_encoder_outlives_larger_attention_calls():
    """A captured encoder forward whose attention splits its keys, replayed after eager
    attention calls that split more: the partials' block is never replaced."""
    ctx = hip.HipContext(0)
    g = np.random.default_rng(12)
    d, frames = 512, 700
    layers = [enc_layer(ctx, g, hip.WDtype.Q8_0, d, 4 * d, scale=0.02)]
    one, zero = np.ones(d, np.float32), np.zeros(d, np.float32)
    enc = hip.Encoder(ctx, hip.WDtype.Q8_0, d, d // 64, 4 * d, layers, one, zero, frames)
    x = g.standard_normal((1, frames, d)).astype(np.float32)
    d_x, d_o = hip.DeviceBuffer.from_array(ctx, x), hip.DeviceBuffer(ctx, x.nbytes)
    enc.forward_dev(1, frames, d_x, d_o)
    ctx.synchronize()
    want = d_o.download(np.float32, x.size)
    graph = ctx.capture(lambda: enc.forward_dev(1, frames, d_x, d_o))
    q, k, v = (g.standard_normal((777, 16 * 128)).astype(np.float32) for _ in range(3))
    other = ctx.attn_f32(q, k, v, 16, causal=True)
    for _ in range(3):
        d_o.upload(np.zeros_like(x))
        graph.launch()
        ctx.synchronize()
        assert np.array_equal(d_o.download(np.float32, x.size), want)
        assert np.array_equal(ctx.attn_f32(q, k, v, 16, causal=True), other)
    del graph, enc
    ctx.close()
