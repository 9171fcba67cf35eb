"""GPU parity of the encoder's conv stem (three bf16 parts per f32 operand) against
float64 at the edges of its tiles, over mixed magnitudes and for values that are
not finite."""
import math

import numpy as np
import pytest

from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


def conv64(x, w, b, stride):
    c, t = x.shape
    xp = np.zeros((c, t + 2))
    xp[:, 1:-1] = x
    n = (t - 1) // stride + 1
    cols = np.stack([xp[:, k:k + stride * (n - 1) + 1:stride] for k in range(3)], 1).reshape(3 * c, n)
    return w.reshape(w.shape[0], -1).astype(np.float64) @ cols + b.astype(np.float64)[:, None]


def gelu64(x):
    return 0.5 * x * (1.0 + np.vectorize(math.erf)(x / math.sqrt(2.0)))


def weights(g, nm, d, wscale):
    return [(wscale * g.standard_normal(s)).astype(np.float32) for s in ((d, nm, 3), (d,), (d, d, 3), (d,))]


def stem(ctx, g, nm, nf, d, wscale, W=None):
    W = weights(g, nm, d, wscale) if W is None else W
    pos = (0.1 * g.standard_normal(((nf - 1) // 2 + 1, d))).astype(np.float32)
    one, zero = np.ones(d, np.float32), np.zeros(d, np.float32)
    enc = hip.Encoder(ctx, hip.WDtype.Q8_0, d, d // 64, 4 * d, [], one, zero, 4 * nf)
    enc.set_stem(nm, nf, *W, pos)
    return enc, W, pos


def run(ctx, enc, x, d):
    b = x.shape[0]
    d_m, d_x = hip.DeviceBuffer.from_array(ctx, x), hip.DeviceBuffer(ctx, b * enc.n_ctx * d * 4)
    enc.stem_dev(b, d_m, d_x)
    ctx.synchronize()
    return d_x.download(np.float32, b * enc.n_ctx * d).reshape(b, enc.n_ctx, d)


def check(got, x, W, pos):
    h = gelu64(conv64(x.astype(np.float64), W[0], W[1], 1))
    y = conv64(h, W[2], W[3], 2)
    # products and f32 sums to 2e-6 of the terms' magnitudes, the GELU polynomial's 1.5e-7, f32 positions
    mag = conv64(np.abs(h) + 1.5e-7, np.abs(W[2]), np.abs(W[3]), 2)
    want = gelu64(y).T + pos
    bound = 2e-6 * mag.T + 2e-7 * np.abs(y).T + 2e-7 + 1e-6 * np.abs(want)
    assert (np.abs(got - want) <= bound).all(), np.max(np.abs(got - want) / bound)


# channels off 16, an odd frame count, few frames, 64- and 128-row tiles (the
# last from 256 of them), inputs and weights far from one
@pytest.mark.parametrize("nm,nf,d,batch,xscale,wscale", [
    (80, 67, 64, 2, 1.0, 0.05), (1, 2, 64, 1, 1.0, 0.3), (33, 131, 128, 3, 1e-30, 0.05), (128, 300, 192, 1, 1e18, 1e-3),
    (17, 4101, 1024, 2, 1.0, 0.03),
])
def test_stem_vs_float64(ctx, nm, nf, d, batch, xscale, wscale):
    print(f"[case] stem mels={nm} frames={nf} d={d} batch={batch} x {xscale}", flush=True)
    g = np.random.default_rng(nm + nf)
    enc, W, pos = stem(ctx, g, nm, nf, d, wscale)
    x = (xscale * g.standard_normal((batch, nm, nf))).astype(np.float32)
    got = run(ctx, enc, x, d)
    for b in {0, batch - 1}:
        check(got[b], x[b], W, pos)
    if batch > 1:  # a clip's result does not depend on its batch
        x2 = x.copy()
        x2[0] *= 3.0
        assert np.array_equal(run(ctx, enc, x2, d)[1:], got[1:])


def test_stem_non_finite_clip_leaves_the_others(ctx):
    g = np.random.default_rng(3)
    enc, _, _ = stem(ctx, g, 80, 90, 64, 0.05)
    x = g.standard_normal((2, 80, 90)).astype(np.float32)
    want = run(ctx, enc, x, 64)
    x[0, 5, 40] = np.nan
    got = run(ctx, enc, x, 64)
    assert np.array_equal(got[1], want[1])
    bad = np.isnan(got[0]).any(1)  # frames 39 .. 41 of the first convolution: frames 19 .. 21 of the second
    assert bad[19:21].all() and not bad[:19].any() and not bad[22:].any()
    assert np.array_equal(got[0][~bad], want[0][~bad])


def test_stem_keeps_small_values_beside_large_ones(ctx):
    """Each operand tensor with values 2^-24 and less of its largest one that alone
    decide some outputs: in f32 products they keep all their bits."""
    g = np.random.default_rng(5)
    nm, nf, d = 20, 70, 64
    W = weights(g, nm, d, 0.05)
    W[0][:, 1:] *= np.float32(2.0 ** 24)  # small channels, large weights, and the other way round
    W[0][1:, 0] = 0.0
    W[1][3] = 2.0 ** 26  # a channel that the second convolution does not weigh
    W[2][:, 3] = 0.0
    W[2][8:16] *= np.float32(2.0 ** 20)
    W[3][8:16] = 0.0
    enc, W, pos = stem(ctx, g, nm, nf, d, 0.05, W)
    x = g.standard_normal((1, nm, nf)).astype(np.float32)
    x[:, 1:] *= np.float32(2.0 ** -24)
    check(run(ctx, enc, x, d)[0], x[0], W, pos)


def test_stem_infinities_and_the_largest_finite_value(ctx):
    """An infinite input gives the infinities that f32 products give, and a finite one
    that has no finite bf16 next to it stays finite."""
    g = np.random.default_rng(6)
    nm, nf, d = 16, 90, 64
    W = [np.abs(w) for w in weights(g, nm, d, 0.05)]
    W[0][:, 7] *= np.float32(1e-30)
    enc, W, pos = stem(ctx, g, nm, nf, d, 0.05, W)
    x = np.abs(g.standard_normal((1, nm, nf))).astype(np.float32)
    x[0, 7, 50] = np.finfo(np.float32).max
    want = run(ctx, enc, x, d)
    check(want[0], x[0], W, pos)
    x[0, 5, 20] = np.inf
    got = run(ctx, enc, x, d)
    hit = np.zeros(enc.n_ctx, bool)
    hit[9:12] = True  # frames 19 .. 21 of the first convolution
    assert (got[0][hit] == np.inf).all() and np.array_equal(got[0][~hit], want[0][~hit])


def test_stem_of_many_short_clips(ctx):
    """Clip and row counts past 16 bits; each clip as alone."""
    g = np.random.default_rng(7)
    n, d = 65537, 64
    W = weights(g, 1, d, 0.3)
    pos = (0.1 * g.standard_normal((1, d))).astype(np.float32)
    enc = hip.Encoder(ctx, hip.WDtype.Q8_0, d, 1, 64, [], np.ones(d, np.float32), np.zeros(d, np.float32), n)
    enc.set_stem(1, 2, *W, pos)
    x = g.standard_normal((n, 1, 2)).astype(np.float32)
    got = run(ctx, enc, x, d)
    for i in (0, 1, 65535, 65536):
        assert np.array_equal(run(ctx, enc, x[i:i + 1], d)[0], got[i])
        check(got[i], x[i], W, pos)
