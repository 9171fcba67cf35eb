"""GPU parity of attention calls whose keys split over workgroups (few query
tiles and heads, several key tiles) and of their merge, against float64, at the
edges of tiles and chunks; an item alone equals the item in a batch, both in one
that splits and in one that runs the chunks in place, bit for bit."""
import numpy as np
import pytest

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


@pytest.mark.parametrize("hd,hq,hkv,t,batch", [(64, 8, 8, 700, 2), (64, 8, 8, 700, 9), (128, 8, 2, 300, 3)])
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
