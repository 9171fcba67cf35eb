"""GPU parity of the paged cache's append at the edges of its launches (one
workgroup for small batches, two launches beyond) and of the matrix-core decode
attention's split of its operands."""
import numpy as np
import pytest

from tests.test_gpu_textdec import make_layers
from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


# width x items on both sides of 2048 values, items on both sides of a wave and up
# to the call's 1024
@pytest.mark.parametrize("H,hd,n", [(2, 128, 1), (2, 128, 8), (2, 128, 9), (1, 64, 32), (1, 64, 33), (3, 64, 10),
                                    (2, 64, 65), (1, 64, 1024)])
def test_append_batches_lockstep(ctx, oracle, H, hd, n):
    print(f"[case] append {n} items of {H} x {hd}", flush=True)
    n_layer, n_stream, bs, max_time = 2, 7, 4, 256
    g = np.random.default_rng(n + hd)
    kv = ctx.kv_cache(n_layer, H, hd, n_stream, max_time, bs)
    ref = oracle.PagedCache(n_layer, H, hd, n_stream, max_time, bs, 3)
    w = H * hd
    for _ in range(3):
        streams = g.integers(0, n_stream, n).astype(np.int32)  # slots and pages repeat within a batch
        times = g.integers(0, max_time, n).astype(np.int32)
        k = g.standard_normal((n, w)).astype(np.float32)
        v = g.standard_normal((n, w)).astype(np.float32)
        k[0, :3] = np.nan, np.inf, -np.inf
        kv.append(1, streams, times, k, v)
        for i in range(n):
            assert ref.append_step(1, int(times[i]), int(streams[i]), k[i], v[i]) == 0
        assert kv.pages() == (ref.free_pages(), ref.pages_in_use())
        for i in g.choice(n, min(n, 12), replace=False):
            got, want = kv.read(1, int(times[i]), int(streams[i])), ref.read_step(1, int(times[i]), int(streams[i]))
            assert all(np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))
                       for a, b in zip(got, want))


def test_append_rows_off_16_bytes(ctx):
    """A small batch whose rows start off 16 bytes takes the two launches: same cache."""
    H, hd, n = 2, 64, 5
    g = np.random.default_rng(9)
    streams, times = np.arange(n, dtype=np.int32) % 3, np.arange(n, dtype=np.int32) * 3
    k, v = (g.standard_normal((n, H * hd)).astype(np.float32) for _ in range(2))
    a, b = (ctx.kv_cache(1, H, hd, 3, 32, 4) for _ in range(2))
    a.append(0, streams, times, k, v)
    d_s, d_t = (hip.DeviceBuffer.from_array(ctx, x) for x in (streams, times))
    rows = [hip.DeviceBuffer.from_array(ctx, np.concatenate([np.full(1, 9.0, np.float32), np.ravel(x)])) for x in (k, v)]

    class Off:
        def __init__(self, buf):
            self.ptr = type(buf.ptr)(buf.ptr.value + 4)
    b.append_dev(0, n, d_s, d_t, *(Off(r) for r in rows))
    b.status()
    assert a.pages() == b.pages()
    for i in range(n):
        x, y = (c.read(0, int(times[i]), int(streams[i])) for c in (a, b))
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])


@pytest.mark.parametrize("bad", [0, 5, 7])
def test_append_stops_at_the_first_invalid_item(ctx, bad):
    kv = ctx.kv_cache(1, 2, 64, 4, 32, 4)
    streams, times = np.arange(8, dtype=np.int32) % 4, np.arange(8, dtype=np.int32) * 3
    times[bad] = 32
    rows = np.ones((8, 128), np.float32)
    with pytest.raises(hip.InvalidArgument):
        kv.append(0, streams, times, rows, rows)
    for i in range(8):
        got = kv.read(0, int(times[i]), int(streams[i])) if i != bad else None
        # (Q8_0 keeps 1.0 to fp16 of its scale; a row that was not stored may lie in a stored one's page, zero)
        assert (got is not None and abs(got[0][0] - 1.0) < 1e-3) if i < bad else (got is None or not np.any(got[0]))
    assert kv.pages()[1] == len({int(t) // 4 for t in times[:bad]})


@pytest.mark.parametrize("hq,bs,lens", [(16, 16, [1, 31, 512, 513, 700]), (4, 12, [33, 129, 385, 1500]),
                                        (8, 5, [127, 4095, 4097])])
def test_gqa_operand_split_against_float64(ctx, hq, bs, lens):
    """Every head within the split's own error: a head whose two fp16 halves
    disagree is off by more than ten times as much."""
    print(f"[case] gqa {hq} heads, pages of {bs}, lens {lens}", flush=True)
    H, hd, n = 2, 128, len(lens)
    g = np.random.default_rng(hq + bs)
    kv = ctx.kv_cache(1, H, hd, n, max(lens), bs)
    items = [(s, t) for s, ln in enumerate(lens) for t in range(ln)]
    rows = g.standard_normal((2, len(items), H * hd)).astype(np.float32)
    for i in range(0, len(items), 1024):
        st, tm = (np.array([x[j] for x in items[i:i + 1024]], np.int32) for j in (0, 1))
        kv.append(0, st, tm, rows[0, i:i + 1024], rows[1, i:i + 1024])
    for rep in range(4):  # 4 x n x hq heads
        q = g.standard_normal((n, hq * hd)).astype(np.float32)
        out = kv.attn(0, np.arange(n), lens, q, hq, hd ** -0.5)
        scale = np.float32(hd ** -0.5)
        for s, ln in enumerate(lens):
            cached = [kv.read(0, t, s) for t in range(ln)] if rep == 0 else cache[s]
            if rep == 0:
                cache = {} if s == 0 else cache
                cache[s] = cached
            K, V = (np.stack([c[j] for c in cached]).astype(np.float64).reshape(ln, H, hd) for j in (0, 1))
            for h in range(hq):
                qs = (q[s, h * hd:(h + 1) * hd] * scale).astype(np.float64)
                sc = K[:, h // (hq // H)] @ qs
                p = np.exp(sc - sc.max())
                want = p @ V[:, h // (hq // H)] / p.sum()
                # scores to 2^-20 of their magnitude (exp doubles as relative error of p), p d_v to 2^-21
                tol = (2.0 ** -20 * np.abs(K[:, h // (hq // H)] * qs).sum(1).max() + 2.0 ** -20) * np.abs(V).max()
                assert np.abs(out[s].reshape(hq, hd)[h] - want).max() <= tol, (rep, s, h)


def test_step_allocates_more_items_than_threads(ctx, oracle):
    """40 layers x 60 streams in one allocation: the same logits and pages as the
    two halves of the batch stepped one after the other."""
    g = np.random.default_rng(11)
    n_layer, d, ff, V, n = 40, 128, 128, 64, 60
    layers = make_layers(oracle, g, n_layer, d, 1, 1, 128, ff, wd=8)
    tok = g.standard_normal((V, d)).astype(np.float32)
    a, b = (hip.TextDecoder(ctx, 8, d, 1, 1, 128, ff, V, 64, n, layers, tok, np.ones(d, np.float32), None, block_size=4)
            for _ in range(2))
    st, h = np.arange(n, dtype=np.int32), n // 2
    for _ in range(6):
        toks = g.integers(0, V, n).astype(np.int32)
        got = a.step(st, toks, True)
        lo, hi = b.step(st[:h], toks[:h], True), b.step(st[h:], toks[h:], True)
        for x, y, z in zip(got, lo, hi):
            assert np.array_equal(x, np.concatenate([y, z]))
    assert a.kv_pages() == b.kv_pages() and a.kv_pages()[1] == n_layer * 2
