"""GPU parity of the tiled K-quant matmul (launches of 1800 and more 16 x 16
output tiles): bit-exact against the oracle at the edges of its tiles, like the
kernel that runs smaller launches, and one grid over three linears equal to
each linear by itself."""
import numpy as np
import pytest

from tests.helpers import Rng, random_kquant_blocks
from tests.test_gpu_sessions import enc_layer, encoder_by_ops, rand_norm
from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


# one row tile (four column waves) and several (2 x 2 waves), with an odd last
# row tile; one and two column tiles per wave (from 3500 tiles), column counts
# off the workgroup's width and off 16; one super-block and an odd number
@pytest.mark.parametrize("wd", [12, 13, 14])
@pytest.mark.parametrize("m,n,k", [(1, 28807, 256), (16, 56017, 256), (33, 9617, 256), (40, 9601, 768),
                                   (1500, 310, 512), (600, 1503, 256)])
def test_tiled_bit_exact(ctx, oracle, wd, m, n, k):
    print(f"[case] k-quant tiled wd={wd} m={m} n={n} k={k}", flush=True)
    g = np.random.default_rng(m + n + k)
    a = g.standard_normal((m, k)).astype(np.float32)
    a[0, :16] = 0.0
    w = random_kquant_blocks(Rng(m + 7 * n), n * (k // 256), wd)
    bias = g.standard_normal(n).astype(np.float32) if m % 2 else None
    got = ctx.gemm_q_f32(m, n, k, a, w, hip.WDtype(wd), bias=bias)
    # the oracle on the first, middle and last rows and on every column
    rows = sorted({0, 1, m // 2, m - 2, m - 1} & set(range(m)))
    want = oracle.gemm_q_f32(wd, len(rows), n, k, a[rows], w, bias)
    assert np.array_equal(got[rows].view(np.uint32), want.view(np.uint32))
    # and every row, on the first and last columns
    cols = np.r_[0:20, n - 20:n]
    wc = w.reshape(n, -1)[cols].reshape(-1)
    want = oracle.gemm_q_f32(wd, m, cols.size, k, a, wc, None if bias is None else bias[cols])
    assert np.array_equal(np.ascontiguousarray(got[:, cols]).view(np.uint32), want.view(np.uint32))


def test_three_linears_in_one_tiled_grid(ctx):
    """q, k and v of an encoder block in one grid (1872 tiles), each smaller
    alone: equal to the entry points one at a time, bit for bit."""
    g = np.random.default_rng(8)
    d, H, ff, T = 256, 4, 512, 620
    L = enc_layer(ctx, g, 12, d, ff)
    lpg, lpb = rand_norm(g, d)
    x = g.standard_normal((1, T, d)).astype(np.float32)
    enc = hip.Encoder(ctx, 12, d, H, ff, [L], lpg, lpb, T)
    assert np.array_equal(enc.forward(x), encoder_by_ops(ctx, 12, [L], lpg, lpb, x, H, ff))
