"""The tied-logits kernel of large vocabularies (three bf16 parts per operand) against
float64, at the edges of its tiles and of the operands' range."""
import numpy as np
import pytest

from tests.test_gpu_f32 import dot_bound, fused_logits
from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


# the smallest such vocabulary and one row less; 64- and 128-row workgroups with one
# row left; every number of column tiles, and more streams than a workgroup holds;
# row distances whose workgroups start along k (4 KiB multiples)
@pytest.mark.parametrize("n,v,d", [(3, 30719, 128), (3, 30720, 128), (16, 30785, 256), (17, 32769, 128), (33, 49153, 128),
                                   (64, 49153, 384), (65, 30721, 128), (33, 30721, 1024), (2, 30720, 2048)])
def test_wide_logits(ctx, oracle, n, v, d):
    print(f"[case] wide logits n={n} v={v} d={d}", flush=True)
    g = np.random.default_rng(n + v + d)
    x = g.standard_normal((n, d)).astype(np.float32)
    e = (g.standard_normal((v, d)) * 0.05).astype(np.float32)
    e[11], e[v - 2] = np.float32(3e38) * np.sign(x[0]), 1e-30 * e[12]  # an overflow, and tiny terms
    e[13, 5], e[14, 6], e[15, 7] = np.inf, -np.inf, np.nan
    x[-1, 9], e[16, 9] = 3.4e38, 1e-38  # rounds to an infinite bf16; the product is finite
    logits, nxt = fused_logits(ctx, x, e)
    with np.errstate(all="ignore"):
        exact = x.astype(np.float64) @ e.astype(np.float64).T
        bound = dot_bound(x, e.T, d)
        fits = np.abs(exact) + bound < 3.4e38  # (false for what is not finite)
        fits[1:, 11] = False  # terms of both signs near the largest float: partial sums overflow in any order
        assert np.all(np.abs(logits - exact)[fits] <= bound[fits] + d * 2.0 ** -126)
    assert not np.isfinite(logits[0, 11])
    assert np.isnan(logits[:, 15]).all()
    assert nxt.tolist() == [oracle.argmax(r) for r in logits]
    _, nxt2 = fused_logits(ctx, x, e, write=False)
    assert np.array_equal(nxt, nxt2)
    for rows in ([0], list(range(min(n, 20)))):  # a stream's logits do not depend on its batch
        part, _ = fused_logits(ctx, np.ascontiguousarray(x[rows]), e)
        assert np.array_equal(part.view(np.uint32), logits[rows].view(np.uint32))
