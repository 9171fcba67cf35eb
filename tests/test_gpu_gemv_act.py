"""The decode linear that quantizes its f32 rows itself: bit-exact against the
oracle, and against the separate activation pass, at the edges of its rule."""
import numpy as np
import pytest

from tests.test_gpu_quant import _gemm_case, bits
from vokra_amd import hip

pytestmark = pytest.mark.gpu
FORMATS = [hip.WDtype.Q4_0, hip.WDtype.Q5_0, hip.WDtype.Q8_0]


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


# one block group, a part of a chunk, a chunk and more, the most a workgroup holds
# and one group beyond it; rows over one tile; 511 and 512 tiles
@pytest.mark.parametrize("act", [hip.ActQuant.AMAX127, hip.ActQuant.POW2])
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(1, 17, 128), (1, 40, 1664), (1, 16, 6144), (1, 16, 6272), (3, 33, 1280), (16, 48, 384),
                                   (17, 40, 512), (64, 24, 384), (2, 8176, 128), (2, 8192, 128)])
def test_rows_quantized_in_the_linear(ctx, oracle, fmt, act, m, n, k):
    print(f"[case] gemv act {fmt.name} {act.name} m={m} n={n} k={k}", flush=True)
    a, wq, bias = _gemm_case(oracle, fmt, m, n, k, seed=m + n + k, zero_rows=(0,) if m > 2 else ())
    a = a.reshape(m, k)
    a[m - 1, 5] = np.nan
    if act == hip.ActQuant.AMAX127:
        a[m - 1, 40], a[0, 70] = np.inf, -np.inf
    w = hip.QWeight(ctx, fmt, n, k, wq)
    d_a, d_b = hip.DeviceBuffer.from_array(ctx, a), hip.DeviceBuffer.from_array(ctx, bias)
    d_o, d_s = hip.DeviceBuffer(ctx, m * n * 4), hip.DeviceBuffer(ctx, m * n * 4)
    ctx.gemm_q_f32_dev(w, m, d_a, d_o, d_b, act)
    qa = ctx.qact(m, k)
    qa.quantize(m, d_a, act)
    ctx.gemm_qact_dev(w, qa, d_s, d_b)
    got, sep = d_o.download(np.float32, m * n), d_s.download(np.float32, m * n)
    assert np.array_equal(bits(got), bits(sep))
    fin = np.isfinite(got.reshape(m, n)).all(1)
    want = oracle.gemm_qblock_i8(int(fmt), m, n, k, a, wq, bias, pow2=act == hip.ActQuant.POW2).reshape(m, n)
    assert np.array_equal(bits(got.reshape(m, n)[fin]), bits(np.ascontiguousarray(want[fin])))


def test_output_over_the_rows(ctx, oracle):
    """In place (n == k), and overlapping by part: as with rows of their own."""
    n = k = 256
    a, wq, bias = _gemm_case(oracle, hip.WDtype.Q4_0, 2, n, k, seed=5)
    w = hip.QWeight(ctx, hip.WDtype.Q4_0, n, k, wq)
    d_b = hip.DeviceBuffer.from_array(ctx, bias)
    want = oracle.gemm_qblock_i8(int(hip.WDtype.Q4_0), 2, n, k, a, wq, bias).reshape(2, n)
    for off in (0, 1024):  # bytes between the rows and the output
        buf = hip.DeviceBuffer.from_array(ctx, np.concatenate([np.ravel(a), np.zeros(1024, np.float32)]))

        class At:
            ptr = buf.ptr if off == 0 else type(buf.ptr)((buf.ptr if isinstance(buf.ptr, int) else buf.ptr.value) + off)
        ctx.gemm_q_f32_dev(w, 2, buf, At, d_b)
        got = buf.download(np.float32, 2 * n + 1024)[off // 4:off // 4 + 2 * n].reshape(2, n)
        assert np.array_equal(bits(got), bits(want))


def test_one_row_makes_room_for_a_capture_of_more(oracle):
    """A warm-up of one row, then a capture of eight, which take the activation pass of
    their own: nothing is left to allocate, and every replay equals the eager call."""
    ctx = hip.HipContext(0)
    m, n, k = 8, 64, 1280
    a, wq, bias = _gemm_case(oracle, hip.WDtype.Q4_0, m, n, k, seed=8)
    w = hip.QWeight(ctx, hip.WDtype.Q4_0, n, k, wq)
    d_a, d_b, d_o = hip.DeviceBuffer.from_array(ctx, a), hip.DeviceBuffer.from_array(ctx, bias), hip.DeviceBuffer(ctx, m * n * 4)
    ctx.gemm_q_f32_dev(w, 1, d_a, d_o, d_b)
    ctx.synchronize()
    graph = ctx.capture(lambda: ctx.gemm_q_f32_dev(w, m, d_a, d_o, d_b))
    want = np.ravel(oracle.gemm_qblock_i8(int(hip.WDtype.Q4_0), m, n, k, a, wq, bias))
    for _ in range(3):
        d_o.upload(np.zeros(m * n, np.float32))
        graph.launch()
        ctx.synchronize()
        assert np.array_equal(bits(d_o.download(np.float32, m * n)), bits(want))
    del graph
    ctx.close()
