"""GPU parity of the block GEMM on launches of few output tiles
(vk_gemm_qblock_deep) and of the Q5_0 decode route: bit-exact against the oracle
at the edges of their tiles, stages and routes."""
import numpy as np
import pytest

from tests.test_gpu_quant import _gemm_case, bits
from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


# 32 x 32 tiles (four blocks a stage): one block, a stage and one more, k off
# the stage; row and column remainders of one. 64 x 64 tiles (two blocks a
# stage; k >= 3072 and over 3200 tiles of 16 x 16): an odd block count.
@pytest.mark.parametrize("act", [hip.ActQuant.AMAX127, hip.ActQuant.POW2])
@pytest.mark.parametrize("m,n,k", [(65, 16, 32), (97, 33, 160), (66, 129, 96), (513, 128, 256), (187, 81, 5152),
                                   (705, 1201, 3104), (1030, 800, 3072)])
def test_small_grids_bit_exact(ctx, oracle, act, m, n, k):
    print(f"[case] block GEMM small grid act={act.name} m={m} n={n} k={k}", flush=True)
    a, wq, bias = _gemm_case(oracle, hip.WDtype.Q8_0, m, n, k, seed=m + n + k, with_bias=m % 2 == 1, zero_rows=(0,))
    ctx.set_act_quant(act)
    try:
        got = ctx.gemm_q_f32(m, n, k, a, wq, hip.WDtype.Q8_0, bias)
    finally:
        ctx.set_act_quant(hip.ActQuant.AMAX127)
    rows = np.r_[0:17, m - 17:m]
    want = oracle.gemm_qblock_i8(8, rows.size, n, k, a[rows], wq, bias, pow2=act == hip.ActQuant.POW2)
    assert np.array_equal(bits(got[rows]), bits(want))
    cols = np.r_[0:5, n - 5:n]
    wc = wq.reshape(n, -1)[cols].reshape(-1)
    want = oracle.gemm_qblock_i8(8, m, cols.size, k, a, wc, None if bias is None else bias[cols],
                                 pow2=act == hip.ActQuant.POW2)
    assert np.array_equal(bits(np.ascontiguousarray(got[:, cols])), bits(want))


@pytest.mark.parametrize("act", [hip.ActQuant.AMAX127, hip.ActQuant.POW2])
@pytest.mark.parametrize("m,n,k", [(1, 40, 128), (17, 33, 640), (64, 5120, 128), (64, 16, 1664)])
def test_q5_0_decode_bit_exact(ctx, oracle, act, m, n, k):
    """Q5_0 rows up to 64 on the decode kernels, both of them (from 512 tiles
    a wave takes a tile), and equal to the block GEMM."""
    print(f"[case] q5_0 decode act={act.name} m={m} n={n} k={k}", flush=True)
    a, wq, bias = _gemm_case(oracle, hip.WDtype.Q5_0, m, n, k, seed=m + n + k)
    ctx.set_act_quant(act)
    try:
        got = ctx.gemm_q_f32(m, n, k, a, wq, hip.WDtype.Q5_0, bias)
        ctx.set_decode_kernel(False)
        gemm = ctx.gemm_q_f32(m, n, k, a, wq, hip.WDtype.Q5_0, bias)
    finally:
        ctx.set_decode_kernel(True)
        ctx.set_act_quant(hip.ActQuant.AMAX127)
    want = oracle.gemm_qblock_i8(6, m, n, k, a, wq, bias, pow2=act == hip.ActQuant.POW2)
    assert np.array_equal(bits(got), bits(want))
    assert np.array_equal(bits(gemm), bits(want))


def test_q5_0_linear_group_stays_refused(ctx, oracle):
    """A linear group takes Q4_0 and Q8_0 weights only."""
    _, wq, _ = _gemm_case(oracle, hip.WDtype.Q5_0, 1, 16, 128, seed=1)
    w = ctx.upload_qweight(hip.WDtype.Q5_0, 16, 128, wq)
    with pytest.raises(hip.UnsupportedOp):
        hip.LinearGroup(ctx, [w], [hip.DeviceBuffer(ctx, 64)])
