"""The grouped-head decode attention's bits at pinned inputs. INT8 activations
follow it in every session, so a last-bit change here comes out as whole
quantization steps behind it: a history decoded on has to give the same logits
from one version of the kernel to the next."""
import zlib

import numpy as np
import pytest

from vokra_amd import hip

pytestmark = pytest.mark.gpu

# (query heads, kv heads, page size, keys) -> CRC-32 of the outputs' bytes on gfx950
BITS = {(16, 2, 16, (1, 31, 512, 513, 1100)): 1000241532,
        (32, 8, 16, (129, 700)): 3947231547,
        (8, 4, 5, (33, 4097)): 1264147713}


def attend(ctx, hq, H, bs, lens):
    hd, n = 128, len(lens)
    g = np.random.default_rng(hq + bs)
    kv = ctx.kv_cache(1, H, hd, n, max(lens), bs)
    items = [(s, t) for s, ln in enumerate(lens) for t in range(ln)]
    rows = g.integers(-4000, 4001, (2, len(items), H * hd)).astype(np.float32) * np.float32(2 ** -11)
    for i in range(0, len(items), 1024):
        st, tm = (np.array([x[j] for x in items[i:i + 1024]], np.int32) for j in (0, 1))
        kv.append(0, st, tm, rows[0, i:i + 1024], rows[1, i:i + 1024])
    q = g.integers(-4000, 4001, (n, hq * hd)).astype(np.float32) * np.float32(2 ** -10 * 1.3)
    return kv.attn(0, np.arange(n), lens, q, hq, hd ** -0.5)


@pytest.mark.parametrize("hq,H,bs,lens", [(16, 2, 16, (1, 31, 512, 513, 1100)), (32, 8, 16, (129, 700)),
                                          (8, 4, 5, (33, 4097))])
def test_bits_of_grouped_decode_attention(hq, H, bs, lens):
    print(f"[case] gqa bits {hq}/{H}, pages of {bs}, lens {lens}", flush=True)
    ctx = hip.HipContext(0)
    out = attend(ctx, hq, H, bs, lens)
    ctx.close()
    assert zlib.crc32(np.ascontiguousarray(out, np.float32).tobytes()) == BITS[(hq, H, bs, lens)]
