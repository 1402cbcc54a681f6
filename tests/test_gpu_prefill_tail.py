"""Rows past the end of a key range read as zero by the tile loads' descriptors: every workgroup shape with a last tile of one,
all but one and all of its keys, one kv head (rows next to each other) and several, ranges cut by the cache's end and by the
last visible key; the rows behind them hold NaN, and so does whatever lies in front of the cache."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (m, past, H, Hkv): 32 rows x 4 waves, 64 x 4, 64 x 2 (two workgroups to a CU: 705 tokens; heads in one list: 1300), 128 x 2,
# 128 and 256 rows, chunks (cut, packed, whole)
CASES = [(129, 0, 12, 1), (191, 0, 12, 2), (513, 0, 28, 4), (575, 0, 14, 1), (640, 0, 40, 8), (705, 0, 40, 8), (1089, 0, 40, 8),
         (1151, 0, 32, 32), (1300, 0, 20, 5), (1665, 0, 40, 8), (1983, 0, 40, 8), (2049, 0, 28, 1), (3, 254, 28, 1), (40, 961, 16, 1), (40, 1047, 28, 4),
         (2, 4095, 28, 4), (255, 1730, 28, 4)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", CASES)
def test_tail(dt, m, past, H, Hkv):
    import llm_simple_amd.ops as ops
    n, pad = m + past, 160
    q = normal_bits(m, (m, H, 128), dt)
    nan = 0x7e00 if dt == DT_FLOAT16 else 0x7fc0
    caches = []
    for seed in (1, 2):
        a = np.full((pad + n + pad, Hkv, 128), nan, dtype=np.uint16)
        a[pad:pad + n] = normal_bits(n + seed, (n, Hkv, 128), dt)
        caches.append(a)
    d_k, d_v = (to_dev(a)[pad:] for a in caches)
    d_q, out = to_dev(q), dev_empty(q.shape)
    k, v = (np.ascontiguousarray(a[pad:pad + n]) for a in caches)
    for rows in sorted({n, n - m // 3}):  # the cache may end before the last row's position
        ops.hip_flash_attn_gqa_layer(out, d_q, d_k, d_v, m, rows, past, H // Hkv, Hkv, 128, dt)
        check_attention(to_host(out), q, k[:rows], v[:rows], rows, past, dt)
