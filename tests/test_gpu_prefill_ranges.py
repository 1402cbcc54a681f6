"""Key ranges of a chunk that go one tile wide through each other (8 kv heads or more) and ones that lie side by side: a last tile of
1, 63, 64, 65, 127 or 128 keys that belongs to the first, a middle or the last range, ranges of unequal numbers of tiles, rows whose last
visible key lies in another range than the next row's, packed and unpacked rows, tiles dealt to XCDs in clusters and one by one.  Behind the last key stands NaN, which no load may
bring in.  (Forms as planned for 256 compute units; that the call is cut at all is asserted.)"""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (m, past, H, Hkv)
CASES = [
    (20, 1900, 32, 32), (40, 4056, 32, 32), (64, 2000, 16, 16), (64, 2001, 16, 16), (64, 1999, 16, 16),  # unpacked, each head its own
    (30, 4130, 40, 8), (33, 8160, 40, 8), (17, 2095, 8, 8), (100, 3101, 40, 8), (200, 2176, 40, 8),       # at the rule's line
    (30, 4130, 35, 7), (33, 8160, 28, 4), (100, 3101, 28, 4), (130, 1999, 12, 2), (65, 3000, 9, 1),         # below it
    (14, 4000, 28, 4), (17, 5561, 12, 2), (62, 9001, 8, 1), (54, 3908, 24, 3), (96, 3930, 30, 6), (40, 2988, 36, 12),  # clusters of tiles (not the third: unpacked)
    (56, 9001, 7, 1), (110, 5000, 21, 3), (110, 5000, 35, 5), (120, 9001, 8, 1), (90, 5000, 35, 5),       # three clusters of them, two of five
    (64, 1983, 16, 16), (64, 2047, 16, 16), (100, 3035, 40, 8), (100, 3037, 40, 8), (100, 3099, 40, 8),  # last tiles of 127 and 63, of 63, 65 and 127 keys
    (130, 1981, 12, 2), (100, 3035, 28, 4), (100, 3037, 28, 4), (100, 3099, 28, 4),                        # of 63, of 63, 65 and 127, side by side
    (128, 1920, 64, 64), (256, 3000, 18, 9), (300, 4500, 40, 40),
]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", CASES)
def test_ranges(dt, m, past, H, Hkv):
    import llm_simple_amd.ops as ops
    n = m + past
    assert ops.lib.llmhip_flash_attn_scratch_bytes(m, n, past, H // Hkv, Hkv) >= 2 * m * H * 130 * 4  # (it is cut)
    q = normal_bits(m, (m, H, 128), dt)
    k, v = normal_bits(n + 1, (n, Hkv, 128), dt), normal_bits(n + 2, (n, Hkv, 128), dt)
    behind = np.full((256, Hkv, 128), 0x7FFF, dtype=k.dtype)
    dq, dk, dv = to_dev(q), to_dev(np.concatenate([k, behind])), to_dev(np.concatenate([v, behind]))
    outs = [dev_empty(q.shape) for _ in range(4)]
    for o in outs:
        ops.hip_flash_attn_gqa_layer(o, dq, dk, dv, m, n, past, H // Hkv, Hkv, 128, dt)
    got = to_host(outs[0])
    check_attention(got, q, k, v, n, past, dt)
    for o in outs[1:]:
        assert np.array_equal(to_host(o), got)
