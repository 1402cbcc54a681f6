"""Workgroup shapes of the prefill kernel at the edges of their ranges: prompts and chunks whose last tile leaves whole
waves without rows, tiles of 64 and 128 keys with a ragged end, packed heads, cut key ranges.  Every call is repeated: a
tile load that overtakes a reader shows as a result that changes from call to call."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (m, past, H, Hkv)
CASES = [
    (17, 0, 12, 2), (33, 0, 28, 4), (96, 0, 28, 4),          # two waves per 64 rows
    (97, 0, 28, 4), (129, 0, 12, 2), (257, 0, 12, 2),        # four waves per 32 rows
    (481, 0, 28, 4), (705, 0, 12, 2),                        # four waves per 64 rows
    (600, 0, 40, 8), (650, 0, 40, 8), (1100, 0, 40, 8),      # two waves per 64, per 128 rows
    (1700, 0, 40, 8), (1801, 0, 40, 8), (1281, 0, 64, 2),    # 128 rows of one wave each, twice; 256 rows
    (3, 300, 28, 4), (9, 4000, 40, 8), (20, 1500, 32, 32), (65, 2000, 12, 2), (130, 3001, 28, 4), (150, 151, 12, 2),
    (300, 300, 40, 8), (300, 2500, 28, 4), (2, 10000, 64, 2), (1, 3000, 20, 1),
]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", CASES)
def test_shapes(dt, m, past, H, Hkv):
    import llm_simple_amd.ops as ops
    n = m + past
    q = normal_bits(m, (m, H, 128), dt)
    k = normal_bits(n + 1, (n, Hkv, 128), dt)
    v = normal_bits(n + 2, (n, Hkv, 128), dt)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    outs = [dev_empty(q.shape) for _ in range(16)]
    for o in outs:
        ops.hip_flash_attn_gqa_layer(o, dq, dk, dv, m, n, past, H // Hkv, Hkv, 128, dt)
    got = to_host(outs[0])
    check_attention(got, q, k, v, n, past, dt)
    for o in outs[1:]:
        assert np.array_equal(to_host(o), got)
