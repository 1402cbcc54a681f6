"""The order in which tiles of the same W rows take the lines of k: two, three, four and more tiles to a band, groups of 8, 4, 2 and 1
lines, a last tile that is padding by less and by more than a quarter, and the tiles of 32 x 64 and 64 x 96.  Against sums in 64 bits."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n", [(30, 2064), (40, 2064), (64, 1040), (64, 5120), (121, 3584), (128, 3584), (120, 3584), (57, 8192),
                                 (190, 3072), (193, 3072), (1024, 1536), (300, 3584), (700, 2048)])
def test_turns(dt, m, n):
    import llm_simple_amd.ops as ops
    for lines in (1, 2, 3, 4, 7, 8, 10, 12, 16, 17):
        k = 64 * lines
        x = normal_bits(m + k, (m, k), dt)
        w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
        ref = orc.widen(x, dt).astype(np.float64) @ orc.widen(w, dt).T.astype(np.float64)
        ref = orc.widen(orc.round_to(ref.astype(np.float32), dt), dt)
        d_out = to_dev(np.full((m, n), 0x7e00 if dt == DT_FLOAT16 else 0x7fc0, dtype=np.uint16))  # NaN
        ops.hip_matmul_layer(d_out, to_dev(x), to_dev(w), m, n, k, dt)
        got = orc.widen(to_host(d_out), dt)
        # one rounding of an fp32 sum: a step of the storage type, 1e-3 where the sum cancels (a NaN fails the comparison)
        assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all(), lines
