"""The few-row projection kernel over a k of several passes: both sides of the lines between eight and four units a pass (lhs rows
times W rows per workgroup, 256 compute units; 13, 14, 16 and 17 units), and of 12 units, where the passes begin.  Against the oracle,
within a step of the storage type."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k", [(8, 2048, 6144), (1, 2048, 6160), (4, 1280, 6672), (7, 768, 6672), (6, 1024, 7168), (8, 1024, 8192),
                                   (5, 1792, 8192), (8, 1024, 8208), (3, 1776, 8960), (8, 2048, 13824), (2, 48, 13824), (8, 16, 18944)])
def test_passes(dt, m, n, k):
    import llm_simple_amd.ops as ops
    x = normal_bits(m + k, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ref = orc.widen(orc.matmul_bias(x, w, b, dt), dt)
    out = dev_empty((m, n))
    ops.hip_matmul_bias_layer(out, to_dev(x), to_dev(w), f32_dev(b), m, n, k, dt)
    got = orc.widen(to_host(out), dt)
    assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
