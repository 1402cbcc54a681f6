"""The few-row projection kernel where a workgroup has at most 8 W rows: both sides of that line (256 compute units), and k on
both sides of 4, 8 and 12 units of 64 per wave, with a ragged last unit; k of whole units for every wave, one pass and several,
one W row and a ragged last share.  Against the oracle, within a step of the storage type."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k", [(1, 2048, 512), (8, 2064, 512), (3, 48, 2048), (1, 272, 2064), (8, 48, 4096), (1, 16, 4112),
                                   (2, 272, 6144), (7, 16, 6160), (8, 16, 1024), (1, 48, 3584), (5, 32, 6656), (1, 2576, 512),
                                   (8, 2320, 3584), (2, 2320, 5120), (1, 2320, 6656), (3, 4112, 2560)])
def test_units(dt, m, n, k):
    import llm_simple_amd.ops as ops
    x = normal_bits(m + k, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ref = orc.widen(orc.matmul_bias(x, w, b, dt), dt)
    out = dev_empty((m, n))
    ops.hip_matmul_bias_layer(out, to_dev(x), to_dev(w), f32_dev(b), m, n, k, dt)
    got = orc.widen(to_host(out), dt)
    assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
