"""9 to 16 lhs rows against a wide weight go to the tiled kernel (more than 4096 rows on 256 compute units): 8 and 9 rows,
both kernels, and k in part stages (which the tiles do not take), against the oracle."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k,bias", [(8, 4112, 64, True), (9, 4112, 64, True), (9, 4096, 192, False), (16, 5120, 320, True),
                                        (12, 8208, 128, False), (16, 4112, 80, True), (13, 16400, 64, True)])
def test_few_rows_wide_weight(dt, m, n, k, bias):
    import torch
    import llm_simple_amd.ops as ops
    x = normal_bits(m + k, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32) if bias else None
    ref = orc.widen(orc.matmul_bias(x, w, b, dt), dt)
    guard = torch.full((m * n + 16,), 0x55, dtype=torch.int16, device="cuda")
    args = (guard[8:8 + m * n], to_dev(x), to_dev(w))
    if bias:
        ops.hip_matmul_bias_layer(*args, f32_dev(b), m, n, k, dt)
    else:
        ops.hip_matmul_layer(*args, m, n, k, dt)
    got = orc.widen(to_host(guard[8:8 + m * n]), dt).reshape(m, n)
    # the tolerance of the other projection tests: one step of the storage type, 1e-3 where the sum cancels
    assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
    assert (guard[:8] == 0x55).all() and (guard[8 + m * n:] == 0x55).all()
