"""NaN and infinity through the projection kernels: a bias or an operand that holds one gives one, whatever its bits, in
the few-row kernel (up to 16 rows) as in the tiled one."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 100])
def test_nan_and_infinity(dt, m):
    import llm_simple_amd.ops as ops
    n, k = 272, 320
    x = orc.widen(normal_bits(m, (m, k), dt), dt)
    w = orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    # payloads that a rounding on the bit pattern carries out of the exponent, the smallest one, infinities, overflow
    b.view(np.uint32)[[3, 18, 100, 255]] = 0xFFFFFFFF, 0x7FFFFFFF, 0x7F800001, 0xFF80FFFF
    b[[5, 200, 271]] = np.inf, -np.inf, 3.4e38 if dt == DT_BFLOAT16 else 7e4
    w[40, 7] = np.nan
    if m > 1:
        x[m - 1, k - 1], x[m // 2, 0] = np.inf, np.nan
    xb, wb = orc.round_to(x.astype(np.float32), dt), orc.round_to(w.astype(np.float32), dt)
    with np.errstate(invalid="ignore", over="ignore"):
        exact = orc.widen(xb, dt).astype(np.float64) @ orc.widen(wb, dt).astype(np.float64).T + b
    out = dev_empty((m, n))
    ops.hip_matmul_bias_layer(out, to_dev(xb), to_dev(wb), f32_dev(b), m, n, k, dt)
    got = orc.widen(to_host(out), dt)
    nan = np.isnan(exact)
    assert np.array_equal(np.isnan(got), nan)
    largest = 3.3895e38 if dt == DT_BFLOAT16 else 65504.0
    inf = ~nan & (np.abs(exact) > largest)
    assert np.array_equal(got[inf], np.copysign(np.inf, exact[inf]))
    rest = ~nan & ~inf
    # the tolerance of the other projection tests: one step of the storage type, 1e-3 where the sum cancels
    assert (np.abs(got[rest] - exact[rest]) <= np.maximum(1.01 * ulp(exact[rest], dt), 1e-3)).all()
