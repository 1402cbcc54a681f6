"""The few-row projection kernel (up to 16 lhs rows) against the oracle, at the edges of its tiles: one and all
operand columns, both layouts (up to 8 rows, 9 to 16), shares of W that are one row, a ragged last share and
two rounds of workgroups, k of less than one unit and with a ragged last unit, an unaligned base."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k,bias", [(1, 16, 16, True), (1, 5120, 5120, False), (8, 272, 1552, True),
                                        (9, 272, 1552, False), (16, 4112, 80, True), (7, 48, 48, False),
                                        (16, 528, 4096, True), (2, 4096, 11008, True)])
def test_few_rows(dt, m, n, k, bias):
    import torch
    import llm_simple_amd.ops as ops
    x = normal_bits(m + k, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32) if bias else None
    ref = orc.widen(orc.matmul_bias(x, w, b, dt), dt)
    for shift in (0, 1):  # a base that is not 16-byte aligned takes the other path
        d_x = torch.empty(m * k + 8, dtype=torch.int16, device="cuda")[shift:shift + m * k]
        d_x.copy_(to_dev(x).flatten())
        guard = torch.full((m * n + 16,), 0x55, dtype=torch.int16, device="cuda")
        args = (guard[8:8 + m * n], d_x, to_dev(w))
        if bias:
            ops.hip_matmul_bias_layer(*args, f32_dev(b), m, n, k, dt)
        else:
            ops.hip_matmul_layer(*args, m, n, k, dt)
        got = orc.widen(to_host(guard[8:8 + m * n]), dt).reshape(m, n)
        assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
        assert (guard[:8] == 0x55).all() and (guard[8 + m * n:] == 0x55).all()
