"""Rotary embedding and append at the edges of the launch: fewer threads than a workgroup, exactly one and two, one row more.
Bit for bit against the oracle; nothing outside the rows is touched, and q and k may be rotated where they lie."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("is_neox", [False, True])
@pytest.mark.parametrize("m,H,Hkv", [(1, 1, 1), (2, 12, 2), (4, 12, 2), (3, 9, 1), (1, 31, 1), (11, 5, 5)])
def test_rows(dt, is_neox, m, H, Hkv):
    import llm_simple_amd.ops as ops
    pos, rows = 7, m + 16
    table = orc.init_freq_cis(128, pos + m, 1e4, dt)
    q, k, v = (normal_bits(i, (m, h, 128), dt) for i, h in ((1, H), (2, Hkv), (3, Hkv)))
    want_q = np.full((m + 1, H, 128), 0xBEEF, dtype=np.uint16)
    want_k, want_v = (np.full((rows, Hkv, 128), 0xCAFE, dtype=np.uint16) for _ in range(2))
    d_q, d_k, d_v = to_dev(want_q), to_dev(want_k), to_dev(want_v)
    want_q[:m] = orc.rope(q, table, pos, is_neox, dt)
    orc.kv_append(want_k, orc.rope(k, table, pos, is_neox, dt), pos)
    orc.kv_append(want_v, v, pos)
    ops.hip_rope_kv_append_layer(d_q, d_k, d_v, f32_dev(table), to_dev(q), to_dev(k), to_dev(v), pos, m, H, Hkv, 128, is_neox, dt)
    for got, want in ((d_q, want_q), (d_k, want_k), (d_v, want_v)):
        assert np.array_equal(to_host(got), want)
    d_q = to_dev(q)
    ops.hip_rope_single_layer(d_q, f32_dev(table), d_q, pos, m, H, H * 128, is_neox, dt)
    assert np.array_equal(to_host(d_q), want_q[:m])
