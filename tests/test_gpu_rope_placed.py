"""Rotary embedding and append where the rows are dealt to XCDs by head: one and two XCDs to a kv head, one to a list of several, odd
token counts, both sides of the bounds in tokens and bytes, a cache that is not empty.  Bit for bit against the oracle, every
row once and nothing beside them."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, f32_dev, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,is_neox", [(DT_FLOAT16, False), (DT_BFLOAT16, True)])
@pytest.mark.parametrize("m,pos,H,Hkv", [(63, 0, 8, 8), (64, 0, 8, 8), (64, 63, 28, 4), (65, 0, 28, 4), (67, 66, 4, 4), (64, 64, 12, 4),
                                         (131, 0, 40, 8), (70, 3, 32, 32), (71, 0, 16, 16), (277, 0, 32, 32), (278, 0, 32, 32),
                                         (739, 0, 28, 4), (739, 0, 29, 4), (100, 0, 12, 2), (100, 0, 7, 1)])
def test_placed(dt, is_neox, m, pos, H, Hkv):
    import llm_simple_amd.ops as ops
    rows = pos + m + 1
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
