"""The rows that are dealt to XCDs, without V (rope of q and k alone: a list is a third shorter) and, with V, in the pairing style
and storage type that test_gpu_rope_placed.py leaves out.  Bit for bit against the oracle, every row once and nothing beside them."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, f32_dev, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("is_neox", [False, True])
@pytest.mark.parametrize("m,pos,H", [(64, 0, 4), (65, 0, 4), (131, 130, 4), (64, 63, 8), (131, 0, 8), (64, 0, 32), (131, 7, 32), (415, 0, 32),
                                     (417, 0, 32), (63, 0, 8), (64, 64, 8), (100, 0, 2)])
def test_without_v(dt, is_neox, m, pos, H):
    import llm_simple_amd.ops as ops
    table = orc.init_freq_cis(128, pos + m, 1e4, dt)
    x = [normal_bits(i, (m, H, 128), dt) for i in (1, 2)]
    want = [np.full((m + 1, H, 128), 0xBEEF, dtype=np.uint16) for _ in x]
    dev = [to_dev(w) for w in want]
    for w, rows in zip(want, x):
        w[:m] = orc.rope(rows, table, pos, is_neox, dt)
    ops.hip_rope_layer(dev[0], dev[1], f32_dev(table), to_dev(x[0]), to_dev(x[1]), pos, m, H, H * 128, is_neox, dt)
    for got, w in zip(dev, want):
        assert np.array_equal(to_host(got), w)


@pytest.mark.parametrize("dt,is_neox", [(DT_FLOAT16, True), (DT_BFLOAT16, False)])
@pytest.mark.parametrize("m,pos,H,Hkv", [(64, 0, 8, 8), (65, 0, 28, 4), (131, 0, 40, 8), (277, 0, 32, 32)])
def test_with_v(dt, is_neox, m, pos, H, Hkv):
    import llm_simple_amd.ops as ops
    table = orc.init_freq_cis(128, pos + m, 1e4, dt)
    q, k, v = (normal_bits(i, (m, h, 128), dt) for i, h in ((1, H), (2, Hkv), (3, Hkv)))
    want_q = np.full((m + 1, H, 128), 0xBEEF, dtype=np.uint16)
    want_k, want_v = (np.full((pos + m + 1, Hkv, 128), 0xCAFE, dtype=np.uint16) for _ in range(2))
    d_q, d_k, d_v = to_dev(want_q), to_dev(want_k), to_dev(want_v)
    want_q[:m] = orc.rope(q, table, pos, is_neox, dt)
    orc.kv_append(want_k, orc.rope(k, table, pos, is_neox, dt), pos)
    orc.kv_append(want_v, v, pos)
    ops.hip_rope_kv_append_layer(d_q, d_k, d_v, f32_dev(table), to_dev(q), to_dev(k), to_dev(v), pos, m, H, Hkv, 128, is_neox, dt)
    for got, want in ((d_q, want_q), (d_k, want_k), (d_v, want_v)):
        assert np.array_equal(to_host(got), want)
