"""Rotary embedding and append with outputs that begin anywhere a call may put them, 16 bytes apart: on a 128-byte line, on a
64-byte sector and off it, on both sides of the size from which the stores differ.  Bit for bit against the oracle, nothing beside
the rows; and such a base may not cost a large call half as much again (4096 tokens of 28 + 2 x 4 heads: 1.08 times the time of whole
lines where the halves of a shared sector meet in the L2, 1.49 where each is written to memory by itself)."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, f32_dev, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _off(buf, elements):
    """The address `elements` storage elements (2 bytes each) into a buffer."""
    return buf.data_ptr() + 2 * elements


@pytest.mark.parametrize("off_q,off_k,off_v", [(8, 8, 8), (16, 0, 0), (0, 24, 0), (0, 0, 8), (32, 32, 32), (64, 0, 96)])
@pytest.mark.parametrize("dt,is_neox,m,pos,H,Hkv", [(DT_FLOAT16, False, 131, 0, 8, 8), (DT_BFLOAT16, True, 77, 100, 12, 2),
                                                    (DT_FLOAT16, True, 470, 3, 32, 32), (DT_BFLOAT16, False, 1409, 0, 33, 33)])
def test_bases(dt, is_neox, m, pos, H, Hkv, off_q, off_k, off_v):
    import llm_simple_amd.ops as ops
    table = orc.init_freq_cis(128, pos + m, 1e4, dt)
    q, k, v = (normal_bits(i, (m, h, 128), dt) for i, h in ((1, H), (2, Hkv), (3, Hkv)))
    guard = 256
    want = [np.full(guard + rows * h * 128 + guard, 0xCAFE, dtype=np.uint16) for rows, h in ((m, H), (pos + m, Hkv), (pos + m, Hkv))]
    dev = [to_dev(w) for w in want]
    for w, off, first, rows in ((want[0], off_q, 0, orc.rope(q, table, pos, is_neox, dt)),
                                (want[1], off_k, pos * Hkv * 128, orc.rope(k, table, pos, is_neox, dt)), (want[2], off_v, pos * Hkv * 128, v)):
        w[off + first:off + first + rows.size] = rows.reshape(-1)
    ops.hip_rope_kv_append_layer(_off(dev[0], off_q), _off(dev[1], off_k), _off(dev[2], off_v), f32_dev(table), to_dev(q), to_dev(k),
                                 to_dev(v), pos, m, H, Hkv, 128, is_neox, dt)
    for got, w in zip(dev, want):
        assert np.array_equal(to_host(got), w)


def test_a_base_off_the_sector_is_not_half_as_slow_again():
    import torch
    import llm_simple_amd.ops as ops
    m, H, Hkv = 4096, 28, 4
    table = torch.zeros(m, 128, device="cuda")
    q, k, v = (torch.zeros(m * h * 128 + 128, dtype=torch.int16, device="cuda") for h in (H, Hkv, Hkv))
    out = [torch.empty_like(x) for x in (q, k, v)]
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

    def batch_ms(off):
        start.record()
        for _ in range(50):
            ops.hip_rope_kv_append_layer(*(_off(x, off) for x in out), table, q, k, v, 0, m, H, Hkv, 128, True, DT_BFLOAT16)
        end.record()
        end.synchronize()
        return start.elapsed_time(end)

    times = [(batch_ms(0), batch_ms(8)) for _ in range(12)][2:]
    on_line, off_sector = (min(t) for t in zip(*times))
    assert off_sector < 1.35 * on_line
