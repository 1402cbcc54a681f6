"""Prompts whose longest rows two workgroups share: head counts that are dealt to XCDs and not, a ragged last tile, tokens cached before,
keys past those that are seen, one and several cut tiles, and the sizes on either side.  Against the oracle on rows of every tile; every call gives
the same bits, with decode calls between that use the same buffer, and under capture, where no rows are shared, the same within the tolerance."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, TOL, dev_empty, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", [(896, 0, 28, 4), (897, 0, 28, 4), (1019, 0, 28, 4), (1088, 0, 28, 4), (1089, 0, 28, 4), (577, 400, 28, 4),
                                          (640, 639, 28, 4), (930, 0, 32, 32), (961, 0, 32, 32), (1480, 0, 12, 2), (950, 31, 30, 6), (1408, 0, 20, 1)])
def test_halves(dt, m, past, H, Hkv):
    import torch
    import llm_simple_amd.ops as ops
    n, g = m + past, H // Hkv
    q, k, v = normal_bits(m, (m, H, 128), dt), normal_bits(n + 1, (n + 64, Hkv, 128), dt), normal_bits(n + 2, (n + 64, Hkv, 128), dt)
    k[n:], v[n:] = 0x7FFF, 0x7FFF  # (not to be read)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    one = dev_empty((1, H, 128))

    def call(out, stream=None):
        ops.hip_flash_attn_gqa_layer(out, dq, dk, dv, m, n, past, g, Hkv, 128, dt, *([] if stream is None else [stream]))

    outs = [dev_empty(q.shape).fill_(0x7FFF) for _ in range(12)]
    for o in outs:
        call(o)
        ops.hip_flash_attn_gqa_layer(one, dq, dk, dv, 1, n, n - 1, g, Hkv, 128, dt)
    got = to_host(outs[0])
    wide = orc.widen(got, dt)
    assert np.isfinite(wide).all()
    rows = np.unique(np.r_[0:m:61, m - 70:m:3, m - 1])
    for r in rows:
        want = orc.attention_f32(q[r:r + 1], k, v, r + 1 + past, r + past, dt)
        assert np.abs(wide[r:r + 1] - want).max() <= TOL[dt], r
    for o in outs[1:]:
        assert np.array_equal(to_host(o), got)
    graph, o = torch.cuda.CUDAGraph(), dev_empty(q.shape)
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        call(o, torch.cuda.current_stream().cuda_stream)
    for _ in range(2):
        o.fill_(0x7FFF)
        graph.replay()
        torch.cuda.synchronize()
        # one rounding of the probabilities and one of the result apart
        assert np.linalg.norm(orc.widen(to_host(o), dt) - wide) <= (4e-3 if dt == DT_BFLOAT16 else 5e-4) * np.linalg.norm(wide)


def test_halves_on_two_streams():
    """Launches of two streams, each with a buffer of its own, that hold each other's workgroups up."""
    import torch
    import llm_simple_amd.ops as ops
    m, H, Hkv, dt = 1019, 28, 4, DT_BFLOAT16
    dq, dk, dv = (to_dev(normal_bits(s, (m, h, 128), dt)) for s, h in ((1, H), (2, Hkv), (3, Hkv)))
    want = dev_empty((m, H, 128))
    ops.hip_flash_attn_gqa_layer(want, dq, dk, dv, m, m, 0, H // Hkv, Hkv, 128, dt)
    streams, outs = [torch.cuda.Stream() for _ in range(2)], [[dev_empty((m, H, 128)) for _ in range(20)] for _ in range(2)]
    torch.cuda.synchronize()
    for i in range(20):
        for s, o in zip(streams, outs):
            ops.hip_flash_attn_gqa_layer(o[i], dq, dk, dv, m, m, 0, H // Hkv, Hkv, 128, dt, s.cuda_stream)
    torch.cuda.synchronize()
    for o in outs[0] + outs[1]:
        assert torch.equal(o, want)
