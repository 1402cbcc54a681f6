"""Prompts whose longest rows two workgroups share: head counts that are dealt to XCDs and not, a ragged last tile, tokens cached before,
keys past those that are seen, one and several cut tiles, and the sizes on either side.  Against the oracle on rows of every tile; every call gives
the same bits, with projections between that use the same buffer, and under capture, where no rows are shared, the same within the tolerance.  Workgroups that do not wait for
the other half give what the captured call gives."""
import ctypes

import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, TOL, dev_empty, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


SHARED = [(896, 0, 28, 4), (897, 0, 28, 4), (1019, 0, 28, 4), (1088, 0, 28, 4), (577, 400, 28, 4), (640, 639, 28, 4), (930, 0, 32, 32),
          (1480, 0, 12, 2), (950, 31, 30, 6), (1408, 0, 20, 1)]
WHOLE = [(1089, 0, 28, 4), (961, 0, 32, 32)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", SHARED + WHOLE)
def test_halves(dt, m, past, H, Hkv):
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    n, g = m + past, H // Hkv
    q, k, v = normal_bits(m, (m, H, 128), dt), normal_bits(n + 1, (n + 64, Hkv, 128), dt), normal_bits(n + 2, (n + 64, Hkv, 128), dt)
    k[n:], v[n:] = 0x7FFF, 0x7FFF  # (not to be read)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    x, weight, y = (dev_empty(s).fill_(0x3c00) for s in ((32, 5120), (1024, 5120), (32, 1024)))

    def call(out, stream=None):
        ops.hip_flash_attn_gqa_layer(out, dq, dk, dv, m, n, past, g, Hkv, 128, dt, *([] if stream is None else [stream]))

    outs = [dev_empty(q.shape).fill_(0x7FFF) for _ in range(12)]
    for o in outs:
        call(o)
        ops.hip_matmul_layer(y, x, weight, 32, 1024, 5120, dt)  # (pieces of k)
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
    alone, ws = dev_empty(q.shape).fill_(0x7FFF), torch.zeros(16 << 20, dtype=torch.uint8, device="cuda")
    call_alone = lambda: bops.hip_flash_attn_gqa_alone_layer(alone, dq, dk, dv, ws, ws.numel(), m, n, past, g, Hkv, 128, dt)
    if (m, past, H, Hkv) in SHARED:
        call_alone()
        assert torch.equal(alone, o)
        assert not torch.equal(alone, outs[0])  # (some row is folded from halves)
    else:
        with pytest.raises(ops.LlmHipError):
            call_alone()
        assert torch.equal(o, outs[0])


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
def test_alone_in_place(dt):
    """Queries and outputs in one buffer: who goes over all keys by itself takes the queries in once more."""
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    m, H, Hkv = 1019, 28, 4
    dq, dk, dv = (to_dev(normal_bits(s, (m, h, 128), dt)) for s, h in ((1, H), (2, Hkv), (3, Hkv)))
    ws, want = torch.zeros(16 << 20, dtype=torch.uint8, device="cuda"), dev_empty((m, H, 128))
    bops.hip_flash_attn_gqa_alone_layer(want, dq, dk, dv, ws, ws.numel(), m, m, 0, H // Hkv, Hkv, 128, dt)
    for _ in range(5):
        both = dq.clone()
        bops.hip_flash_attn_gqa_alone_layer(both, both, dk, dv, ws, ws.numel(), m, m, 0, H // Hkv, Hkv, 128, dt)
        assert torch.equal(both, want)


def test_alone_arguments():
    import llm_simple_amd.bench_ops as bops
    buf = ctypes.create_string_buffer(96)
    p = (ctypes.addressof(buf) + 15) & ~15  # (refused before anything is launched)
    call = lambda at, m, dim, dt, room: bops.lib.llmhip_bench_flash_attn_gqa_alone(at, p, p, p, p, room, m, m, 0, 7, 4, dim, dt, None)
    assert call(p + 2, 1019, 128, DT_BFLOAT16, 16 << 20) == -1 and call(p, 0, 128, DT_BFLOAT16, 16 << 20) == -1
    assert call(p, 1019, 128, 0, 16 << 20) == -1 and call(p, 1019, 64, DT_BFLOAT16, 16 << 20) == -2
    assert call(p, 2, 128, DT_BFLOAT16, 16 << 20) == -2 and call(p, 1019, 128, DT_BFLOAT16, 1 << 20) == -3


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
