"""Prompts whose longest rows two workgroups share, when the second one of a pair does not wait for the other half of the keys but goes over all of them by
itself (the measurement library's copy): bit for bit what a captured call gives, which shares no rows.  Which sizes share rows; calls that share
them give the same bits with projections between that use the same buffer."""
import ctypes

import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, normal_bits, to_dev

pytestmark = pytest.mark.gpu

SHARED = [(896, 0, 28, 4), (897, 0, 28, 4), (1019, 0, 28, 4), (1088, 0, 28, 4), (577, 400, 28, 4), (640, 639, 28, 4), (930, 0, 32, 32),
          (1480, 0, 12, 2), (950, 31, 30, 6), (1408, 0, 20, 1)]
WHOLE = [(1089, 0, 28, 4), (961, 0, 32, 32)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", SHARED + WHOLE)
def test_alone(dt, m, past, H, Hkv):
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    n, g = m + past, H // Hkv
    dq, dk, dv = (to_dev(normal_bits(s, (r, h, 128), dt)) for s, r, h in ((m, m, H), (n + 1, n, Hkv), (n + 2, n, Hkv)))
    x, weight, y = (dev_empty(s).fill_(0x3c00) for s in ((32, 5120), (1024, 5120), (32, 1024)))
    outs = [dev_empty((m, H, 128)).fill_(0x7FFF) for _ in range(6)]
    for o in outs:
        ops.hip_flash_attn_gqa_layer(o, dq, dk, dv, m, n, past, g, Hkv, 128, dt)
        ops.hip_matmul_layer(y, x, weight, 32, 1024, 5120, dt)  # (pieces of k)
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    graph, whole = torch.cuda.CUDAGraph(), dev_empty((m, H, 128))
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        ops.hip_flash_attn_gqa_layer(whole, dq, dk, dv, m, n, past, g, Hkv, 128, dt, torch.cuda.current_stream().cuda_stream)
    graph.replay()
    alone, ws = dev_empty((m, H, 128)).fill_(0x7FFF), torch.zeros(16 << 20, dtype=torch.uint8, device="cuda")
    call_alone = lambda: bops.hip_flash_attn_gqa_alone_layer(alone, dq, dk, dv, ws, ws.numel(), m, n, past, g, Hkv, 128, dt)
    if (m, past, H, Hkv) in SHARED:
        call_alone()
        assert torch.equal(alone, whole)
        assert not torch.equal(alone, outs[0])  # (some row is folded from halves)
    else:
        with pytest.raises(ops.LlmHipError):
            call_alone()
        assert torch.equal(whole, outs[0])


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
