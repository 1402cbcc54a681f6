"""Chunks whose query rows go through the decode kernel in tiles of up to 16: two tiles and eight, a short last tile, whole
tiles of 16 rows, one partial and many, keys behind the last visible one (NaN), the edges of the rule -- against the oracle, the same bits
when repeated and from a HIP graph, which folds otherwise, and on a stream without scratch under capture, which takes key ranges."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (m, past, H, Hkv)
CASES = [(3, 40, 28, 4), (3, 200, 28, 4), (4, 127, 28, 4), (5, 1000, 28, 4), (6, 2049, 28, 4), (16, 1100, 28, 4), (17, 1100, 28, 4), (3, 4095, 12, 2),
         (16, 2000, 12, 2), (7, 900, 40, 8), (9, 600, 40, 8), (9, 1500, 16, 1), (2, 3000, 16, 1), (8, 31000, 16, 1), (17, 1500, 2, 1), (63, 700, 4, 2),
         (64, 700, 4, 2), (20, 20, 6, 1), (12, 500, 40, 8)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,past,H,Hkv", CASES)
def test_tiles(dt, m, past, H, Hkv):
    import torch
    import llm_simple_amd.ops as ops
    n = m + past
    q, k, v = normal_bits(m, (m, H, 128), dt), normal_bits(n + 1, (n, Hkv, 128), dt), normal_bits(n + 2, (n, Hkv, 128), dt)
    behind = np.full((128, Hkv, 128), 0x7FFF, dtype=k.dtype)
    args = (to_dev(q), to_dev(np.concatenate([k, behind])), to_dev(np.concatenate([v, behind])), m, n, past, H // Hkv, Hkv, 128, dt)
    side, bare = torch.cuda.Stream(), torch.cuda.Stream()
    out, replayed, cold = (dev_empty(q.shape) for _ in range(3))
    torch.cuda.synchronize()
    ops.hip_flash_attn_gqa_layer(out, *args, side.cuda_stream)
    side.synchronize()
    want = to_host(out)
    check_attention(want, q, k, v, n, past, dt)
    graph, bare_graph = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.hip_flash_attn_gqa_layer(replayed, *args, torch.cuda.current_stream().cuda_stream)
    bare_call = n < 2048  # (a longer cache may insist on scratch)
    if bare_call:
        with torch.cuda.graph(bare_graph, stream=bare):
            ops.hip_flash_attn_gqa_layer(cold, *args, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        for o in (out, replayed, cold):
            o.fill_(0x7FFF)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        if bare_call:
            bare_graph.replay()
            torch.cuda.synchronize()
            check_attention(to_host(cold), q, k, v, n, past, dt)
        assert np.array_equal(to_host(replayed), want)
        ops.hip_flash_attn_gqa_layer(out, *args, side.cuda_stream)
        side.synchronize()
        assert np.array_equal(to_host(out), want)
