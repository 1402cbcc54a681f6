"""Decode over short caches: the partials are folded inside the decode kernel (up to 16 of them), in blocks of 64 keys
where the launch is thin.  The edges of that dispatch against the oracle, each call repeated on a workspace full of
garbage and replayed from a HIP graph between eager calls."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (batch, n, H, Hkv): 64-key blocks with a ragged last one, 8 of them, one past; 16 blocks of 128, one past; a launch too
# wide for 64-key blocks; 8, 15 and 16 query rows per kv head (column of the flag free, free, taken)
CASES = [(1, 129, 12, 2), (1, 385, 28, 4), (1, 512, 32, 32), (1, 513, 12, 2), (1, 2048, 40, 8), (1, 2049, 40, 8),
         (3, 500, 40, 8), (1, 400, 8, 1), (2, 700, 15, 1), (1, 900, 16, 1)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("batch,n,H,Hkv", CASES)
def test_folded_decode(dt, batch, n, H, Hkv):
    import torch
    import llm_simple_amd.ops as ops
    g = H // Hkv
    q = normal_bits(n, (batch, 1, H, 128), dt)
    k = normal_bits(n + 1, (batch, n + 3, Hkv, 128), dt)
    v = normal_bits(n + 2, (batch, n + 3, Hkv, 128), dt)
    k[:, n:] = 0x7FFF
    v[:, n:] = 0x7FFF
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    nb = -(-n // 128)
    ws_bytes = ops.flash_decode_workspace_bytes(batch, g, Hkv, 128, nb)
    ws = torch.randint(-2 ** 31, 2 ** 31, (max(ws_bytes, 16) // 4,), dtype=torch.int64).to(torch.int32).cuda()
    outs = [dev_empty((batch, 1, H, 128)) for _ in range(3)]

    def call(out, stream=0):
        ops.hip_flash_decode_gqa_layer(out, dq, dk, dv, ws, ws_bytes, batch, n, n + 3, g, Hkv, 128, nb, dt, stream)

    call(outs[0])
    want = to_host(outs[0])
    check_attention(want, q, k, v, n, n - 1, dt, batch=True)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(outs[1], torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        outs[1].fill_(0x7FFF)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(to_host(outs[1]), want)
        call(outs[2])
        assert np.array_equal(to_host(outs[2]), want)
