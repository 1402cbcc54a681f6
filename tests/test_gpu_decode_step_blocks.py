"""The fused decode step in blocks of 64 keys: 8, 9, 16, 17 and 32 of them, a last block of one key and a whole one, one block more than
the form takes, no CU left to the workgroups that fold, 7 query rows and 8 -- against the oracle, the same bits when repeated and from a
HIP graph, which folds by flags (up to 8 blocks, 4 rows) or by a second launch."""
import numpy as np
import pytest

import oracle.oracle as orc
from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, f32_dev, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (past, H, Hkv)
CASES = [(511, 28, 4), (512, 28, 4), (575, 12, 2), (576, 12, 2), (1023, 28, 4), (1024, 28, 4), (1087, 40, 8), (1900, 40, 8), (1921, 40, 8),
         (1985, 7, 1), (2047, 28, 4), (2048, 28, 4), (1500, 8, 1), (700, 32, 32), (1600, 12, 12)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("past,H,Hkv", CASES)
def test_step_blocks(dt, past, H, Hkv):
    import torch
    import llm_simple_amd.ops as ops
    n = past + 1
    k, v = normal_bits(n + 1, (n, Hkv, 128), dt), normal_bits(n + 2, (n, Hkv, 128), dt)
    k[past], v[past] = 0x7FFF, 0x7FFF  # the step's own to write
    q, new_k, new_v = normal_bits(5, (1, H, 128), dt), normal_bits(6, (1, Hkv, 128), dt), normal_bits(7, (1, Hkv, 128), dt)
    table = orc.init_freq_cis(128, n, 1e4, dt)
    kc, vc, out = to_dev(k), to_dev(v), dev_empty((1, H, 128))
    args = (kc, vc, f32_dev(table), to_dev(q), to_dev(new_k), to_dev(new_v), past, H // Hkv, Hkv, 128, True, dt)
    side = torch.cuda.Stream()
    ops.hip_decode_step_gqa_layer(out, *args, side.cuda_stream)  # (the stream's scratch)
    side.synchronize()
    want, k_after, v_after = to_host(out), to_host(kc), to_host(vc)
    assert np.array_equal(k_after[past:], orc.rope(new_k, table, past, True, dt)) and np.array_equal(v_after[past:], new_v)
    check_attention(want, orc.rope(q, table, past, True, dt), k_after, v_after, n, past, dt)
    replayed, graph = dev_empty((1, H, 128)), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.hip_decode_step_gqa_layer(replayed, *args, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        kc[past:].fill_(0x7FFF)
        replayed.fill_(0x7FFF)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(to_host(replayed), want)
        out.fill_(0x7FFF)
        torch.cuda.synchronize()
        ops.hip_decode_step_gqa_layer(out, *args, side.cuda_stream)
        side.synchronize()
        assert np.array_equal(to_host(out), want) and np.array_equal(to_host(kc), k_after)
