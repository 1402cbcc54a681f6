"""Two workgroups to a CU in the batched decode: from one block of keys and one workgroup more than CUs on, one split and several, a last block of one key
and a whole one, folded by folders, and under capture by flags or a second launch.  Against the oracle; and a workspace of the count that one workgroup
to a CU would take still does."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("batch,n,H,Hkv", [(9, 1, 32, 32), (9, 128, 32, 32), (9, 257, 32, 32), (16, 384, 32, 32), (10, 700, 64, 32), (10, 1172, 32, 32),
                                           (5, 1025, 64, 64), (16, 250, 40, 20)])
def test_two_to_a_cu(dt, batch, n, H, Hkv):
    import torch
    import llm_simple_amd.ops as ops
    g = H // Hkv
    q = normal_bits(n, (batch, 1, H, 128), dt)
    k, v = normal_bits(n + 1, (batch, n, Hkv, 128), dt), normal_bits(n + 2, (batch, n, Hkv, 128), dt)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    default = ops.flash_decode_default_splits(batch, n, Hkv)
    for splits in sorted({1, 2, 3, 5, default}):
        need = ops.flash_decode_workspace_bytes(batch, g, Hkv, 128, splits)
        ws = torch.full((need // 4 + 4,), 0x7fc00001, dtype=torch.int64).to(torch.int32).cuda()
        args = (dq, dk, dv, ws, need, batch, n, n, g, Hkv, 128, splits, dt)
        out, replayed, graph = dev_empty(q.shape), dev_empty(q.shape), torch.cuda.CUDAGraph()
        ops.hip_flash_decode_gqa_layer(out, *args)
        check_attention(to_host(out), q, k, v, n, n - 1, dt, batch=True)
        with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
            ops.hip_flash_decode_gqa_layer(replayed, *args, torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            replayed.fill_(0x7FFF)
            graph.replay()
            assert np.array_equal(to_host(replayed), to_host(out)), splits


def test_workspace_of_the_count_for_one_to_a_cu():
    import torch
    import llm_simple_amd.ops as ops
    batch, n, Hkv, one = 10, 1172, 32, 2
    assert ops.flash_decode_default_splits(batch, n, Hkv) > one
    q = normal_bits(1, (batch, 1, Hkv, 128), DT_BFLOAT16)
    k, v = (normal_bits(s, (batch, n, Hkv, 128), DT_BFLOAT16) for s in (2, 3))
    room = ops.flash_decode_workspace_bytes(batch, 1, Hkv, 128, one)
    ws, out = torch.empty(room, dtype=torch.uint8, device="cuda"), dev_empty(q.shape)
    ops.hip_flash_decode_gqa_layer(out, to_dev(q), to_dev(k), to_dev(v), ws, room, batch, n, n, 1, Hkv, 128, 0, DT_BFLOAT16)
    check_attention(to_host(out), q, k, v, n, n - 1, DT_BFLOAT16, batch=True)
