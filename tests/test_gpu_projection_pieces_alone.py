"""Projections in pieces of k, when the workgroups that add up make all sums by themselves (the measurement library's copy): every tile's does, and the bits
are those of a call whose workgroups pass their sums on, also with prompts between that use the same buffer."""
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k", [(9, 1024, 5120), (16, 512, 3584), (17, 16, 3072), (31, 1008, 4160), (32, 4096, 3072), (33, 1024, 6080), (64, 2032, 3648),
                                   (65, 496, 5120), (97, 1024, 5056), (128, 1024, 3136), (40, 528, 6016)])
def test_alone(m, n, k, dt):
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    x, w, b = to_dev(normal_bits(m + k, (m, k), dt)), to_dev(normal_bits(n, (n, k), dt)), f32_dev([1.0] * n)
    q, kv, o = (to_dev(normal_bits(s, (1019, h, 128), dt)) for s, h in ((1, 28), (2, 4), (3, 28)))
    outs = [dev_empty((m, n)).fill_(0x7fff) for _ in range(4)]
    for out in outs:
        ops.hip_matmul_bias_layer(out, x, w, b, m, n, k, dt)
        ops.hip_flash_attn_gqa_layer(o, q, kv, kv, 1019, 1019, 0, 7, 4, 128, dt)  # (halves)
    alone, ws = dev_empty((m, n)).fill_(0x7fff), torch.zeros(2 << 20, dtype=torch.uint8, device="cuda")
    bops.hip_matmul_alone_layer(alone, x, w, b, ws, ws.numel(), m, n, k, dt)
    for out in outs:
        assert torch.equal(alone, out)
    # who makes all sums itself keeps those so far in the last piece's place among the words (per tile of 32 x 32 and piece 8192 bytes, 4096 of sums)
    tiles = -(-m // 32) * -(-n // 32)
    pieces = min(256 // tiles, k // 64 // 12, 8)
    kept = ws[:tiles * pieces * 8192].view(torch.int32).view(tiles, pieces, 2048)[:, -1, :1024]
    assert (kept != 0).any(1).all()
