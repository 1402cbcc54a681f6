"""Attention whose output goes to the queries' own buffer: the same bits as with a buffer of its own.  One token and a few, tiles of rows of
which the last is short, launches of more workgroups than are resident at once, key ranges, prompts, batches, the fused step, and
folders that find no partials and compute their rows from the caches (the measurement library's copy)."""
import pytest

import oracle.oracle as orc
from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, f32_dev, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu


# (m, past, H, Hkv): tiles of rows are those of 3 to 63 tokens; 8 tiles of 4 kv heads in 8 to 11 parts, and of 8 in 9, are two rounds
@pytest.mark.parametrize("m,past,H,Hkv", [(1, 700, 28, 4), (2, 3000, 28, 4), (4, 1200, 28, 4), (5, 1000, 28, 4), (7, 900, 40, 8), (15, 1100, 28, 4),
                                          (22, 1300, 40, 8), (29, 1200, 16, 4), (57, 1200, 8, 4), (9, 1500, 16, 1), (61, 700, 4, 2), (30, 4130, 40, 8),
                                          (33, 8160, 28, 4), (200, 0, 12, 2), (512, 0, 28, 4), (1019, 0, 28, 4), (1700, 0, 28, 4),
                                          (2100, 0, 40, 8), (3500, 0, 28, 4), (400, 1000, 32, 32)])
@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
def test_attention(dt, m, past, H, Hkv):
    import llm_simple_amd.ops as ops
    n = m + past
    q, k, v = normal_bits(m, (m, H, 128), dt), normal_bits(n + 1, (n, Hkv, 128), dt), normal_bits(n + 2, (n, Hkv, 128), dt)
    dq, dk, dv, out = to_dev(q), to_dev(k), to_dev(v), dev_empty(q.shape)
    ops.hip_flash_attn_gqa_layer(out, dq, dk, dv, m, n, past, H // Hkv, Hkv, 128, dt)
    want = to_host(out)
    if m < 100:
        check_attention(want, q, k, v, n, past, dt)
    for _ in range(3):
        buf = to_dev(q)
        ops.hip_flash_attn_gqa_layer(buf, buf, dk, dv, m, n, past, H // Hkv, Hkv, 128, dt)
        assert (to_host(buf) == want).all()


@pytest.mark.parametrize("batch,n,H,Hkv,splits", [(1, 500, 12, 2, 4), (3, 1000, 40, 8, 6), (2, 3000, 28, 4, 16), (1, 4100, 16, 2, 32), (1, 2000, 30, 2, 12),
                                                  (2, 1100, 16, 1, 9), (1, 9000, 12, 2, 70), (1, 17000, 6, 1, 129), (9, 3000, 40, 8, 5)])
@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
def test_decode(dt, batch, n, H, Hkv, splits):
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    g = H // Hkv
    q = normal_bits(n, (batch, 1, H, 128), dt)
    k, v = normal_bits(n + 1, (batch, n, Hkv, 128), dt), normal_bits(n + 2, (batch, n, Hkv, 128), dt)
    dk, dv = to_dev(k), to_dev(v)
    ws = torch.zeros(2 * ops.flash_decode_workspace_bytes(batch, g, Hkv, 128, splits), dtype=torch.uint8, device="cuda")
    table = f32_dev(orc.init_freq_cis(128, n, 1e4, dt))
    new_k, new_v = to_dev(normal_bits(6, (1, Hkv, 128), dt)), to_dev(normal_bits(7, (1, Hkv, 128), dt))
    for module, alone in ((ops, ""), (bops, "_alone")):
        def decode(out, src):
            getattr(module, f"hip_flash_decode_gqa{alone}_layer")(out, src, dk, dv, ws, ws.numel(), batch, n, n, g, Hkv, 128, splits, dt)

        def step(out, src):
            head = (out, to_dev(k[0]), to_dev(v[0]), table, src, new_k, new_v)
            if alone:
                bops.hip_decode_step_gqa_alone_layer(*head, ws, ws.numel(), n - 1, g, Hkv, 128, 1, splits, dt)
            else:
                ops.hip_decode_step_gqa_layer(*head, n - 1, g, Hkv, 128, True, dt)

        for call, src in ((decode, q), (step, q[0])):
            out = dev_empty(src.shape)
            call(out, to_dev(src))
            want = to_host(out)
            if call is decode:
                check_attention(want, q, k, v, n, n - 1, dt, batch=True)
            for _ in range(3):
                buf = to_dev(src)
                call(buf, buf)
                assert (to_host(buf) == want).all(), (alone, call.__name__)
