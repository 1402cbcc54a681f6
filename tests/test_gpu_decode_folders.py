"""Decode partials folded by workgroups of the same launch: the edges of that form (4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 128 splits and 129, 8, 9, 15 and
16 query rows, 1023 (sequence, kv head) pairs and 1024, no CU left idle, more than one round of workgroups), each against the oracle,
bit for bit the same when repeated over the words of other calls and from a HIP graph, which folds otherwise.  And what a folder does
that finds no partials in time: its rows from the caches by itself, in the measurement library's copy, where none waits."""
import numpy as np
import pytest

import oracle.oracle as orc
from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, f32_dev, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (batch, n, H, Hkv, splits)
CASES = [(1, 1030, 40, 8, 4), (1, 1030, 7, 1, 5), (1, 2000, 28, 4, 16), (1, 2100, 8, 1, 16), (1, 2177, 5, 1, 17), (2, 4095, 8, 1, 31),
         (1, 4097, 40, 8, 32), (1, 4300, 40, 8, 33), (1, 8200, 7, 1, 64), (1, 8400, 14, 2, 65), (1, 12700, 12, 2, 99), (2, 16500, 8, 1, 128),
         (1, 17000, 6, 1, 129), (1, 700, 15, 1, 6), (1, 2000, 16, 1, 16), (2, 2100, 30, 2, 17), (1, 12700, 32, 2, 99), (1, 1100, 45, 5, 9), (1, 2000, 9, 1, 9), (3, 4000, 24, 8, 11), (9, 1500, 14, 2, 12),
         (1023, 257, 1, 1, 2), (1024, 257, 1, 1, 2), (1, 40000, 4, 4, 32)]


@pytest.mark.parametrize("room", [1, 2])  # (9 to 16 rows take folders where there is twice the room)
@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
def test_folders(dt, room):
    import torch
    import llm_simple_amd.ops as ops
    ws_bytes = max(ops.flash_decode_workspace_bytes(b, H // Hkv, Hkv, 128, s) for b, n, H, Hkv, s in CASES) * room
    ws = torch.full((ws_bytes // 4,), 0x7fc00001, dtype=torch.int64).to(torch.int32).cuda()
    calls = []
    for b, n, H, Hkv, splits in CASES:
        print(b, n, H, Hkv, splits, flush=True)
        q = normal_bits(n, (b, 1, H, 128), dt)
        k, v = normal_bits(n + 1, (b, n, Hkv, 128), dt), normal_bits(n + 2, (b, n, Hkv, 128), dt)
        need = ops.flash_decode_workspace_bytes(b, H // Hkv, Hkv, 128, splits) * room
        args = (to_dev(q), to_dev(k), to_dev(v), ws, need, b, n, n, H // Hkv, Hkv, 128, splits, dt)
        out = dev_empty((b, 1, H, 128))
        ops.hip_flash_decode_gqa_layer(out, *args)
        want = to_host(out)
        check_attention(want, q, k, v, n, n - 1, dt, batch=True)
        replayed, graph = dev_empty((b, 1, H, 128)), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
            ops.hip_flash_decode_gqa_layer(replayed, *args, torch.cuda.current_stream().cuda_stream)
        calls.append((args, want, graph, replayed))
    rng = np.random.default_rng(7)
    for _ in range(60):
        args, want, graph, replayed = calls[rng.integers(len(calls))]
        out = torch.full(want.shape, 0x7FFF, dtype=torch.int16, device="cuda")
        ops.hip_flash_decode_gqa_layer(out, *args)
        assert np.array_equal(to_host(out), want)
        if rng.random() < 0.3:
            replayed.fill_(0x7FFF)
            graph.replay()
            assert np.array_equal(to_host(replayed), want)


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("batch,n,H,Hkv,splits", [(1, 500, 12, 2, 4), (3, 1000, 40, 8, 6), (2, 3000, 28, 4, 16), (1, 4100, 16, 2, 32), (1, 2000, 30, 2, 12), (2, 1100, 16, 1, 9),
                                                   (1, 9000, 12, 2, 70)])
def test_folder_alone(dt, batch, n, H, Hkv, splits):
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    q = normal_bits(n, (batch, 1, H, 128), dt)
    k, v = normal_bits(n + 1, (batch, n + 2, Hkv, 128), dt), normal_bits(n + 2, (batch, n + 2, Hkv, 128), dt)
    ws = torch.zeros(max(4 << 20, ops.flash_decode_workspace_bytes(batch, H // Hkv, Hkv, 128, splits)), dtype=torch.uint8, device="cuda")
    out = dev_empty((batch, 1, H, 128))
    bops.hip_flash_decode_gqa_alone_layer(out, to_dev(q), to_dev(k), to_dev(v), ws, ws.numel(), batch, n, n + 2, H // Hkv, Hkv, 128,
                                          splits, dt)
    check_attention(to_host(out), q, k, v, n, n - 1, dt, batch=True)
    # the fused step: also the new row of either cache, which its owner stores as well
    table = orc.init_freq_cis(128, n + 2, 1e4, dt)
    new_q, new_k, new_v = normal_bits(5, (1, H, 128), dt), normal_bits(6, (1, Hkv, 128), dt), normal_bits(7, (1, Hkv, 128), dt)
    caches = []
    for alone in (False, True):
        kc, vc, out = to_dev(k[0]), to_dev(v[0]), dev_empty((1, H, 128))
        head = (out, kc, vc, f32_dev(table), to_dev(new_q), to_dev(new_k), to_dev(new_v))
        if alone:
            bops.hip_decode_step_gqa_alone_layer(*head, ws, ws.numel(), n - 1, H // Hkv, Hkv, 128, 1, splits, dt)
        else:
            ops.hip_decode_step_gqa_layer(*head, n - 1, H // Hkv, Hkv, 128, True, dt)
        caches.append((to_host(kc), to_host(vc)))
    assert np.array_equal(caches[0][0], caches[1][0]) and np.array_equal(caches[0][1], caches[1][1])
    check_attention(to_host(out), orc.rope(new_q, table, n - 1, True, dt), caches[1][0], caches[1][1], n, n - 1, dt)
