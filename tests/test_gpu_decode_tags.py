"""Decode partials whose words carry a tag: the edges of that form (8 splits and 9, 8 query rows and 9, one row, a workspace
that holds no more than an exact call needs, 96 and 112 partials of 8 rows), calls that take turns on one workspace so
that each finds the words of another, and a workspace full of numbers that look like tags.  Against the oracle, and bit for bit
against the same call from a HIP graph, which folds by flags (up to 8 partials of 8 rows, 16 of 4) or by a second launch."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, check_attention, dev_empty, normal_bits, to_dev, to_host

pytestmark = pytest.mark.gpu

# (batch, n, H, Hkv, splits)
CASES = [(1, 129, 12, 2, 2), (1, 300, 7, 1, 3), (1, 512, 32, 32, 4), (2, 1024, 8, 1, 8), (1, 1025, 28, 4, 9), (2, 800, 9, 1, 7),
         (3, 2999, 16, 2, 6), (1, 640, 2, 2, 5), (4, 7168, 8, 1, 8), (1, 260, 24, 3, 3), (6, 1024, 16, 2, 8), (7, 1024, 16, 2, 8)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("room", [1, 4])
def test_tagged_partials(dt, room):
    import torch
    import llm_simple_amd.ops as ops
    calls = []
    ws_bytes = max(ops.flash_decode_workspace_bytes(b, H // Hkv, Hkv, 128, s) for b, n, H, Hkv, s in CASES) * room
    ws = torch.full((ws_bytes // 4,), 0x7fc00001, dtype=torch.int64).to(torch.int32).cuda()
    for b, n, H, Hkv, splits in CASES:
        q = normal_bits(n, (b, 1, H, 128), dt)
        k, v = normal_bits(n + 1, (b, n, Hkv, 128), dt), normal_bits(n + 2, (b, n, Hkv, 128), dt)
        # room 1: what flags need and not a byte more
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
    rng = np.random.default_rng(5)
    for _ in range(150):
        args, want, graph, replayed = calls[rng.integers(len(calls))]
        out = torch.full(want.shape, 0x7FFF, dtype=torch.int16, device="cuda")
        ops.hip_flash_decode_gqa_layer(out, *args)
        assert np.array_equal(to_host(out), want)
        if rng.random() < 0.3:
            replayed.fill_(0x7FFF)
            graph.replay()
            assert np.array_equal(to_host(replayed), want)


@pytest.mark.parametrize("halves", [(1, 0), (0, 1), (0, 0)])
def test_half_a_number_is_not_the_number(halves):
    """A workspace full of partials with one half of the launch's own number beside every word (the sequence of numbers:
    tests/cpp/test_device_host.cpp): none of them may be folded."""
    import torch
    import llm_simple_amd.ops as ops
    # 9 blocks in 7 splits, the last workgroups in a second round: some look long before others have stored
    b, n, H, Hkv, splits, dt = 10, 1100, 12, 4, 7, DT_BFLOAT16
    q = normal_bits(1, (b, 1, H, 128), dt)
    k, v = normal_bits(2, (b, n, Hkv, 128), dt), normal_bits(3, (b, n, Hkv, 128), dt)
    need = ops.flash_decode_workspace_bytes(b, H // Hkv, Hkv, 128, splits)
    ws = torch.zeros(need // 4, dtype=torch.int32, device="cuda")
    args = (to_dev(q), to_dev(k), to_dev(v), ws, need, b, n, n, H // Hkv, Hkv, 128, splits, dt)
    out = dev_empty((b, 1, H, 128))
    ops.hip_flash_decode_gqa_layer(out, *args)
    want = to_host(out)
    check_attention(want, q, k, v, n, n - 1, dt, batch=True)

    def number():  # of the last launch: beside the first two words of the first partial
        words = ws[:4].cpu().numpy().view(np.uint32)
        return int(words[1]) | int(words[3]) << 32

    for _ in range(20):
        due = (number() + 0x9E3779B97F4A7C15) % 2 ** 64
        piece = np.array([1e3, 0, 1e3, 0], dtype=np.float32).view(np.uint32)
        piece[1] = (due & 0xffffffff) ^ (0 if halves[0] else 1 << 17)
        piece[3] = (due >> 32) ^ (0 if halves[1] else 1 << 17)
        ws.copy_(torch.from_numpy(np.tile(piece, need // 16).view(np.int32)))
        out.fill_(0x7FFF)
        ops.hip_flash_decode_gqa_layer(out, *args)
        assert np.array_equal(to_host(out), want)
        assert number() == due  # tags, and of the number foreseen
