"""Few rows over some thousands of k, cut into pieces that workgroups of their own sum up: two to six pieces of equal and unequal numbers of
lines, ragged tiles, either side of the lines in rows, features and k.  Against sums in 64 bits; the same bits from call to call, with other users of
the stream's buffer between, on two streams at once, and by workgroups that make all sums by themselves; and under capture, where nothing is cut."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, dev_empty, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

CUT = [(9, 1024, 5120), (16, 512, 3584), (17, 16, 3072), (31, 1008, 4160), (32, 4096, 3072), (33, 1024, 6080), (64, 2032, 3648), (65, 496, 5120),
       (97, 1024, 5056), (128, 1024, 3136), (40, 528, 6016)]
WHOLE = [(8, 1024, 5120), (23, 3584, 3584), (9, 1024, 3008), (33, 2064, 3584), (17, 4112, 3072), (16, 1024, 6144), (24, 1024, 4000)]


def inputs(m, n, k, dt):
    x = normal_bits(m + k, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ref = orc.widen(x, dt).astype(np.float64) @ orc.widen(w, dt).T.astype(np.float64) + b
    return to_dev(x), to_dev(w), f32_dev(b), orc.widen(orc.round_to(ref.astype(np.float32), dt), dt)


def nan(m, n, dt):
    return to_dev(np.full((m, n), 0x7e00 if dt == DT_FLOAT16 else 0x7fc0, dtype=np.uint16))


def near(got, ref, dt):
    # one rounding of an fp32 sum: a step of the storage type, 1e-3 where the sum cancels (a NaN fails the comparison)
    return (np.abs(orc.widen(got, dt) - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k", CUT + WHOLE)
def test_pieces(m, n, k, dt):
    import torch
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    x, w, b, ref = inputs(m, n, k, dt)
    out = nan(m, n, dt)
    ops.hip_matmul_bias_layer(out, x, w, b, m, n, k, dt)
    got = to_host(out).copy()
    assert near(got, ref, dt)
    q, kv, o = (to_dev(normal_bits(s, (r, h, 128), dt)) for s, r, h in ((1, 1, 40), (2, 3000, 8), (3, 1, 40)))
    for _ in range(5):
        ops.hip_flash_attn_gqa_layer(o, q, kv, kv, 1, 3000, 2999, 5, 8, 128, dt)  # partials in the same buffer
        again = nan(m, n, dt)
        ops.hip_matmul_bias_layer(again, x, w, b, m, n, k, dt)
        assert torch.equal(again, out)
    alone, ws = nan(m, n, dt), torch.zeros(2 << 20, dtype=torch.uint8, device="cuda")
    call = lambda: bops.hip_matmul_alone_layer(alone, x, w, b, ws, ws.numel(), m, n, k, dt)
    if (m, n, k) in CUT:
        call()
        assert torch.equal(alone, out)
    else:
        with pytest.raises(ops.LlmHipError):
            call()
    graph, captured = torch.cuda.CUDAGraph(), dev_empty((m, n))
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        ops.hip_matmul_bias_layer(captured, x, w, b, m, n, k, dt, torch.cuda.current_stream().cuda_stream)
    for _ in range(2):
        captured.fill_(0x7fff)
        graph.replay()
        torch.cuda.synchronize()
        assert near(to_host(captured), ref, dt)


def test_pieces_on_two_streams():
    import torch
    import llm_simple_amd.ops as ops
    m, n, k, dt = 32, 2048, 5120, DT_BFLOAT16
    x, w, b, ref = inputs(m, n, k, dt)
    streams, outs = [torch.cuda.Stream() for _ in range(2)], [[nan(m, n, dt) for _ in range(30)] for _ in range(2)]
    torch.cuda.synchronize()
    for i in range(30):
        for s, o in zip(streams, outs):
            ops.hip_matmul_bias_layer(o[i], x, w, b, m, n, k, dt, s.cuda_stream)
    torch.cuda.synchronize()
    assert near(to_host(outs[0][0]), ref, dt)
    for o in outs[0] + outs[1]:
        assert torch.equal(o, outs[0][0])
