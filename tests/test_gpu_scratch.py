"""Calls that take split-KV scratch when there is none to be had: on a stream under capture whose buffer would have to
grow they run with what there is, except those that insist on theirs (a short chunk or a token over a long cache:
LLMHIP_ERR_WORKSPACE); the batched decode does the same with a workspace smaller than its default count takes; and a
buffer grows on one stream while another is being captured; and a graph is replayed on another stream than its own."""
import contextlib
import ctypes

import numpy as np
import pytest

from helpers import DT_BFLOAT16, check_attention, dev_empty, f32_dev, normal_bits, to_dev, to_host
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DT = DT_BFLOAT16


@contextlib.contextmanager
def fresh_stream():
    """A stream the library has not seen, so without scratch."""
    import torch
    import llm_simple_amd.ops as ops
    s = ctypes.c_void_p()
    assert ops.lib.llmhip_stream_create(ctypes.byref(s)) == 0
    try:
        yield torch.cuda.ExternalStream(s.value)
    finally:
        torch.cuda.synchronize()
        assert ops.lib.llmhip_stream_destroy(s) == 0


def inputs(m, n, H, Hkv):
    q, k, v = (normal_bits(s + n, (r, h, 128), DT) for s, r, h in ((1, m, H), (2, n, Hkv), (3, n, Hkv)))
    return (q, k, v), [to_dev(a) for a in (q, k, v)]


def replays_match(graph, out, bits, n, past):
    import torch
    first = None
    for _ in range(3):
        out.fill_(0x7FFF)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = to_host(out).copy()
        if first is None:
            first = got
            check_attention(got, *bits, n, past, DT)
        assert np.array_equal(got, first)


# (tokens, cached, query heads, kv heads): a token over a short cache; chunks behind less than 2048 keys, or less than 8
# times their length; `insists`: a chunk that may not do with less than 1.9 MB, where its fastest plan takes 6.6
@pytest.mark.parametrize("m,past,H,Hkv,insists", [(1, 300, 12, 2, False), (2, 255, 32, 32, False), (20, 1500, 28, 4, False),
                                                  (65, 1900, 12, 2, False), (300, 1500, 12, 2, False),
                                                  (700, 1900, 12, 2, False), (65, 2500, 28, 4, True)])
@pytest.mark.parametrize("warm", [False, True])
def test_captured_without_room(m, past, H, Hkv, insists, warm):
    import torch
    import llm_simple_amd.ops as ops
    n = m + past
    need = ops.lib.llmhip_flash_attn_scratch_bytes(m, n, past, H // Hkv, Hkv)
    assert need > 0
    bits, (q, k, v) = inputs(m, n, H, Hkv)
    out = dev_empty(q.shape)
    with fresh_stream() as s:
        if warm:  # the smallest buffer: 4 MiB
            ops.hip_flash_attn_gqa_layer(dev_empty((1, H, 128)), q, k, v, 1, 257, 256, H // Hkv, Hkv, 128, DT, s.cuda_stream)
            s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out.fill_(0)
            rc = ops.lib.llmhip_flash_attn_gqa(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), m, n, past, H // Hkv,
                                               Hkv, 128, DT, s.cuda_stream)
        assert rc == (-3 if insists and not warm else 0), rc
        if rc == 0:
            replays_match(graph, out, bits, n, past)


def test_captured_decode_step_without_room():
    """The fused step over 384 keys, captured first thing: cache and output as without a graph."""
    import torch
    import llm_simple_amd.ops as ops
    pos, H, Hkv = 383, 12, 2
    assert ops.lib.llmhip_flash_attn_scratch_bytes(1, pos + 1, pos, H // Hkv, Hkv) > 0
    bits, (q, k, v) = inputs(1, pos + 1, H, Hkv)
    table = orc.init_freq_cis(128, pos + 1, 1e6, DT)
    new_k, new_v = normal_bits(7, (1, Hkv, 128), DT), normal_bits(8, (1, Hkv, 128), DT)
    want_q = orc.rope(bits[0], table, pos, True, DT)
    kc, vc = bits[1].copy(), bits[2].copy()
    orc.kv_append(kc, orc.rope(new_k, table, pos, True, DT), pos)
    orc.kv_append(vc, new_v, pos)
    d_table, d_k, d_v, out = f32_dev(table), to_dev(new_k), to_dev(new_v), dev_empty(q.shape)
    with fresh_stream() as s:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            ops.hip_decode_step_gqa_layer(out, k, v, d_table, q, d_k, d_v, pos, H // Hkv, Hkv, 128, True, DT, s.cuda_stream)
        replays_match(graph, out, (want_q, kc, vc), pos + 1, pos)
    assert np.array_equal(to_host(k), kc) and np.array_equal(to_host(v), vc)


@pytest.mark.parametrize("m,past,H,Hkv", [(1, 32767, 40, 8), (1, 511, 32, 32), (24, 40000, 40, 8), (200, 16001, 28, 4)])
def test_refused_without_room(m, past, H, Hkv):
    """What insists on its scratch is refused under capture, and the capture stays usable; warmed up, the same call is
    captured and replays give the eager bits."""
    import torch
    import llm_simple_amd.ops as ops
    n = m + past
    bits, (q, k, v) = inputs(m, n, H, Hkv)
    out, eager, small = dev_empty(q.shape), dev_empty(q.shape), dev_empty((1, H, 128))
    args = (m, n, past, H // Hkv, Hkv, 128, DT)
    with fresh_stream() as s:
        for warmed in (False, True):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=s):
                ops.hip_flash_attn_gqa_layer(small, q, k, v, 1, 64, 63, H // Hkv, Hkv, 128, DT, s.cuda_stream)
                rc = ops.lib.llmhip_flash_attn_gqa(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), *args, s.cuda_stream)
            assert rc == (0 if warmed else -3), rc
            small.fill_(0x7FFF)
            out.fill_(0x7FFF)
            for _ in range(3):
                graph.replay()
                torch.cuda.synchronize()
            check_attention(to_host(small), bits[0][:1], *bits[1:], 64, 63, DT)
            if warmed:
                assert np.array_equal(to_host(out), to_host(eager))
            ops.hip_flash_attn_gqa_layer(eager, q, k, v, *args, s.cuda_stream)
            torch.cuda.synchronize()


def test_buffer_grows_while_another_stream_is_captured():
    import torch
    import llm_simple_amd.ops as ops
    m, past, H, Hkv = 200, 3001, 28, 4
    n = m + past
    bits, (q, k, v) = inputs(m, n, H, Hkv)
    out, small = dev_empty(q.shape), dev_empty((1, H, 128))
    with fresh_stream() as captured, fresh_stream() as s:
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=captured):  # (capture mode "global")
            ops.hip_flash_attn_gqa_layer(small, q, k, v, 1, 64, 63, H // Hkv, Hkv, 128, DT, captured.cuda_stream)
            ops.hip_flash_attn_gqa_layer(out, q, k, v, m, n, past, H // Hkv, Hkv, 128, DT, s.cuda_stream)
        s.synchronize()
        check_attention(to_host(out), *bits, n, past, DT)
        replays_match(graph, small, (bits[0][:1],) + bits[1:], 64, 63)


def test_replay_elsewhere_beside_calls_that_need_no_partials():
    """A graph keeps its stream's partials and is replayed on another stream, while prompts and projections run on its own: what workgroups of
    those pass each other lies elsewhere."""
    import torch
    import llm_simple_amd.ops as ops
    (n, H, Hkv), m, (rows, width, k_dim) = (32768, 40, 8), 1019, (32, 1024, 5120)
    bits, (q, k, v) = inputs(1, n, H, Hkv)
    _, (pq, pk, pv) = inputs(m, m, 28, 4)
    x, w = to_dev(normal_bits(4, (rows, k_dim), DT)), to_dev(normal_bits(5, (width, k_dim), DT))
    out, prompts, sums = dev_empty(q.shape), [dev_empty(pq.shape) for _ in range(30)], [dev_empty((rows, width)) for _ in range(30)]
    with fresh_stream() as s, fresh_stream() as other:
        one = lambda: ops.hip_flash_attn_gqa_layer(out, q, k, v, 1, n, n - 1, H // Hkv, Hkv, 128, DT, s.cuda_stream)
        one()  # (the buffer)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            one()
        replays_match(graph, out, bits, n, n - 1)
        want = to_host(out).copy()
        for i, (p, y) in enumerate(zip(prompts, sums)):  # (the first ones by themselves)
            if i:
                with torch.cuda.stream(other):
                    graph.replay()
            ops.hip_flash_attn_gqa_layer(p, pq, pk, pv, m, m, 0, 7, 4, 128, DT, s.cuda_stream)
            ops.hip_matmul_layer(y, x, w, rows, width, k_dim, DT, s.cuda_stream)
            if not i:
                torch.cuda.synchronize()
        torch.cuda.synchronize()
        assert np.array_equal(to_host(out), want)
        for o in prompts[1:] + sums[1:]:
            assert torch.equal(o, prompts[0] if o.dim() == 3 else sums[0])


def test_batched_decode_with_less_workspace_than_the_default_count_takes():
    import torch
    import llm_simple_amd.ops as ops
    batch, n, H, Hkv = 3, 300, 12, 2
    g = H // Hkv
    assert ops.flash_decode_default_splits(batch, n, Hkv) > 1
    q = normal_bits(1, (batch, 1, H, 128), DT)
    k, v = (normal_bits(s, (batch, n, Hkv, 128), DT) for s in (2, 3))
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    two = ops.flash_decode_workspace_bytes(batch, g, Hkv, 128, 2)
    ws = torch.empty(two, dtype=torch.uint8, device="cuda")
    for room in (0, 16, two):
        out = dev_empty(q.shape)
        ops.hip_flash_decode_gqa_layer(out, dq, dk, dv, ws if room else None, room, batch, n, n, g, Hkv, 128, 0, DT)
        check_attention(to_host(out), q, k, v, n, n - 1, DT, batch=True)
    # an explicit count, and a default that insists on its room, are refused as ever
    args = (dq.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), None, 0)
    assert ops.lib.llmhip_flash_decode_gqa(*args, batch, n, n, g, Hkv, 128, 2, DT, None) == -3
    assert ops.lib.llmhip_flash_decode_gqa(*args, 1, 32768, 32768, 5, 8, 128, 0, DT, None) == -3


def test_workspace_of_an_earlier_default_count():
    """A workspace that held the default count by the model before the present one (7 splits, 10 now) still does."""
    import torch
    import llm_simple_amd.ops as ops
    batch, n, H, Hkv = 3, 3584, 40, 8
    q = normal_bits(1, (batch, 1, H, 128), DT)
    k, v = (normal_bits(s, (batch, n, Hkv, 128), DT) for s in (2, 3))
    seven = ops.flash_decode_workspace_bytes(batch, H // Hkv, Hkv, 128, 7)
    assert ops.flash_decode_default_splits(batch, n, Hkv) > 7
    ws, out = torch.empty(seven, dtype=torch.uint8, device="cuda"), dev_empty(q.shape)
    ops.hip_flash_decode_gqa_layer(out, to_dev(q), to_dev(k), to_dev(v), ws, seven, batch, n, n, H // Hkv, Hkv, 128, 0, DT)
    check_attention(to_host(out), q, k, v, n, n - 1, DT, batch=True)


def test_a_growing_buffer_stays_bounded():
    """Chunks that need more and more: what the stream holds, replaced buffers included, stays under twice the power
    of two that holds the largest, and goes with the stream."""
    import torch
    import llm_simple_amd.ops as ops
    sizes = [(700, 1900, 12, 2), (700, 4000, 28, 4), (1500, 9000, 28, 4), (3000, 9000, 28, 4), (3000, 16384, 32, 32),
             (3000, 16384, 28, 4)]
    needs = [ops.lib.llmhip_flash_attn_scratch_bytes(m, m + p, p, H // Hkv, Hkv) for m, p, H, Hkv in sizes]
    assert sorted(needs) == needs and sum(needs) > 256 << 20
    q, k, v = (torch.zeros(r, h, 128, dtype=torch.int16, device="cuda") for r, h in ((3000, 32), (19384, 32), (19384, 32)))
    out = dev_empty(q.shape)
    with fresh_stream() as s:
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for m, past, H, Hkv in sizes:
            ops.hip_flash_attn_gqa_layer(out, q, k, v, m, m + past, past, H // Hkv, Hkv, 128, DT, s.cuda_stream)
        s.synchronize()
        held = free - torch.cuda.mem_get_info()[0]
        assert max(needs) <= held < 256 << 20  # (128 MiB and the smaller powers of two)
    assert free - torch.cuda.mem_get_info()[0] < 4 << 20
