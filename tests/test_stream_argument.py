"""What the Python operators take as a stream: an address, None, or the ctypes object that llmhip_stream_create fills."""
import ctypes

import numpy as np
import pytest

from helpers import DT_FLOAT16, dev_empty, normal_bits, to_dev, to_host


def test_forms_of_a_stream():
    import torch
    import llm_simple_amd.ops as ops
    handle = ctypes.c_void_p(0x1230)

    class Wrapped:  # (as torch.cuda.Stream has it)
        _as_parameter_ = handle

    for stream in (None, 0, 0x1230, ctypes.c_void_p(), handle, ctypes.byref(handle), Wrapped()):
        for call in (lambda: ops.hip_add_layer(0, 0, 0, 8, DT_FLOAT16, stream),
                     lambda: ops.hip_add_layer(0, 0, 0, 8, DT_FLOAT16, stream=stream)):
            with pytest.raises(ops.LlmHipError) as e:  # parsed, then refused for its null buffers
                call()
            assert e.value.status == -1
    for stream in (1.5, object(), torch.zeros(1)):  # neither an address nor something that holds one
        with pytest.raises(Exception) as e:
            ops.hip_add_layer(0, 0, 0, 8, DT_FLOAT16, stream)
        assert not isinstance(e.value, ops.LlmHipError)
    for buffer in (handle, 1.5):  # a buffer is an address or has data_ptr()
        with pytest.raises(AttributeError):
            ops.hip_add_layer(buffer, 0, 0, 8, DT_FLOAT16)


@pytest.mark.gpu
def test_created_stream_handle():
    """A call under capture on the stream that the handle names: on any other it would not be recorded."""
    import torch
    import llm_simple_amd.ops as ops
    a, b = normal_bits(1, (64,), DT_FLOAT16), normal_bits(2, (64,), DT_FLOAT16)
    d_a, d_b, out, want = to_dev(a), to_dev(b), dev_empty((64,)).zero_(), dev_empty((64,))
    ops.hip_add_layer(want, d_a, d_b, 64, DT_FLOAT16)
    s = ctypes.c_void_p()
    assert ops.lib.llmhip_stream_create(ctypes.byref(s)) == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(s.value)):
        ops.hip_add_layer(out, d_a, d_b, 64, DT_FLOAT16, s)
    assert not to_host(out).any()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(to_host(out), to_host(want))
    assert ops.lib.llmhip_stream_destroy(s) == 0
