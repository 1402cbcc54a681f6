"""Few rows over a long k: every call of 17 rows or more whose tiles fit one round of workgroups runs on a kernel of this library,
which allocates nothing and can be captured with nothing warmed up.  On both sides of k = 6144, against sums in 64 bits."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(17, 1024, 6144), (17, 1024, 6208), (32, 4096, 6208), (33, 2048, 8192), (64, 1536, 8960),
                                   (24, 512, 18944), (32, 4096, 11008)])
def test_few_rows_long_k(m, n, k):
    import torch
    import llm_simple_amd.ops as ops
    for dt in (DT_FLOAT16, DT_BFLOAT16):
        x = normal_bits(m + k, (m, k), dt)
        w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
        ref = orc.widen(x, dt).astype(np.float64) @ orc.widen(w, dt).T.astype(np.float64)
        ref = orc.widen(orc.round_to(ref.astype(np.float32), dt), dt)
        args, out = (to_dev(x), to_dev(w), m, n, k, dt), to_dev(np.full((m, n), 0x7fff, dtype=np.uint16))
        torch.cuda.synchronize()
        ops.lib.llmhip_release_internal_workspace()
        free = torch.cuda.mem_get_info()[0]
        ops.hip_matmul_layer(out, *args)
        eager = to_host(out)
        # (a kernel's first launch takes 2 MiB for its code; the workspace of hipBLASLt alone is 64)
        assert torch.cuda.mem_get_info()[0] >= free - (16 << 20)
        got = orc.widen(eager, dt)
        # one rounding of an fp32 sum: a step of the storage type, 1e-3 where the sum cancels
        assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
            ops.hip_matmul_layer(out, *args, torch.cuda.current_stream().cuda_stream)
        for _ in range(2):
            out.fill_(0x7fff)
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(to_host(out), eager)
