"""How much per-stream scratch a chunk may ask for (no GPU: the sizes for 256 compute units)."""
import pytest


@pytest.mark.parametrize("H,Hkv", [(32, 32), (12, 2), (28, 4), (40, 8), (64, 1)])
def test_no_chunk_takes_more_than_256_mib(H, Hkv):
    import llm_simple_amd.ops as ops
    g, most = H // Hkv, 0
    for m in (17, 100, 512, 1165, 2276, 4096, 5912, 7151, 8192, 30000):
        for past in (m, 2 * m, 16384, 31536, 65536, 131072):
            need = ops.lib.llmhip_flash_attn_scratch_bytes(m, m + past, past, g, Hkv)
            assert need <= 256 << 20, (m, past, need)
            most = max(most, need)
    assert most > 16 << 20  # (long chunks still are cut)
