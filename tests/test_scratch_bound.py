"""How much per-stream scratch a chunk may ask for, and the default counts of decode (no GPU: those for 256 compute units)."""
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


# 32 MiB of K and V are what the L2s hold: beyond, 64-row workgroups that all read everything take 62.7 us for 440 tokens
# over 3694 keys of 32 heads, with the key range cut in two 45.5; below, uncut is the fastest (315 over 1615: 23.2 us)
@pytest.mark.parametrize("m,past,H,Hkv,ranges", [(440, 3694, 32, 32, 2), (315, 1615, 32, 32, 1), (4, 131072, 40, 8, 32)])
def test_cut_of_a_chunk(m, past, H, Hkv, ranges):
    import llm_simple_amd.ops as ops
    need = ops.lib.llmhip_flash_attn_scratch_bytes(m, m + past, past, H // Hkv, Hkv)
    assert need == (0 if ranges == 1 else ranges * m * H * 130 * 4)


# (us of the fused step, which runs one workgroup to a CU, with the count for one / for two: 3072 keys of 66 kv heads 21.05 / 22.15, 2000 of 100 21.1 / 22.1)
@pytest.mark.parametrize("batch,n,Hkv,count", [(1, 3072, 66, 3), (1, 2000, 100, 2), (1, 2000, 88, 8), (2, 2000, 50, 5), (2, 3072, 33, 7)])
def test_counts_for_two_workgroups_to_a_cu_are_for_batches(batch, n, Hkv, count):
    import llm_simple_amd.ops as ops
    for other in (1, 2, batch):  # (as many pairs as before in one sequence or several)
        assert ops.flash_decode_default_splits(other, n, Hkv * batch // other) > 0
    assert ops.flash_decode_default_splits(batch, n, Hkv) == count
