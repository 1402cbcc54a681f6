"""Tiles that leave as whole rows, each tile shown to be the one that runs: a last row and a last column of tiles that are cut off, rows that are whole sectors
and rows that are not, by their width or by where the output begins.  Against sums in 64 bits; nothing beside the output changes."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# (16 x 16 tiles each; of 64 x 96, before which 96 x 64 is tried, the last one lacks 16 or 32 columns, of the others it has 16 or 32)
SIZES = [(64, 64), (96, 64), (64, 96), (128, 64), (96, 96), (96, 128), (128, 96), (128, 128), (128, 160), (128, 192), (160, 160),
         (128, 224), (160, 192), (128, 256)]


@pytest.mark.parametrize("tile_m,tile_n", SIZES)
def test_tile(tile_m, tile_n):
    import llm_simple_amd.bench_ops as bops
    for last in (80, 64) if (tile_m, tile_n) == (64, 96) else (16, 32):
        assert bops.lib.llmhip_bench_matmul_tile(16 * tile_m - 5, 15 * tile_n + last, 64) == tile_m << 16 | tile_n


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("n,offset", [(1520, 0), (1504, 0), (1504, 8), (1504, 32)])
def test_rows_of_64_x_96(dt, n, offset):
    import llm_simple_amd.bench_ops as bops
    import llm_simple_amd.ops as ops
    m, k = 1019, 64
    assert bops.lib.llmhip_bench_matmul_tile(m, n, k) == 64 << 16 | 96
    x = normal_bits(m, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    ref = orc.widen(x, dt).astype(np.float64) @ orc.widen(w, dt).T.astype(np.float64)
    ref = orc.widen(orc.round_to(ref.astype(np.float32), dt), dt)
    nan = 0x7e00 if dt == DT_FLOAT16 else 0x7fc0
    flat = to_dev(np.full(64 + m * n + 64, nan, dtype=np.uint16))
    ops.hip_matmul_layer(flat[offset:offset + m * n].view(m, n), to_dev(x), to_dev(w), m, n, k, dt)
    got = to_host(flat)
    assert (got[:offset] == nan).all() and (got[offset + m * n:] == nan).all()
    got = orc.widen(got[offset:offset + m * n].reshape(m, n), dt)
    # one rounding of an fp32 sum: a step of the storage type, 1e-3 where the sum cancels (a NaN fails the comparison)
    assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
