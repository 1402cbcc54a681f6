"""Tiles that leave as whole rows: each tile size with a last row and a last column of tiles that are cut off, rows that are whole sectors
(past the L2) and rows that are not, by their width or by where the output begins.  Against sums in 64 bits; nothing beside the output changes."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

TILES = [(64, 64), (96, 64), (64, 96), (128, 64), (96, 96), (96, 128), (128, 96), (128, 128), (128, 160), (128, 192), (160, 160),
         (128, 224), (160, 192), (128, 256)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("tile_m,tile_n", TILES)
def test_rows(dt, tile_m, tile_n):
    import llm_simple_amd.ops as ops
    k = 64
    # 16 x 16 tiles; the last of each row holds 16 columns or 32, the last of each column of tiles all but 5 rows
    for n, offset in ((15 * tile_n + 16, 0), (15 * tile_n + 32, 0), (15 * tile_n + 32, 8), (15 * tile_n + 32, 32)):
        m = 16 * tile_m - 5
        x = normal_bits(m, (m, k), dt)
        w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
        ref = orc.widen(x, dt).astype(np.float64) @ orc.widen(w, dt).T.astype(np.float64)
        ref = orc.widen(orc.round_to(ref.astype(np.float32), dt), dt)
        nan = 0x7e00 if dt == DT_FLOAT16 else 0x7fc0
        flat = to_dev(np.full(64 + m * n + 64, nan, dtype=np.uint16))
        ops.hip_matmul_layer(flat[offset:offset + m * n].view(m, n), to_dev(x), to_dev(w), m, n, k, dt)
        got = to_host(flat)
        assert (got[:offset] == nan).all() and (got[offset + m * n:] == nan).all(), (n, offset)
        got = orc.widen(got[offset:offset + m * n].reshape(m, n), dt)
        # one rounding of an fp32 sum: a step of the storage type, 1e-3 where the sum cancels (a NaN fails the comparison)
        assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all(), (n, offset)
