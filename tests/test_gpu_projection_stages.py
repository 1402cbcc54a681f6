"""Every tile shape of the projection kernel at the values of k where its pipeline can go wrong: a single line of k, fewer
lines than are kept in flight, as many, one more, and stages of four lines with one to three of them in use; the last
rows and features of a tile missing.  Against sums in 64 bits on the CPU."""
import numpy as np
import pytest

from helpers import DT_BFLOAT16, DT_FLOAT16, f32_dev, normal_bits, to_dev, to_host, ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# (rows and features of the tile, lhs rows and features of a call that takes it on 256 compute units, lines kept in flight)
TILES = [((32, 32), (31, 4112), 16), ((64, 32), (61, 8176), 12), ((64, 64), (129, 5360), 9), ((96, 64), (191, 8176), 7),
         ((128, 64), (381, 5104), 6), ((96, 96), (287, 8160), 6), ((96, 128), (191, 16368), 5),
         ((128, 96), (1000, 3072), 5), ((128, 128), (1023, 4080), 4), ((128, 160), (1023, 5104), 4),
         ((128, 192), (1153, 4784), 3), ((160, 160), (159, 40944), 3), ((128, 224), (1025, 6256), 3),
         ((160, 192), (319, 24560), 3), ((128, 256), (127, 65520), 3)]


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("tile,size,depth", TILES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_stages(tile, size, depth, dt):
    import llm_simple_amd.ops as ops
    m, n = size
    for lines in sorted({1, 2, depth - 1, depth, depth + 1, 2 * depth + 3}):
        k = 64 * lines
        x = normal_bits(m + k, (m, k), dt)
        w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
        b = np.random.default_rng(n).standard_normal(n).astype(np.float32) if lines % 2 else None
        rows = np.unique(np.r_[:17, m // 2 - 3:m // 2 + 3, m - 17:m])  # compared with the 64-bit sums; all rows are written
        ref = orc.widen(x, dt)[rows].astype(np.float64) @ orc.widen(w, dt).T.astype(np.float64) + (0.0 if b is None else b)
        ref = orc.widen(orc.round_to(ref.astype(np.float32), dt), dt)
        d_out = to_dev(np.full((m, n), 0x7e00 if dt == DT_FLOAT16 else 0x7fc0, dtype=np.uint16))  # NaN
        if b is None:
            ops.hip_matmul_layer(d_out, to_dev(x), to_dev(w), m, n, k, dt)
        else:
            ops.hip_matmul_bias_layer(d_out, to_dev(x), to_dev(w), f32_dev(b), m, n, k, dt)
        got = orc.widen(to_host(d_out), dt)
        assert np.isfinite(got).all(), lines
        # one rounding of an fp32 sum: a step of the storage type, 1e-3 where the sum cancels
        assert (np.abs(got[rows] - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all(), lines


@pytest.mark.parametrize("dt", [DT_FLOAT16, DT_BFLOAT16])
@pytest.mark.parametrize("m,n,k", [(9, 2048, 320), (9, 2064, 320), (16, 2064, 64), (8, 2064, 128), (13, 3584, 704),
                                   (11, 4096, 320), (12, 4096, 320), (9, 4112, 320), (8, 4112, 320), (10, 3328, 7232),
                                   (11, 3328, 7232), (11, 3328, 7168), (16, 2064, 7232), (8, 4112, 7232)])
def test_few_rows_line(dt, m, n, k):
    """Up to 16 rows, either side of the lines from which the tiles take such calls: 8 rows; 4096 features; rows times features
    per compute unit of 190, and of 130 where k is beyond 7168."""
    import llm_simple_amd.ops as ops
    x = normal_bits(m + k, (m, k), dt)
    w = orc.round_to(orc.widen(normal_bits(n, (n, k), dt), dt) / np.sqrt(k), dt)
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ref = orc.widen(orc.matmul_bias(x, w, b, dt), dt)
    d_out = to_dev(np.zeros((m, n), dtype=np.uint16))
    ops.hip_matmul_bias_layer(d_out, to_dev(x), to_dev(w), f32_dev(b), m, n, k, dt)
    got = orc.widen(to_host(d_out), dt)
    assert (np.abs(got - ref) <= np.maximum(1.01 * ulp(ref, dt), 1e-3)).all()
