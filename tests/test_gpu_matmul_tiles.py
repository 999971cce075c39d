"""The fp32 GEMM at the edges of its tiles.

Each shape is one where a tile, its k chunk or its last columns can go wrong:
fewer rows, columns or k than a tile, one more or less than a whole number of
them, and a ragged shape for every form that the launch chooses among
(tile_choice.py says which a shape takes, test_cpu_tiles.py that all are there).
The bound is that of any summation order in fp32: every output's error is at most
k 2^-23 sum |a b| (k fused steps of half an ulp each, doubled for the partial
sums' additions)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


SHAPES = [
    (1, 1, 1), (1, 33, 2), (3, 31, 3), (2, 64, 5), (17, 32, 16), (16, 33, 17),
    (15, 95, 31), (33, 4001, 130), (48, 257, 768), (768, 100, 768),
    (1000, 63, 1531), (313, 313, 313), (64, 1000, 63), (500, 65, 777),
    (65, 129, 4100), (2049, 40, 129),
    # 48 x 64; the widest tile with four waves, with eight and with two accumulators;
    # the 2 x 2 tile with eight waves and with four
    (1000, 65, 1531), (1757, 69, 849), (963, 291, 961), (967, 97, 953), (2145, 281, 33),
    (67, 69, 1747),
    # a tile to each wave (k < 64): its last rows and columns, one k, a whole
    # chunk, a chunk and one; the smallest grid that has it and one less
    (8191, 1, 1), (8129, 37, 15), (8200, 5, 16), (8177, 32, 17), (9001, 33, 32), (8321, 63, 33),
    (1, 47, 8190), (3, 31, 8195), (515, 32, 1030), (1000, 61, 1537),
    (1024, 63, 512), (1024, 63, 448), (1024, 64, 512),
]


@pytest.mark.parametrize("mkn", SHAPES)
def test_matmul_tile_edges(gpu, mkn):
    m, k, n = mkn
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    c = gpu.matmul_f32(a, b)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    bound = k * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(c - exact) <= bound)
    assert np.array_equal(gpu.matmul_f32(a, b), c)


def test_matmul_non_finite_rows_stay_apart(gpu):
    """A row of A or a column of B that holds a NaN or an infinity changes
    that row or column alone, at every ragged edge."""
    rng = np.random.default_rng(5)
    a = rng.standard_normal((37, 45)).astype(np.float32)
    b = rng.standard_normal((45, 51)).astype(np.float32)
    a[36, 44] = np.nan
    b[44, 50] = np.inf
    c = gpu.matmul_f32(a, b)
    assert np.all(np.isnan(c[36]))
    assert not np.any(np.isfinite(c[:, 50]))
    assert np.all(np.isfinite(c[:36, :50]))


def test_matmul_rows_past_one_grid_dimension(gpu):
    """More workgroups (64 rows each) than the launch puts into one dimension
    of a grid, 2^22: products of one term each, which are exact."""
    m = 270_000_000
    a = np.arange(m, dtype=np.float32)
    c = gpu.matmul_f32(a.reshape(m, 1), np.full((1, 1), 0.5, np.float32))
    assert np.array_equal(c.ravel(), 0.5 * a)
