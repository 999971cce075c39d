// gemm.hip — fp32 C = A B on gfx950 matrix cores (matmul_threaded,
// src/threading.cpp:163-181): the tile kernel of gemm_f32.hpp at the tile
// that the shape asks for.
#include "gemm_f32.hpp"
#include "kernels.hpp"
#include "runtime.hpp"

namespace nut {

namespace {

template <int TI, int TJ, int WK, int NA, int D>
void launch_tile(const float *a, const float *b, float *c, int m, int k, int n,
                 hipStream_t stream)
{
    const int tiles_m = (m - 1) / (16 * TI) + 1, tiles_n = (n - 1) / (16 * TJ) + 1;
    // one dimension of a grid holds less than 2^32 threads
    const unsigned count = gemm_f32_grid(tiles_m, tiles_n), row = 1u << 22;
    const dim3 grid = count <= row ? dim3(count) : dim3(row, (count + row - 1) / row);
    hipLaunchKernelGGL((matmul_f32_wave<TI, TJ, WK, NA, D>), grid, dim3(64 * WK), 0, stream, a, b,
                       c, m, k, n, tiles_m, tiles_n);
}

} // namespace

void launch_matmul_f32(const float *a, const float *b, float *c, int m, int k,
                       int n, hipStream_t stream)
{
    const GemmTile t = gemm_f32_choose(m, k, n);
    // Eight waves per tile where the grid gives a CU one workgroup of a small
    // tile and k gives every wave a chunk (33 x 4001 x 3333: 25.7 us against
    // 30.4 with four), four elsewhere.
    // Two accumulators per output keep a chain of additions as short as eight
    // waves' (768^3: rel error 1.8e-7 against 2.5e-7 with one). The 64 x 64
    // tile has the registers for one: where it leaves CUs idle it has eight
    // waves for that (960 x 2048 x 960: 2.9e-7 against 4.1e-7 with four, at 43
    // and 41 us), or two accumulators where k has fewer than eight chunks.
    const bool deep = k >= 8 * kChunk, few = size_t(m / 64) * (n / 64) < 256;
    switch (t.ti * 10 + t.tj) {
    case 44:
        if (few)
            deep ? launch_tile<4, 4, 8, 1, 1>(a, b, c, m, k, n, stream)
                 : launch_tile<4, 4, 4, 2, 1>(a, b, c, m, k, n, stream);
        else
            launch_tile<4, 4, 4, 1, 1>(a, b, c, m, k, n, stream);
        break;
    case 34:
        launch_tile<3, 4, 4, 2, 2>(a, b, c, m, k, n, stream);
        break;
    case 33:
        launch_tile<3, 3, 4, 2, 2>(a, b, c, m, k, n, stream);
        break;
    case 24:
        launch_tile<2, 4, 4, 2, 2>(a, b, c, m, k, n, stream);
        break;
    case 22:
        deep && t.count <= 256 ? launch_tile<2, 2, 8, 2, 1>(a, b, c, m, k, n, stream)
                               : launch_tile<2, 2, 4, 2, 1>(a, b, c, m, k, n, stream);
        break;
    case 12:
        launch_tile<1, 2, 4, 2, 2>(a, b, c, m, k, n, stream);
        break;
    default:
        launch_tile<1, 1, 8, 2, 2>(a, b, c, m, k, n, stream);
    }
    check_launch("threaded matmul");
}

} // namespace nut
