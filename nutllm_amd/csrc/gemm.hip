// gemm.hip — fp32 C = A B on gfx950 matrix cores (matmul_threaded,
// src/threading.cpp:163-181): the tile kernel of gemm_f32.hpp at the tile
// that the shape asks for.
#include "gemm_f32.hpp"
#include "kernels.hpp"
#include "runtime.hpp"

namespace nut {

namespace {

// C = A B where k has fewer than two chunks: nothing to share among a tile's
// waves, whose partial tiles would take longer to add than to form. Each wave
// has 16 x (16 TJ) outputs of its own over all of k and stores them from its
// registers; four of them, one below the other, make a workgroup. Bound by the
// latency of a chunk's loads where the grid is small; a large one stores C at
// 2.3 TB/s (12000 x 63 x 12000: 252 us, 451 with four waves a tile), as each wave
// loads, multiplies and stores once. 16 x 32 outputs a wave took 341 us there,
// two by two waves a workgroup 255.
template <int TJ>
__global__ __launch_bounds__(256) void matmul_f32_shallow(const float *__restrict__ a,
                                                          const float *__restrict__ b,
                                                          float *__restrict__ c, int m, int k,
                                                          int n, int tiles_m, int tiles_n)
{
    __shared__ __attribute__((aligned(16))) float lds[4 * 16 * kChunkLd];
    int tm, tn;
    if (!gemm_f32_tile(tiles_m, tiles_n, blockIdx.y * gridDim.x + blockIdx.x, tm, tn))
        return;
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // counted from the tile: m and n may be as large as an int holds
    const int row0 = 64 * tm, rows = m - row0, r0 = 16 * wave;
    const int col0 = 16 * TJ * tn, cols = n - col0, off = TJ * li;
    if (r0 >= rows)
        return; // the whole wave; no barrier follows
    const int at = min(off, cols - TJ); // n >= TJ: from column n - TJ at the edge
    const float *pa[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
        pa[t] = a + size_t(row0 + min(r0 + 8 * t + (lane >> 3), rows - 1)) * k + 4 * (lane & 7);
    const float *pb[1] = {b + size_t(8 * g) * n + col0 + at};
    floatx4 acc[2][1][TJ];
    float sq[2] = {};
    gemm_f32_clear(acc);
    gemm_f32_run<1, TJ, 1, 2, 1, false, Tail::last>(pa, pb, size_t(n), nullptr, k, 0, k / kChunk,
                                                    k % kChunk != 0, lds + wave * 16 * kChunkLd,
                                                    acc, sq);
    if (off >= cols)
        return;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = r0 + 4 * g + v;
        if (row >= rows)
            continue;
        float out[TJ];
#pragma unroll
        for (int j = 0; j < TJ; j++)
            out[j] = acc[0][0][j][v] + acc[1][0][j][v];
        float *dst = c + size_t(row0 + row) * n + col0 + at;
        if (at == off) {
            store_u<TJ>(dst, out);
        } else {
#pragma unroll
            for (int j = 0; j < TJ; j++)
                if (at + j >= off) // the columns before are another lane's
                    dst[j] = out[j];
        }
    }
}

// One dimension of a grid holds less than 2^32 threads.
inline dim3 tile_grid(int tiles_m, int tiles_n)
{
    const unsigned count = gemm_f32_grid(tiles_m, tiles_n), row = 1u << 22;
    return count <= row ? dim3(count) : dim3(row, (count + row - 1) / row);
}

// The tail's code by k, in whole chunks or ragged; measured for each form.
template <int TI, int TJ, int WK, int NA, int D, Tail WHOLE = Tail::none, Tail RAGGED = Tail::first>
void launch_tile(const float *a, const float *b, float *c, int m, int k, int n,
                 hipStream_t stream)
{
    const int tiles_m = (m - 1) / (16 * TI) + 1, tiles_n = (n - 1) / (16 * TJ) + 1;
    const auto kernel = k % kChunk ? matmul_f32_wave<TI, TJ, WK, NA, D, RAGGED>
                                   : matmul_f32_wave<TI, TJ, WK, NA, D, WHOLE>;
    hipLaunchKernelGGL(kernel, tile_grid(tiles_m, tiles_n), dim3(64 * WK), 0, stream, a, b, c, m,
                       k, n, tiles_m, tiles_n);
}

template <int TJ>
void launch_shallow(const float *a, const float *b, float *c, int m, int k, int n,
                    hipStream_t stream)
{
    const int tiles_m = (m - 1) / 64 + 1, tiles_n = (n - 1) / (16 * TJ) + 1;
    hipLaunchKernelGGL((matmul_f32_shallow<TJ>), tile_grid(tiles_m, tiles_n), dim3(256), 0, stream,
                       a, b, c, m, k, n, tiles_m, tiles_n);
}

} // namespace

void launch_matmul_f32(const float *a, const float *b, float *c, int m, int k,
                       int n, hipStream_t stream)
{
    // Few chunks, many outputs: a tile to each wave (4000 x 30 x 3000: 20.0 us
    // against 34.3 with four waves a tile; 50000 x 8 x 4: 4.0 against 21.2). Not
    // from two chunks on, where waves that share k keep the chains of additions
    // shorter (1100 x 64 x 1100: rel error 8.3e-8 against 1.1e-7), and not where
    // the grid leaves half of the CUs idle (170 x 56 x 2366, 111 workgroups: 4.6
    // us against 4.4; 700 x 48 x 700, 121: 4.7 against 4.6).
    const int wide = n > 32 ? 4 : n > 16 ? 2 : 1; // column tiles of a wave
    if (k < 2 * kChunk && size_t((m - 1) / 64 + 1) * ((n - 1) / (16 * wide) + 1) >= 128) {
        wide == 4   ? launch_shallow<4>(a, b, c, m, k, n, stream)
        : wide == 2 ? launch_shallow<2>(a, b, c, m, k, n, stream)
                    : launch_shallow<1>(a, b, c, m, k, n, stream);
        check_launch("threaded matmul");
        return;
    }
    const GemmTile t = gemm_f32_choose(m, k, n);
    // Eight waves per tile where the grid gives a CU one workgroup of a small
    // tile and k gives every wave a chunk (33 x 4001 x 3333: 25.7 us against
    // 30.4 with four), four elsewhere.
    // Two accumulators per output keep a chain of additions as short as eight
    // waves' (768^3: rel error 1.8e-7 against 2.5e-7 with one). The 64 x 64
    // tile has the registers for one: where it leaves CUs idle it has eight
    // waves for that (960 x 2048 x 960: 2.9e-7 against 4.1e-7 with four, at 43
    // and 41 us), or two accumulators where k has fewer than eight chunks.
    // Where the tail's code stands changes the loop's schedule: 960 x 2048 x 960
    // 41.8 us with it last, 43.4 without; 64 x 4096 x 64 9.1 and 10.0; 33 x 4096
    // x 3333 24.7 us with it first, 28.6 without.
    const bool deep = k >= 8 * kChunk, few = size_t(m / 64) * (n / 64) < 256;
    switch (t.ti * 10 + t.tj) {
    case 44:
        if (few)
            deep ? launch_tile<4, 4, 8, 1, 1, Tail::last, Tail::last>(a, b, c, m, k, n, stream)
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
        deep && t.count <= 256
            ? launch_tile<2, 2, 8, 2, 1, Tail::first>(a, b, c, m, k, n, stream)
            : launch_tile<2, 2, 4, 2, 1>(a, b, c, m, k, n, stream);
        break;
    case 12:
        launch_tile<1, 2, 4, 2, 2>(a, b, c, m, k, n, stream);
        break;
    default:
        launch_tile<1, 1, 8, 2, 2, Tail::last, Tail::last>(a, b, c, m, k, n, stream);
    }
    check_launch("threaded matmul");
}

} // namespace nut
