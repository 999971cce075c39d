// gemm_f32.hpp — the fp32 matrix-core product shared by the standalone GEMM
// (gemm.hip) and the fp32 model path (fmodel.hip): C = A B with
// v_mfma_f32_16x16x4f32, fp32 inputs and accumulation.
//
// A wave computes a (16 TI) x (16 TJ) tile of C; the WK waves that share a
// tile each take a share of K, so that a tile's chain of products is spread
// over the SIMDs and small grids still fill them. B goes from memory
// straight to registers and A through a few KB of LDS of the wave's own
// (only to change its lane layout), in a ring of D chunks of 32 k: an fp32
// MFMA takes 32 cycles on a SIMD for one float of A and one of B per lane,
// which L2 delivers several times over, so no staging is shared and no
// barrier stands in the loop.
// In MFMA step s of a chunk, lane group g (lanes 16 g .. 16 g + 15) supplies
// k = 8 g + s of both operands: the k order inside a chunk is permuted alike
// for A and B. Columns are permuted too: column tile j of lane li is column
// TJ li + j, so a lane's B values of one k are TJ consecutive floats and so
// are its outputs. All vector accesses to memory are 4-byte aligned only
// (unaligned vector access is on for this target), so one kernel serves
// every row length. Rows past m read row m - 1, columns past n the last TJ
// columns; what they give is not stored. The k tail is read value by value
// and is zeros past the end. Partial tiles are added in LDS in a fixed order:
// the result does not depend on timing.
#pragma once

#include "device.hpp"

namespace nut {

typedef float floatx4 __attribute__((ext_vector_type(4)));

template <int N> struct VecU {
    typedef float type __attribute__((ext_vector_type(N), aligned(4)));
};
template <> struct VecU<1> {
    typedef float type;
};

template <int N> __device__ __forceinline__ void load_u(const float *p, float *out)
{
    if constexpr (N == 1) {
        out[0] = *p;
    } else {
        const typename VecU<N>::type v = *reinterpret_cast<const typename VecU<N>::type *>(p);
#pragma unroll
        for (int i = 0; i < N; i++)
            out[i] = v[i];
    }
}

template <int N> __device__ __forceinline__ void store_u(float *p, const float *in)
{
    if constexpr (N == 1) {
        *p = in[0];
    } else {
        typename VecU<N>::type v;
#pragma unroll
        for (int i = 0; i < N; i++)
            v[i] = in[i];
        *reinterpret_cast<typename VecU<N>::type *>(p) = v;
    }
}

constexpr int kChunk = 32;
constexpr int kChunkLd = 36; // floats per A row in LDS: 16-byte reads of 16
                             // rows fall in distinct banks

// One wave's share of a tile: acc += A B over the kChunk-wide chunks
// [c0, c1) and, when `tail`, the k values from kChunk (k / kChunk) on.
// pa[t]: row 8 t + lane / 8 of A at k = 4 (lane % 8), so that eight lanes
// read a whole 128-byte line (a lane per row, as the MFMA wants A, made
// every 16-byte piece a request of its own); the rows reach the fragment
// layout through `as`, 16 TI x kChunkLd floats of LDS of this wave alone.
// pb[q]: row 8 g of the q-th of NB operands, at this lane's first column of
// it (each supplies TJ / NB columns per lane). NORM: A's values are
// multiplied by nw[k] (nw at 4 (lane % 8)) and sq[t] gathers the squares of
// the values before that. NA: accumulators per output, each taking a run of
// a chunk's k (shorter chains of additions, a smaller rounding error); NA < 0:
// one accumulator, to which every chunk's own sum, formed in -NA chains, is
// added, the shortest chains of all.
// T: where the tail's code stands, if it is there at all. Before the loop, its
// loads are hidden behind the other waves' work (1612 x 207 x 1566: 21.4 us,
// 26.1 after it), but it takes registers, which a kernel with no loop to speak
// of has not to give (5236 x 5 x 7775: 62.3 us, 48.0 after it). A GEMM of whole
// chunks is faster without it (4096^3: 1,082 us, 1,118 with it before the loop).
enum class Tail { none, first, last };
constexpr int gemm_f32_accs(int na) { return na < 0 ? 1 : na; }

template <int TI, int TJ, int NB, int NA, int D, bool NORM, Tail T>
__device__ __forceinline__ void gemm_f32_run(const float *const (&pa)[2 * TI],
                                             const float *const (&pb)[NB], size_t ldb,
                                             const float *nw, int k, int c0, int c1, bool tail,
                                             float *as, floatx4 (&acc)[gemm_f32_accs(NA)][TI][TJ],
                                             float (&sq)[2 * TI])
{
    constexpr int TB = TJ / NB;
    static_assert(TB * NB == TJ, "columns split evenly over the operands");
    const int lane = threadIdx.x & 63;
    float *put = as + (lane >> 3) * kChunkLd + 4 * (lane & 7);
    const float *get = as + (lane & 15) * kChunkLd + 8 * (lane >> 4);
    float ra[D][2 * TI][4], rb[D][8][TJ], rn[D][4];
    const float *bp[NB];
    size_t ao = size_t(c0) * kChunk;
#pragma unroll
    for (int q = 0; q < NB; q++)
        bp[q] = pb[q] + size_t(c0) * kChunk * ldb;
    auto load = [&](int slot) {
#pragma unroll
        for (int t = 0; t < 2 * TI; t++)
            load_u<4>(pa[t] + ao, ra[slot][t]);
        if (NORM)
            load_u<4>(nw + ao, rn[slot]);
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int q = 0; q < NB; q++)
                load_u<TB>(bp[q] + s * ldb, &rb[slot][s][q * TB]);
        ao += kChunk;
#pragma unroll
        for (int q = 0; q < NB; q++)
            bp[q] += kChunk * ldb;
    };
    auto multiply = [&](float (&ga)[2 * TI][4], float (&fb)[8][TJ], float (&fn)[4]) {
        // LDS operations of one wave keep their order: no barrier
#pragma unroll
        for (int t = 0; t < 2 * TI; t++) {
            float4 v = make_float4(ga[t][0], ga[t][1], ga[t][2], ga[t][3]);
            if (NORM) {
                sq[t] = fmaf(v.x, v.x, sq[t]);
                sq[t] = fmaf(v.y, v.y, sq[t]);
                sq[t] = fmaf(v.z, v.z, sq[t]);
                sq[t] = fmaf(v.w, v.w, sq[t]);
                asm volatile("" : "+v"(sq[t])); // now: not with every chunk's values kept
                v.x *= fn[0];
                v.y *= fn[1];
                v.z *= fn[2];
                v.w *= fn[3];
            }
            *reinterpret_cast<float4 *>(put + 8 * t * kChunkLd) = v;
        }
        __builtin_amdgcn_wave_barrier();
        float fa[TI][8];
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4 v =
                    *reinterpret_cast<const float4 *>(get + 16 * i * kChunkLd + 4 * h);
                fa[i][4 * h] = v.x;
                fa[i][4 * h + 1] = v.y;
                fa[i][4 * h + 2] = v.z;
                fa[i][4 * h + 3] = v.w;
            }
        __builtin_amdgcn_wave_barrier();
        if constexpr (NA < 0) {
            constexpr int P = -NA;
            floatx4 part[P][TI][TJ];
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++)
                        part[s % P][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            fa[i][s], fb[s][j],
                            s < P ? floatx4{0.0f, 0.0f, 0.0f, 0.0f} : part[s % P][i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++) {
#pragma unroll
                    for (int step = 1; step < P; step *= 2)
#pragma unroll
                        for (int u = 0; u < P; u += 2 * step)
                            part[u][i][j] += part[u + step][i][j];
                    acc[0][i][j] += part[0][i][j];
                }
        } else {
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++)
                        acc[s * NA / 8][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            fa[i][s], fb[s][j], acc[s * NA / 8][i][j], 0, 0, 0);
        }
    };
    auto remainder = [&] {
        // every value is loaded, from the last k where it is past the end, and
        // replaced by a zero there: loads behind a condition each took as long
        // as several chunks
        const int kt = k & ~(kChunk - 1), k4 = 4 * (lane & 7), g8 = 8 * (lane >> 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int at = min(kt + k4 + e, k - 1) - k4;
#pragma unroll
            for (int t = 0; t < 2 * TI; t++)
                ra[0][t][e] = pa[t][at];
            if (NORM)
                rn[0][e] = nw[at];
        }
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const ptrdiff_t at = min(kt + g8 + s, k - 1) - g8;
#pragma unroll
            for (int q = 0; q < NB; q++)
                load_u<TB>(pb[q] + at * ptrdiff_t(ldb), &rb[0][s][q * TB]);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool in = kt + k4 + e < k;
#pragma unroll
            for (int t = 0; t < 2 * TI; t++)
                ra[0][t][e] = in ? ra[0][t][e] : 0.0f;
            if (NORM)
                rn[0][e] = in ? rn[0][e] : 0.0f;
        }
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
                rb[0][s][j] = kt + g8 + s < k ? rb[0][s][j] : 0.0f;
        multiply(ra[0], rb[0], rn[0]);
    };
    if (T == Tail::first && tail) // wave-uniform
        remainder();
    const int count = c1 - c0;
#pragma unroll
    for (int d = 0; d < D; d++)
        if (d < count)
            load(d);
    int q0 = 0;
    // whole rounds whose every slot loads again
    for (; q0 + 2 * D <= count; q0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            multiply(ra[d], rb[d], rn[d]);
            load(d);
        }
    }
    for (; q0 < count; q0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++)
            if (q0 + d < count) { // wave-uniform
                multiply(ra[d], rb[d], rn[d]);
                if (q0 + d + D < count)
                    load(d);
            }
    }
    if (T == Tail::last && tail)
        remainder();
}

// Chunks [c0, c1) of share `i` of `count` of k, and whether it takes the tail:
// the first, which has no more chunks than any other.
__device__ __forceinline__ void gemm_f32_share(int k, int i, int count, int &c0, int &c1,
                                               bool &tail)
{
    const int full = k / kChunk;
    c0 = int((long long)full * i / count);
    c1 = int((long long)full * (i + 1) / count);
    tail = i == 0 && k % kChunk != 0;
}

template <int TI, int TJ, int NA>
__device__ __forceinline__ void gemm_f32_clear(floatx4 (&acc)[NA][TI][TJ])
{
#pragma unroll
    for (int u = 0; u < NA; u++)
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
                acc[u][i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
}

// Adds the partial tiles of the WK waves that share a tile (`red`: theirs,
// WK * TJ * 256 floats of LDS; wk: this wave's place) and hands every output
// row's columns to epi(i, v, vals): row 16 i + 4 g + v of the tile, this
// lane's TJ columns, from wave v for each of the four v; called by the whole
// workgroup.
template <int TI, int TJ, int WK, int NS, class Epi>
__device__ __forceinline__ void gemm_f32_reduce(floatx4 (&parts)[NS][TI][TJ], float *red,
                                                int wk, Epi &&epi)
{
    static_assert(WK >= 4, "wave v takes element v");
    const int lane = threadIdx.x & 63;
    floatx4(&acc)[TI][TJ] = parts[0];
#pragma unroll
    for (int u = 1; u < NS; u++)
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
                acc[i][j] += parts[u][i][j];
#pragma unroll
    for (int i = 0; i < TI; i++) {
        if (i > 0)
            __syncthreads();
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                red[((wk * TJ + j) * 4 + v) * 64 + lane] = acc[i][j][v];
        __syncthreads();
        if (wk < 4) {
            float out[TJ];
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                float part[WK];
#pragma unroll
                for (int w = 0; w < WK; w++)
                    part[w] = red[((w * TJ + j) * 4 + wk) * 64 + lane];
#pragma unroll
                for (int step = 1; step < WK; step *= 2)
#pragma unroll
                    for (int w = 0; w < WK; w += 2 * step)
                        part[w] += part[w + step];
                out[j] = part[0];
            }
            epi(i, wk, out);
        }
    }
}

// Tile of this workgroup: workgroups go to the 8 XCDs round-robin, each XCD
// takes a contiguous run of the tiles, and the run goes through blocks of
// eight tile rows, so that the operands of the tiles an XCD has in flight
// share its L2. id: the workgroup's place in the grid. False for the grid's
// padding (gemm_f32_grid).
__device__ __forceinline__ bool gemm_f32_tile(int tiles_m, int tiles_n, unsigned id, int &tm,
                                              int &tn)
{
    const int tiles = tiles_m * tiles_n, per = (tiles + 7) / 8;
    const int t = int(id & 7) * per + int(id >> 3);
    if (int(id >> 3) >= per || t >= tiles)
        return false;
    const int group = t / (8 * tiles_n), in = t - group * 8 * tiles_n;
    const int rows = min(8, tiles_m - 8 * group);
    tm = 8 * group + in % rows;
    tn = in / rows;
    return true;
}

inline unsigned gemm_f32_grid(int tiles_m, int tiles_n)
{
    return unsigned((size_t(tiles_m) * tiles_n + 7) / 8 * 8);
}

// The tile (16 ti x 16 tj) that a shape takes least time with, by a model
// measured on this device: a CU runs ceil(tiles / 256) of them, each the
// MFMA cycles of the whole tile times what L2 traffic and the waves' own
// overhead add for that tile at 4096^3 (44: 1.24, 34: 1.39, 33: 1.31, 24:
// 1.45, 22: 1.48, 12: 1.8, 11: 2.4), plus a start and an end. Measured, the
// pick against the others: 768^3 33 12.1 us (44 18.6, 34 14.8, 22 16.3),
// 1000 x 2047 x 1531 34 66 us (44 80, 24 67, 22 72), 313^3 12 4.6 us (22 5.6,
// 44 12.6), 64 x 4096 x 256 11 10.5 us (12 13.4, 22 23.5), 4096^3 44
// 1,080 us (24 1,266, 22 1,340).
struct GemmTile {
    int ti, tj;
    double factor;
    long long count;
};

template <size_t N>
inline GemmTile gemm_f32_pick(const GemmTile (&tiles)[N], int m, int k, int n)
{
    GemmTile best{};
    double least = 0.0;
    for (const GemmTile &t : tiles) {
        if (n < t.tj)
            continue;
        const int rows = 16 * t.ti, cols = 16 * t.tj;
        const long long count =
            ((long long)m + rows - 1) / rows * (((long long)n + cols - 1) / cols);
        const double cycles =
            double((count + 255) / 256) * (double(rows) * cols * k / 128.0 * t.factor + 2000.0);
        if (best.count == 0 || cycles < least) {
            least = cycles;
            best = t;
            best.count = count;
        }
    }
    return best;
}

inline GemmTile gemm_f32_choose(int m, int k, int n)
{
    const GemmTile tiles[] = {{4, 4, 1.24, 0}, {3, 4, 1.39, 0}, {3, 3, 1.31, 0}, {2, 4, 1.45, 0},
                              {2, 2, 1.48, 0}, {1, 2, 1.8, 0},  {1, 1, 2.4, 0}};
    return gemm_f32_pick(tiles, m, k, n);
}

// C = A B, a tile per workgroup, whose WK waves share its k.
template <int TI, int TJ, int WK, int NA, int D, Tail T>
__global__ __launch_bounds__(64 * WK) void matmul_f32_wave(
    const float *__restrict__ a, const float *__restrict__ b, float *__restrict__ c, int m, int k,
    int n, int tiles_m, int tiles_n)
{
    // the waves' A chunks, then their partial tiles
    constexpr int kStage = WK * 16 * TI * kChunkLd;
    constexpr int kRed = WK * TJ * 256;
    __shared__ __attribute__((aligned(16))) float lds[kStage > kRed ? kStage : kRed];
    int tm, tn;
    if (!gemm_f32_tile(tiles_m, tiles_n, blockIdx.y * gridDim.x + blockIdx.x, tm, tn))
        return; // workgroup-uniform
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // rows and columns of the tile counted from its first: m and n may be as
    // large as an int holds
    const int row0 = tm * 16 * TI, rows = m - row0;
    const int col0 = tn * 16 * TJ, off = TJ * li, cols = n - col0;
    const int first = col0 + min(off, cols - TJ); // n >= TJ
    const float *pa[2 * TI];
#pragma unroll
    for (int t = 0; t < 2 * TI; t++)
        pa[t] = a + size_t(row0 + min(8 * t + (lane >> 3), rows - 1)) * k + 4 * (lane & 7);
    const float *pb[1] = {b + size_t(8 * g) * n + first};
    floatx4 acc[gemm_f32_accs(NA)][TI][TJ];
    float sq[2 * TI] = {};
    gemm_f32_clear(acc);
    int c0, c1;
    bool tail;
    gemm_f32_share(k, wave, WK, c0, c1, tail);
    gemm_f32_run<TI, TJ, 1, NA, D, false, T>(pa, pb, size_t(n), nullptr, k, c0, c1, tail,
                                             lds + wave * 16 * TI * kChunkLd, acc, sq);
    __syncthreads();
    gemm_f32_reduce<TI, TJ, WK>(
        acc, lds, wave,
        [&](int i, int v, const float (&out)[TJ]) {
            const int row = 16 * i + 4 * g + v;
            if (row >= rows || off >= cols)
                return;
            float *dst = c + size_t(row0 + row) * n + first;
            if (first == col0 + off) {
                store_u<TJ>(dst, out);
            } else {
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    if (first + j >= col0 + off)
                        dst[j] = out[j];
            }
        });
}

} // namespace nut
