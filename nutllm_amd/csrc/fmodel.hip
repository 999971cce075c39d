// fmodel.hip — the fp32 model path on gfx950: decode_token and
// prefill_tokens (src/kvcache.cpp:237-284) over the device KV cache, with
// ModelWeights' [in x out] fp32 projections resident in HBM.
//
// All tokens of a call go through a layer together, in five launches:
//   Q/K/V     rmsnorm prologue, RoPE, q and the K/V cache rows
//   attention causal, fp32 MFMA (a decode step: the split attention of the
//             quantised step kernels, step.hip)
//   Wo        added into the hidden rows
//   gate/up   rmsnorm prologue, silu(gate) * up
//   W2        added into the hidden rows
// The four projections are the fp32 matrix-core tile of gemm_f32.hpp with an
// epilogue of their own (fgemm_kernel). One token is a tile of one row: what
// the matrix cores do for the fifteen rows it leaves unused takes less time
// than the weights take from HBM (a 16-column tile takes 2 KB of weights in
// 256 cycles of a SIMD, 19 TB/s over the chip against the 6.2 of HBM).
// RMSNorm (src/ops.cpp:111-134) is folded in: the norm weights multiply A on
// its way to the tile, every wave gathers its share of the row's squares,
// and the row's factor 1 / sqrt(mean + 1e-5) multiplies the finished sums.
#include "fmodel.hpp"
#include "gemm_f32.hpp"
#include "prefill.hpp"
#include "project.hpp"
#include "runtime.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>

namespace nut {

namespace {

struct FGemm {
    const float *x, *norm_w; // rows [m][k], norm weights [k] (not kAdd)
    int m, k;
    // the matrices, [k][n] each: q, k, v (kQkv, column tiles in that order),
    // gate and up (kSwiglu, both in every tile) or the one (kAdd)
    const float *w[3];
    int n[3], tiles[3];
    int tiles_m, tiles_n;
    ProjectOut to;
    // kAdd: k in gridDim.y runs; run 0 adds to the hidden rows, run r stores
    // to parts + (r - 1) * m * n[0]
    float *parts;
};

template <int TI, int TJ, int WK, int D, int P, int EPI>
__global__ __launch_bounds__(64 * WK) void fgemm_kernel(FGemm f)
{
    constexpr bool NORM = EPI != kAdd;
    constexpr int NB = EPI == kSwiglu ? 2 : 1, TB = TJ / NB;
    constexpr int kStage = WK * 16 * TI * kChunkLd, kRed = WK * TJ * 256;
    __shared__ __attribute__((aligned(16))) float lds[kStage > kRed ? kStage : kRed];
    __shared__ float squares[NORM ? WK : 1][16 * TI];
    int tm, tn;
    if (!gemm_f32_tile(f.tiles_m, f.tiles_n, blockIdx.x, tm, tn))
        return; // workgroup-uniform
    int seg = 0;
    if (EPI == kQkv)
        while (seg < 2 && tn >= f.tiles[seg])
            tn -= f.tiles[seg++]; // workgroup-uniform
    const int n = f.n[seg], m = f.m, k = f.k;
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = tm * 16 * TI, col = tn * 16 * TB + TB * li;
    const int first = min(col, n - TB); // n >= TB
    const float *pa[2 * TI];
#pragma unroll
    for (int t = 0; t < 2 * TI; t++)
        pa[t] = f.x + size_t(min(row0 + 8 * t + (lane >> 3), m - 1)) * k + 4 * (lane & 7);
    const float *pb[NB];
#pragma unroll
    for (int q = 0; q < NB; q++)
        pb[q] = f.w[EPI == kSwiglu ? q : seg] + size_t(8 * g) * n + first;
    floatx4 acc[1][TI][TJ];
    float sq[2 * TI] = {};
    gemm_f32_clear(acc);
    int c0, c1;
    bool tail;
    const int run = EPI == kAdd ? blockIdx.y : 0, runs = EPI == kAdd ? gridDim.y : 1;
    gemm_f32_share(k, run * WK + wave, runs * WK, c0, c1, tail);
    // the tail's code first also where k has none: a prompt of 301 tokens over
    // four layers takes 1,971 us, 2,003 with it after the loop, 2,032 without it
    gemm_f32_run<TI, TJ, NB, -P, D, NORM, Tail::first>(
        pa, pb, size_t(n), NORM ? f.norm_w + 4 * (lane & 7) : nullptr, k, c0, c1, tail,
        lds + wave * 16 * TI * kChunkLd, acc, sq);
    if (NORM) {
        // eight lanes hold a row's squares of this wave's share
#pragma unroll
        for (int t = 0; t < 2 * TI; t++) {
            float s = sq[t];
            s += __shfl_xor(s, 1);
            s += __shfl_xor(s, 2);
            s += __shfl_xor(s, 4);
            if ((lane & 7) == 0)
                squares[wave][8 * t + (lane >> 3)] = s;
        }
    }
    __syncthreads();
    gemm_f32_reduce<TI, TJ, WK>(acc, lds, wave, [&](int i, int v, float (&out)[TJ]) {
        const int r = 16 * i + 4 * g + v, row = row0 + r;
        if (row >= m || col >= n)
            return;
        if constexpr (NORM) {
            const float scale = row_scale<WK>(squares, r, k);
#pragma unroll
            for (int j = 0; j < TJ; j++)
                out[j] *= scale;
        }
        if (EPI == kAdd && run > 0) {
            float *dst = f.parts + (size_t(run - 1) * m + row) * n + first;
#pragma unroll
            for (int j = 0; j < TJ; j++)
                if (first + j >= col)
                    dst[j] = out[j];
            return;
        }
        project_store<EPI, TJ>(f.to, seg, n, row, col, first, out);
    });
}

// h += the runs' products, in order; n floats a run.
__global__ __launch_bounds__(256) void add_parts_kernel(float *h, const float *parts, int count,
                                                        int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    float v = h[i];
    for (int p = 0; p < count; p++)
        v += parts[size_t(p) * n + i];
    h[i] = v;
}

template <int TI, int TJ, int WK, int D, int P, int EPI>
void launch_ftile(FGemm &f, hipStream_t stream, int runs = 1)
{
    const int cols = 16 * TJ / (EPI == kSwiglu ? 2 : 1);
    f.tiles_m = (f.m + 16 * TI - 1) / (16 * TI);
    f.tiles_n = 0;
    for (int s = 0; s < (EPI == kQkv ? 3 : 1); s++) {
        f.tiles[s] = (f.n[s] + cols - 1) / cols;
        f.tiles_n += f.tiles[s];
    }
    hipLaunchKernelGGL((fgemm_kernel<TI, TJ, WK, D, P, EPI>),
                       dim3(gemm_f32_grid(f.tiles_m, f.tiles_n), runs), dim3(64 * WK), 0, stream, f);
    check_launch("fp32 model: projection");
}

constexpr int kFRuns = 4; // most runs of k

// The tile by the model of gemm_f32_choose over all the launch's columns
// (gate and up count twice), with factors measured here, where the weights
// come from HBM and a chunk's sums are added apart: gate/up of 301 rows 24 176
// us (44 194, 34 187, 22 192, 14 202), of 64 22 49 (44 51, 24 59), of 20 24 31
// (44 50, 22 41); W2 of 301 rows 34 87 (44 110, 22 98), of 150 24 62 (34 87,
// 22 64), of 64 12 28 (22 37, 14 37); Q/K/V of 301 rows 14 38 (44 48, 24 47).
// A chunk's sum is formed in four chains (2 x 2: two) where the tile has the
// registers and the time for it, which is where narrow widths need it: their
// sums have few chunks (width 256 block 64, 70 tokens: error 2.4e-7 with one
// chain, 1.9e-7 so). More chains cost time: two at 14 and 24 made 301 tokens of
// four layers 2.15 ms instead of 2.00, four at 22 64 rows of two 334 us instead
// of 317, eight in a decode step's tiles two steps at 700 770 us instead of 680.
// Up to 16 rows the weights' way from HBM is what
// counts: sixteen waves share the k of a narrow tile, so that the whole chip
// has its loads in flight at once.
template <int EPI> void launch_fgemm(FGemm f, hipStream_t stream)
{
    int n = f.n[0];
    if (EPI == kQkv)
        n += f.n[1] + f.n[2];
    if (EPI == kSwiglu)
        n *= 2;
    if (f.m <= 16) {
        if constexpr (EPI == kAdd) {
            // k of a long product (W2) in runs, so that all CUs read whole
            // 128-byte lines of it: 46 MB 24 -> 14 us with the sums'
            // launch. A product as short as Wo takes as long either way.
            const int tiles = (n + 31) / 32;
            const int runs = std::min(kFRuns, 256 / tiles);
            if (f.parts != nullptr && runs > 1 && f.k >= 4096) {
                launch_ftile<1, 2, 8, 2, 4, EPI>(f, stream, runs);
                hipLaunchKernelGGL(add_parts_kernel, dim3((f.m * n + 255) / 256), dim3(256), 0,
                                   stream, f.to.out, f.parts, runs - 1, f.m * n);
                check_launch("fp32 model: sums");
                return;
            }
            n >= 4096 ? launch_ftile<1, 2, 16, 2, 4, EPI>(f, stream)
                      : launch_ftile<1, 1, 16, 3, 4, EPI>(f, stream);
        } else {
            // four chains spill here: from width 2048, where two are as good,
            // Q/K/V takes 13.7 us instead of 16
            n >= 8192     ? launch_ftile<1, 4, 8, 1, 4, EPI>(f, stream)
            : f.k >= 2048 ? launch_ftile<1, 2, 16, 2, 2, EPI>(f, stream)
                          : launch_ftile<1, 2, 16, 2, 4, EPI>(f, stream);
        }
        return;
    }
    const GemmTile tiles[] = {{4, 4, 1.6, 0},  {3, 4, 1.65, 0}, {2, 4, 1.65, 0},
                              {2, 2, 1.85, 0}, {1, 4, 1.95, 0}, {1, 2, 2.4, 0}};
    const GemmTile t = gemm_f32_pick(tiles, f.m, f.k, n);
    switch (t.ti * 10 + t.tj) {
    case 44:
        launch_ftile<4, 4, 4, 1, 1, EPI>(f, stream);
        break;
    case 34:
        launch_ftile<3, 4, 4, 1, 1, EPI>(f, stream);
        break;
    case 24:
        launch_ftile<2, 4, 4, 2, 1, EPI>(f, stream);
        break;
    case 22:
        launch_ftile<2, 2, 4, 2, 2, EPI>(f, stream);
        break;
    case 14:
        launch_ftile<1, 4, 4, 1, 1, EPI>(f, stream);
        break;
    default:
        launch_ftile<1, 2, 8, 2, 4, EPI>(f, stream);
    }
}

// Causal attention of a prompt's T rows (src/kvcache.cpp:102-130 for every
// row) on v_mfma_f32_16x16x4f32: one wave per (16 query rows, head), over
// blocks of KB keys. Scores S = Q K^T with both operands read as rows, lane
// group g holding dims [g HD / 4, (g + 1) HD / 4) of row li, so a lane's
// values are consecutive; the online softmax on S in registers (a score row
// is one 16-lane DPP row); P through LDS into the A layout; O += P V with V
// read as rows (lane li: dims TJ li ..). The next block's K and V loads are
// in flight while one block is used.
// A key past a row's own position has weight 0; where such a key's V is not
// finite (0 times it would not be 0) the block is summed key by key instead.
template <int HD>
__global__ __launch_bounds__(64) void fattention_kernel(const float *q, const float *k_layer,
                                                        const float *v_layer, float *ctx, int t,
                                                        int heads, int kv_heads, int max_seq,
                                                        float scale)
{
    constexpr int QS = HD / 4;             // dims per lane group
    constexpr int KT = HD == 128 ? 2 : 4;  // 16-key tiles per block
    constexpr int KB = 16 * KT;
    constexpr int TJ = HD / 16;            // output columns per lane
    constexpr int PLD = KB + 4;
    __shared__ __attribute__((aligned(16))) float ps[16 * PLD];
    const int lane = threadIdx.x, li = lane & 15, g = lane >> 4;
    const int head = blockIdx.x, kvh = head / (heads / kv_heads);
    // the last rows (the most keys) are dispatched first
    const int row0 = int(gridDim.y - 1 - blockIdx.y) * 16;
    const size_t ldq = size_t(heads) * HD;
    const float *kh = k_layer + size_t(kvh) * max_seq * HD;
    const float *vh = v_layer + size_t(kvh) * max_seq * HD;
    float qf[QS];
    {
        const float *src = q + size_t(min(row0 + li, t - 1)) * ldq + size_t(head) * HD + g * QS;
#pragma unroll
        for (int s = 0; s < QS; s += 4)
            load_u<4>(src + s, &qf[s]);
    }
    floatx4 o[TJ];
#pragma unroll
    for (int j = 0; j < TJ; j++)
        o[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float mx[4], sum[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        mx[v] = -INFINITY;
        sum[v] = 0.0f;
    }
    const int keys = min(row0 + 16, t); // keys any of the rows sees
    float kf[KT][QS], vf[KB / 4][TJ];
    auto load_k = [&](int b) {
#pragma unroll
        for (int u = 0; u < KT; u++) {
            const float *src = kh + size_t(min(b + 16 * u + li, t - 1)) * HD + g * QS;
#pragma unroll
            for (int s = 0; s < QS; s += 4)
                load_u<4>(src + s, &kf[u][s]);
        }
    };
    // key 16 u + 4 g + s of the block in vf[4 u + s]
    auto load_v = [&](int b) {
#pragma unroll
        for (int u = 0; u < KT; u++)
#pragma unroll
            for (int s = 0; s < 4; s++)
                load_u<TJ>(vh + size_t(min(b + 16 * u + 4 * g + s, t - 1)) * HD + TJ * li,
                           vf[4 * u + s]);
    };
    load_k(0);
    load_v(0);
    for (int b = 0; b < keys; b += KB) {
        floatx4 sc[KT], sd[KT];
#pragma unroll
        for (int u = 0; u < KT; u++)
            sc[u] = sd[u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < QS / 2; s++)
#pragma unroll
            for (int u = 0; u < KT; u++) {
                sc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[s], kf[u][s], sc[u], 0, 0, 0);
                sd[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[QS / 2 + s], kf[u][QS / 2 + s],
                                                             sd[u], 0, 0, 0);
            }
#pragma unroll
        for (int u = 0; u < KT; u++)
            sc[u] += sd[u];
        if (b + KB < keys)
            load_k(b + KB);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = row0 + 4 * g + v;
            float m = mx[v];
#pragma unroll
            for (int u = 0; u < KT; u++) {
                const float x = sc[u][v] * scale;
                sc[u][v] = b + 16 * u + li <= row ? x : -INFINITY;
                m = fmaxf(m, sc[u][v]);
            }
            m = row16_max(m);
            // no key with a score above -inf yet: weights 0, not NaN
            const float base = m == -INFINITY ? 0.0f : m;
            const float alpha = expf(mx[v] - base);
            mx[v] = m;
            float part = 0.0f;
#pragma unroll
            for (int u = 0; u < KT; u++) {
                const float e = expf(sc[u][v] - base);
                part += e;
                ps[(4 * g + v) * PLD + 16 * u + li] = e;
            }
            sum[v] = sum[v] * alpha + row16_sum(part);
#pragma unroll
            for (int j = 0; j < TJ; j++)
                o[j][v] *= alpha;
        }
        __syncthreads(); // one wave: orders the LDS accesses
        bool apart = false;
        if (b + KB > row0 + 1) { // wave-uniform: keys past some row
            bool finite = true;
#pragma unroll
            for (int e = 0; e < KB / 4; e++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    finite = finite && isfinite(vf[e][j]);
            apart = !__all(finite);
        }
        if (!apart) {
            float p[KT][4];
#pragma unroll
            for (int u = 0; u < KT; u++) {
                const float4 p4 =
                    *reinterpret_cast<const float4 *>(&ps[li * PLD + 16 * u + 4 * g]);
                p[u][0] = p4.x;
                p[u][1] = p4.y;
                p[u][2] = p4.z;
                p[u][3] = p4.w;
            }
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                floatx4 part[KT];
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int u = 0; u < KT; u++)
                        part[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            p[u][s], vf[4 * u + s][j],
                            s == 0 ? floatx4{0.0f, 0.0f, 0.0f, 0.0f} : part[u], 0, 0, 0);
#pragma unroll
                for (int u = 1; u < KT; u++)
                    part[0] += part[u];
                o[j] += part[0];
            }
        } else {
            for (int e = 0; e < KB && b + e < keys; e++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (b + e <= row0 + 4 * g + v)
#pragma unroll
                        for (int j = 0; j < TJ; j++)
                            o[j][v] = fmaf(ps[(4 * g + v) * PLD + e],
                                           vh[size_t(b + e) * HD + TJ * li + j], o[j][v]);
        }
        if (b + KB < keys)
            load_v(b + KB);
        __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = row0 + 4 * g + v;
        if (row < t) {
            float out[TJ];
#pragma unroll
            for (int j = 0; j < TJ; j++)
                out[j] = o[j][v] / sum[v];
            store_u<TJ>(ctx + size_t(row) * ldq + size_t(head) * HD + TJ * li, out);
        }
    }
}

template <int HD>
void launch_fattention(const DecodeShape &s, const float *q, const float *kc, const float *vc,
                       float *ctx, int t, hipStream_t stream)
{
    hipLaunchKernelGGL(fattention_kernel<HD>, dim3(s.heads, (t + 15) / 16), dim3(64), 0, stream,
                       q, kc, vc, ctx, t, s.heads, s.kv_heads, s.max_seq, s.attn_scale);
    check_launch("fp32 prefill: attention");
}

void check_fready(const nut_fmodel &m)
{
    require(m.globals_set, NUT_EINVAL, "kv cache: model weights not uploaded");
    for (const nut_fmodel::Layer &l : m.layers)
        require(l.set, NUT_EINVAL, "kv cache: layer count mismatch");
}

// One layer for t rows at positions first .. first + t - 1; `attend` puts
// the rows' context into ctx from q and the layer's cache. weights(i, n, w):
// w = the matrices i .. i + n - 1 (query, key, value, output, gate, up, down),
// asked for before each launch in turn. parts: room for kFRuns - 1 products of
// 16 rows, or null.
template <class Weights, class Attend>
void launch_layer(const DecodeShape &s, Weights &&weights, const float *attention_norm,
                  const float *ffn_norm, const float2 *rope, float *kc, float *vc, float *h,
                  float *q, float *ctx, float *act, float *parts, int t, int first,
                  hipStream_t stream, Attend &&attend)
{
    const int kvd = s.kv_heads * s.head_dim;
    FGemm f{};
    f.m = t;
    f.parts = parts;
    f.to = ProjectOut{nullptr, rope, kc, vc, first, s.head_dim, s.max_seq};
    auto gemm = [&](const float *x, const float *norm, int k, int w0, int count, int n0,
                    float *out) {
        f.x = x;
        f.norm_w = norm;
        f.k = k;
        weights(w0, count, f.w);
        for (int i = 0; i < count; i++)
            f.n[i] = i == 0 ? n0 : w0 == 0 ? kvd : n0;
        f.to.out = out;
    };
    gemm(h, attention_norm, s.dim, 0, 3, s.dim, q);
    launch_fgemm<kQkv>(f, stream);
    attend();
    gemm(ctx, nullptr, s.dim, 3, 1, s.dim, h);
    launch_fgemm<kAdd>(f, stream);
    gemm(h, ffn_norm, s.dim, 4, 2, s.ffn_dim, act);
    launch_fgemm<kSwiglu>(f, stream);
    gemm(act, nullptr, s.ffn_dim, 6, 1, s.dim, h);
    launch_fgemm<kAdd>(f, stream);
}

// The t tokens whose embeddings stand in h through every layer at positions
// first .. first + t - 1 (first == 0 unless t == 1); their hidden states
// stay in h.
void enqueue_layers(nut_fmodel &m, nut_kvcache &kv, float *h, int t, int first, float *q,
                    float *ctx, float *act)
{
    const DecodeShape &s = m.shape;
    const size_t layer_elems = kv.layer_elements();
    const StepState *state = m.state.as<StepState>();
    const int *length = kv.device_length.as<int>();
    for (size_t l = 0; l < m.config.layers; l++) {
        const nut_fmodel::Layer &L = m.layers[l];
        float *kc = kv.keys.as<float>() + l * layer_elems;
        float *vc = kv.values.as<float>() + l * layer_elems;
        const auto weights = [&](int i, int n, const float **w) {
            for (int j = 0; j < n; j++)
                w[j] = L.w[i + j].as<float>();
        };
        launch_layer(s, weights, L.attention_norm.as<float>(), L.ffn_norm.as<float>(),
                     m.rope.as<float2>(), kc, vc, h, q, ctx, act, m.parts.as<float>(), t, first,
                     m.stream, [&]() {
            if (t == 1 && m.split_attention) {
                launch_attention_split(s, q, kc, vc, length, m.attn_part.as<uint64_t>(),
                                       m.attn_count.as<int>(), ctx, state, m.stream);
            } else if (first == 0 && attention_f32_supported(s)) {
                launch_attention_f32(s, q, kc, vc, ctx, t, m.stream);
            } else {
                for (int i = 0; i < t; i++) {
                    if (t > 1)
                        launch_set_int(kv.device_length.as<int>(), first + i, m.stream);
                    launch_attention(s, q + size_t(i) * s.dim, kc, vc, length,
                                     ctx + size_t(i) * s.dim, state, m.stream);
                }
            }
        });
    }
}

// dense[c][r] = row r, column c of m as fp32 (code times scale, exact): the
// [in x out] layout of the projections here. A 32 x 32 tile per workgroup,
// transposed in LDS so that both sides are read and written in rows.
__global__ __launch_bounds__(256) void dense_kernel(QMat m, float *dense)
{
    __shared__ float tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
    for (int y = ty; y < 32; y += 8) {
        const int r = r0 + y, c = c0 + tx;
        if (r < m.rows && c < m.cols) {
            const size_t i = size_t(r) * m.cols + c;
            int q;
            if (m.type == 1)
                q = int(uint32_t(m.data[i >> 1]) << ((i & 1) ? 24 : 28)) >> 28;
            else
                q = int(int8_t(m.data[i]));
            tile[y][tx] = float(q) * half_bits_to_float(m.scales[i / m.block_size]);
        }
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
        const int r = r0 + tx, c = c0 + y;
        if (r < m.rows && c < m.cols)
            dense[size_t(c) * m.rows + r] = tile[tx][y];
    }
}

void check_cache(const nut_fmodel &m, const nut_kvcache &kv)
{
    require(config_valid(m.config), NUT_EINVAL, "model config: invalid dimensions");
    require(kv_compatible(kv, m.config), NUT_EINVAL, "kv cache: model configuration mismatch");
    check_fready(m);
}

void upload_to(DeviceBuffer &b, const float *src, size_t count)
{
    b.allocate(count * sizeof(float));
    hip_check(hipMemcpy(b.get(), src, count * sizeof(float), hipMemcpyHostToDevice),
              "hipMemcpy to device");
}

} // namespace

bool attention_f32_supported(const DecodeShape &s)
{
    return s.head_dim == 16 || s.head_dim == 32 || s.head_dim == 64 || s.head_dim == 128;
}

void launch_attention_f32(const DecodeShape &s, const float *q, const float *k_layer,
                          const float *v_layer, float *ctx, int t, hipStream_t stream)
{
    s.head_dim == 128  ? launch_fattention<128>(s, q, k_layer, v_layer, ctx, t, stream)
    : s.head_dim == 64 ? launch_fattention<64>(s, q, k_layer, v_layer, ctx, t, stream)
    : s.head_dim == 32 ? launch_fattention<32>(s, q, k_layer, v_layer, ctx, t, stream)
                       : launch_fattention<16>(s, q, k_layer, v_layer, ctx, t, stream);
}

size_t dense_group_floats(const DecodeShape &s)
{
    const size_t d = s.dim, kvd = size_t(s.kv_heads) * s.head_dim, f = s.ffn_dim;
    return std::max(d * d + 2 * d * kvd, 2 * d * f);
}

void launch_layer_dense(const DecodeShape &s, const LayerView &w, const float2 *rope,
                        float *k_layer, float *v_layer, const RowBuffers &b, int t, float *dense,
                        hipStream_t stream)
{
    const QMat *mats[7] = {&w.query, &w.key, &w.value, &w.output, &w.gate, &w.up, &w.down};
    // the launch before has read its matrices when the next ones are written
    const auto weights = [&](int i, int n, const float **at) {
        float *to = dense;
        for (int j = 0; j < n; j++) {
            const QMat &m = *mats[i + j];
            hipLaunchKernelGGL(dense_kernel, dim3((m.cols + 31) / 32, (m.rows + 31) / 32),
                               dim3(256), 0, stream, m, to);
            at[j] = to;
            to += size_t(m.rows) * m.cols;
        }
        check_launch("prefill: dense weights");
    };
    launch_layer(s, weights, w.attention_norm, w.ffn_norm, rope, k_layer, v_layer, b.hidden, b.query,
                 b.context, b.act, nullptr, t, 0, stream, [&]() {
        launch_attention_f32(s, b.query, k_layer, v_layer, b.context, t, stream);
    });
}

nut_fmodel *create_fmodel(const nut_config &config, bool tied)
{
    require(config_valid(config), NUT_EINVAL, "model config: invalid dimensions");
    require(config.head_dim % 4 == 0 && config.dim <= 65536 && config.ffn_dim <= 65536 &&
                config.max_seq <= 15000 && config.vocab_size <= 0x7fffffff,
            NUT_EINVAL, "fp32 model: shape exceeds device kernel limits");
    ensure_device();
    std::unique_ptr<nut_fmodel> m(new nut_fmodel());
    m->config = config;
    m->tied = tied;
    DecodeShape &s = m->shape;
    s.dim = int(config.dim);
    s.heads = int(config.heads);
    s.kv_heads = int(config.kv_heads == 0 ? config.heads : config.kv_heads);
    s.head_dim = int(config.head_dim);
    s.ffn_dim = int(config.ffn_dim);
    s.vocab = int(config.vocab_size);
    s.max_seq = int(config.max_seq);
    s.eos = int(config.eos_token);
    s.attn_scale = 1.0f / std::sqrt(float(config.head_dim));
    m->layers.resize(config.layers);
    const std::vector<float> rope = rope_table(config);
    upload_to(m->rope, rope.data(), rope.size());
    m->hidden.allocate(config.dim * sizeof(float));
    m->query.allocate(config.dim * sizeof(float));
    m->context.allocate(config.dim * sizeof(float));
    m->act.allocate(config.ffn_dim * sizeof(float));
    m->host.allocate(config.dim * sizeof(float));
    m->parts.allocate(size_t(kFRuns - 1) * 16 * config.dim * sizeof(float));
    m->state.allocate(sizeof(StepState));
    m->token.allocate(sizeof(int));
    hip_check(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "hipStreamCreate");
    // the attention kernels' stop flag: never set on this path
    launch_reset_state(m->state.as<StepState>(), 0, m->stream);
    m->split_attention = attention_split_supported(s);
    if (m->split_attention) {
        // one token's partial results (no word carries a live tag) and
        // arrival counters
        const size_t part = step_attn_part_words(s) / kStepTokensMax * sizeof(uint64_t);
        const size_t count = 2 * size_t(s.heads) * sizeof(int);
        m->attn_part.allocate(part);
        m->attn_count.allocate(count);
        hip_check(hipMemsetAsync(m->attn_part.get(), 0xff, part, m->stream), "hipMemsetAsync");
        hip_check(hipMemsetAsync(m->attn_count.get(), 0, count, m->stream), "hipMemsetAsync");
    }
    return m.release();
}

void set_fglobals(nut_fmodel &m, const float *embeddings, const float *final_norm,
                  const float *lm_head)
{
    require(embeddings != nullptr && final_norm != nullptr && (m.tied || lm_head != nullptr),
            NUT_EINVAL, "fp32 model: null weights");
    const size_t n = m.config.vocab_size * m.config.dim;
    upload_to(m.embeddings, embeddings, n);
    upload_to(m.final_norm, final_norm, m.config.dim);
    if (!m.tied)
        upload_to(m.lm_head, lm_head, n);
    m.globals_set = true;
}

void set_flayer(nut_fmodel &m, size_t layer, const float *const w[7],
                const float *attention_norm, const float *ffn_norm)
{
    const nut_config &c = m.config;
    require(layer < c.layers, NUT_EOUTOFRANGE, "fp32 model: layer out of range");
    require(attention_norm != nullptr && ffn_norm != nullptr, NUT_EINVAL,
            "fp32 model: null norm weights");
    const size_t kvd = (c.kv_heads == 0 ? c.heads : c.kv_heads) * c.head_dim;
    const size_t sizes[7] = {c.dim * c.dim,     c.dim * kvd,       c.dim * kvd, c.dim * c.dim,
                             c.dim * c.ffn_dim, c.dim * c.ffn_dim, c.ffn_dim * c.dim};
    nut_fmodel::Layer &L = m.layers[layer];
    for (int i = 0; i < 7; i++) {
        require(w[i] != nullptr, NUT_EINVAL, "fp32 model: null projection");
        upload_to(L.w[i], w[i], sizes[i]);
    }
    upload_to(L.attention_norm, attention_norm, c.dim);
    upload_to(L.ffn_norm, ffn_norm, c.dim);
    L.set = true;
}

void decode_token(nut_fmodel &m, nut_kvcache &kv, int token, float *hidden)
{
    check_cache(m, kv);
    require(kv.length < m.config.max_seq, NUT_ELENGTH, "kv cache: context is full");
    require(token >= 0 && size_t(token) < m.config.vocab_size, NUT_EOUTOFRANGE,
            "kv cache: token id out of range");
    kv.sync_length(m.stream);
    launch_set_int(m.token.as<int>(), token, m.stream);
    launch_embed_rows(m.embeddings.as<float>(), m.token.as<int>(), m.hidden.as<float>(), 1,
                      m.shape.dim, m.stream);
    enqueue_layers(m, kv, m.hidden.as<float>(), 1, int(kv.length), m.query.as<float>(),
                   m.context.as<float>(), m.act.as<float>());
    launch_copy_words(m.hidden.get(), m.host.as<float>(), m.config.dim, nullptr, nullptr,
                      m.stream);
    hip_check(hipStreamSynchronize(m.stream), "hipStreamSynchronize");
    if (hidden != nullptr)
        std::memcpy(hidden, m.host.as<float>(), m.config.dim * sizeof(float));
    kv.length += 1;
}

namespace {

// Rows of every activation for the longest prompt so far: false where there is
// no memory for them (token by token needs none).
bool reserve_rows(nut_fmodel &m, size_t count)
{
    if (count <= m.rows_held)
        return true;
    m.rows_held = 0;
    const size_t row = count * m.config.dim * sizeof(float);
    if (m.pf_tokens.try_allocate(count * sizeof(int)) && m.pf_h.try_allocate(row) &&
        m.pf_q.try_allocate(row) && m.pf_ctx.try_allocate(row) &&
        m.pf_act.try_allocate(count * m.config.ffn_dim * sizeof(float))) {
        m.rows_held = count;
        return true;
    }
    for (DeviceBuffer *b : {&m.pf_tokens, &m.pf_h, &m.pf_q, &m.pf_ctx, &m.pf_act})
        b->release();
    return false;
}

} // namespace

void prefill_tokens(nut_fmodel &m, nut_kvcache &kv, const int *tokens, size_t count,
                    float *rows)
{
    check_cache(m, kv);
    require(tokens != nullptr && count != 0 && count <= m.config.max_seq, NUT_EINVAL,
            "kv cache: invalid prefill length");
    kv.length = 0;
    // the reference embeds every token before the first layer, so a bad id
    // fails with nothing computed (src/kvcache.cpp:247-250)
    for (size_t t = 0; t < count; t++)
        require(tokens[t] >= 0 && size_t(tokens[t]) < m.config.vocab_size, NUT_EOUTOFRANGE,
                "kv cache: token id out of range");
    if (!reserve_rows(m, count)) {
        for (size_t t = 0; t < count; t++) {
            float *row = rows == nullptr ? nullptr : rows + t * m.config.dim;
            decode_token(m, kv, tokens[t], row);
        }
        return;
    }
    hip_check(hipMemcpyAsync(m.pf_tokens.get(), tokens, count * sizeof(int),
                             hipMemcpyHostToDevice, m.stream),
              "hipMemcpyAsync");
    launch_set_int(kv.device_length.as<int>(), 0, m.stream);
    launch_embed_rows(m.embeddings.as<float>(), m.pf_tokens.as<int>(), m.pf_h.as<float>(),
                      int(count), m.shape.dim, m.stream);
    enqueue_layers(m, kv, m.pf_h.as<float>(), int(count), 0, m.pf_q.as<float>(),
                   m.pf_ctx.as<float>(), m.pf_act.as<float>());
    if (rows != nullptr)
        hip_check(hipMemcpyAsync(rows, m.pf_h.get(), count * m.config.dim * sizeof(float),
                                 hipMemcpyDeviceToHost, m.stream),
                  "hipMemcpyAsync");
    hip_check(hipStreamSynchronize(m.stream), "hipStreamSynchronize");
    kv.length = count;
}

} // namespace nut

nut_fmodel::~nut_fmodel()
{
    if (stream != nullptr)
        (void)hipStreamDestroy(stream);
}
