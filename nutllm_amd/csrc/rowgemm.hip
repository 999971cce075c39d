// rowgemm.hip — a short prompt's projections (prefill_quantized,
// src/quant_model.cpp:208-220, a few dozen tokens at once).
//
// Up to kRowGemmMax rows a layer's weights are read once, and what counts is
// that the whole chip has its loads in flight (TinyLlama INT4, a layer of 20
// tokens: 104 us on the step kernels, which dot every row once a token, 141
// in the batched GEMM's 64 x 128 tiles, 73 here; 16 tokens 88 -> 49): 16 TJ
// outputs per workgroup, its WK waves sharing k, so that a 2,048-wide matrix
// is 64 to 128 workgroups of 8 or 16 waves. Codes are
// exact in bf16 and an fp32 activation is the sum of three bf16 limbs
// without a remainder (8 bits each, fp32's own exponent range, so rows that
// are not normalised yet may be of any size and RMSNorm needs no pass of its
// own); products on v_mfma_f32_16x16x32_bf16, whose K = 32 is one quant
// block, the block's scale applied in fp32. Two f16 limbs, as the batched
// GEMM has them for its normalised rows, are one product less but lose small
// rows to f16's subnormals (100 tokens through 12 layers: error 3.5e-6; so,
// 6 to 64 tokens, 6.3e-7 to 8.7e-7) and large ones to its range.
//
// Weights go from memory to registers: lane (li, g) (li = lane % 16, g =
// lane / 16) loads 16 bytes of output row TJ li + j, 64 consecutive bytes a
// row over the four lane groups, and permlane swaps turn "a lane group per
// block" into "an eighth of k per lane group" (INT4: four blocks by a 4 x 4
// transpose; INT8: two blocks by one swap, which leaves k in the order 0,
// 16, 8, 24 of eights, and the activations are read in that order too).
// Activations go through a few KB of LDS of the wave's own, as in
// gemm_f32.hpp, whose reduction over the waves and whose epilogues this
// shares.
#include "kernels.hpp"
#include "project.hpp"
#include "runtime.hpp"

namespace nut {

namespace {

constexpr int kRun = 128; // k per step: four quant blocks

struct RowGemm {
    const float *x, *norm_w; // rows [m][k], norm weights [k] (not kAdd)
    int m, k;
    QMat w[3]; // q, k, v; gate, up; or one
    int tiles[3];
    int tiles_m, tiles_n;
    ProjectOut to;
};

__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// One output row's 128 weights as loaded: INT4 one 16-byte piece a lane
// (lane group g: block g), INT8 two (pieces g of the first and second two
// blocks); and its four scales.
template <int QT> struct Codes {
    uint4 raw[QT == 1 ? 1 : 2];
    uint2 scales;
};

template <int QT>
__device__ __forceinline__ void load_codes(const uint8_t *data, const uint16_t *scales,
                                           uint32_t row, uint32_t scale, uint32_t c, Codes<QT> &o)
{
#pragma unroll
    for (uint32_t h = 0; h < (QT == 1 ? 1 : 2); h++)
        o.raw[h] = *reinterpret_cast<const uint4 *>(data + (row + c * (QT == 1 ? 64 : 128) +
                                                            64 * h));
    o.scales = *reinterpret_cast<const uint2 *>(scales + (scale + 4 * c));
}

// In place: block b's codes of this lane's k in out[b].
template <int QT>
__device__ __forceinline__ void spread_codes(const Codes<QT> &in, uint2 (&out)[4])
{
    if constexpr (QT == 1) {
        uint32_t d0 = in.raw[0].x, d1 = in.raw[0].y, d2 = in.raw[0].z, d3 = in.raw[0].w;
        swap32(d0, d2);
        swap32(d1, d3);
        swap16(d0, d1);
        swap16(d2, d3);
        out[0] = make_uint2(d0, 0u);
        out[1] = make_uint2(d1, 0u);
        out[2] = make_uint2(d2, 0u);
        out[3] = make_uint2(d3, 0u);
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t a0 = in.raw[h].x, a1 = in.raw[h].y, b0 = in.raw[h].z, b1 = in.raw[h].w;
            swap32(a0, b0);
            swap32(a1, b1);
            out[2 * h] = make_uint2(a0, a1);
            out[2 * h + 1] = make_uint2(b0, b1);
        }
    }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The top halves of two fp32 values as two bf16 (a in the low half).
__device__ __forceinline__ uint32_t top_halves(float a, float b)
{
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// Eight codes (INT8: 8 bytes, INT4: 4, even k in the low nibble) as bf16:
// whole numbers of at most 8 bits, whose fp32 form ends in zeros.
template <int QT> __device__ __forceinline__ bf16x8 codes_bf16(uint2 raw)
{
    uint32_t out[4];
    if constexpr (QT == 1) {
        const uint32_t t = raw.x ^ 0x88888888u;
        const uint32_t lo = opaque(t & 0x0f0f0f0fu), hi = opaque((t >> 4) & 0x0f0f0f0fu);
        out[0] = top_halves(ubyte0(lo) - 8.0f, ubyte0(hi) - 8.0f);
        out[1] = top_halves(ubyte1(lo) - 8.0f, ubyte1(hi) - 8.0f);
        out[2] = top_halves(ubyte2(lo) - 8.0f, ubyte2(hi) - 8.0f);
        out[3] = top_halves(ubyte3(lo) - 8.0f, ubyte3(hi) - 8.0f);
    } else {
        const uint32_t w[2] = {raw.x ^ 0x80808080u, raw.y ^ 0x80808080u};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            out[2 * h] = top_halves(ubyte0(w[h]) - 128.0f, ubyte1(w[h]) - 128.0f);
            out[2 * h + 1] = top_halves(ubyte2(w[h]) - 128.0f, ubyte3(w[h]) - 128.0f);
        }
    }
    return __builtin_bit_cast(bf16x8, make_uint4(out[0], out[1], out[2], out[3]));
}

// v without its low 16 bits: the bf16 limb of v, as fp32.
__device__ __forceinline__ float top_limb(float v)
{
    return __uint_as_float(__float_as_uint(v) & 0xffff0000u);
}

template <int QT, int TI, int TJ, int WK, int EPI>
__global__ __launch_bounds__(64 * WK) void rowgemm_kernel(RowGemm f)
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
    const int n = f.w[seg].rows, m = f.m, k = f.k;
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = tm * 16 * TI, col = tn * 16 * TB + TB * li;
    const int first = min(col, n - TB); // n >= TB
    // 32-bit offsets from the matrices' (uniform) bases: a matrix holds at
    // most 15,000 x 15,000 weights, the activations kRowGemmMax rows
    const QMat &q0 = f.w[seg], &q1 = f.w[EPI == kSwiglu ? 1 : seg];
    uint32_t wo[TB], so[TB];
#pragma unroll
    for (int j = 0; j < TB; j++) {
        wo[j] = uint32_t(first + j) * (QT == 1 ? uint32_t(k) / 2 : uint32_t(k)) + 16 * g;
        so[j] = uint32_t(first + j) * (uint32_t(k) / 32);
    }
    auto load_w = [&](int c, Codes<QT> (&o)[TJ]) {
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const QMat &q = j < TB ? q0 : q1;
            load_codes<QT>(q.data, q.scales, wo[j % TB], so[j % TB], uint32_t(c), o[j]);
        }
    };
    // activations: 8 rows a load, 128 bytes each (see gemm_f32_run)
    uint32_t xo[2 * TI];
#pragma unroll
    for (int t = 0; t < 2 * TI; t++)
        xo[t] = uint32_t(min(row0 + 8 * t + (lane >> 3), m - 1)) * uint32_t(k) + 4 * (lane & 7);
    const uint32_t no = 4 * (lane & 7);
    float *stage = lds + wave * 16 * TI * kChunkLd;
    float *put = stage + (lane >> 3) * kChunkLd + 4 * (lane & 7);
    const int eighth = QT == 1 ? g : (g & 1) * 2 + (g >> 1);
    const float *get = stage + li * kChunkLd + 8 * eighth;

    floatx4 acc[1][TI][TJ];
    gemm_f32_clear(acc);
    float sq[2 * TI] = {};
    const int runs = k / kRun;
    const int c0 = runs * wave / WK, c1 = runs * (wave + 1) / WK;
    Codes<QT> cur[TJ], next[TJ];
    // two blocks of activations in flight
    float4 ra[2][2 * TI], rn[2];
    auto load_x = [&](int slot, uint32_t at) {
#pragma unroll
        for (int t = 0; t < 2 * TI; t++)
            ra[slot][t] = *reinterpret_cast<const float4 *>(f.x + (xo[t] + at));
        if (NORM)
            rn[slot] = *reinterpret_cast<const float4 *>(f.norm_w + (no + at));
    };
    if (c0 < c1) {
        load_w(c0, cur);
        load_x(0, uint32_t(c0) * kRun);
        load_x(1, uint32_t(c0) * kRun + 32);
    }
    for (int c = c0; c < c1; c++) {
        const bool more = c + 1 < c1; // wave-uniform
        if (more)
            load_w(c + 1, next);
        uint2 codes[TJ][4];
#pragma unroll
        for (int j = 0; j < TJ; j++)
            spread_codes<QT>(cur[j], codes[j]);
#pragma unroll
        for (int b = 0; b < 4; b++) {
#pragma unroll
            for (int t = 0; t < 2 * TI; t++) {
                float4 v = ra[b & 1][t];
                if (NORM) {
                    sq[t] = fmaf(v.x, v.x, sq[t]);
                    sq[t] = fmaf(v.y, v.y, sq[t]);
                    sq[t] = fmaf(v.z, v.z, sq[t]);
                    sq[t] = fmaf(v.w, v.w, sq[t]);
                    asm volatile("" : "+v"(sq[t]));
                    v.x *= rn[b & 1].x;
                    v.y *= rn[b & 1].y;
                    v.z *= rn[b & 1].z;
                    v.w *= rn[b & 1].w;
                }
                *reinterpret_cast<float4 *>(put + 8 * t * kChunkLd) = v;
            }
            if (b < 2 || more)
                load_x(b & 1, uint32_t(c) * kRun + 32 * (b + 2));
            __builtin_amdgcn_wave_barrier(); // a wave's LDS accesses keep their order
            bf16x8 w[TJ];
            float s[TJ];
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                w[j] = codes_bf16<QT>(codes[j][b]);
                const uint32_t pair = b < 2 ? cur[j].scales.x : cur[j].scales.y;
                s[j] = half_bits_to_float(uint16_t(b & 1 ? pair >> 16 : pair));
            }
#pragma unroll
            for (int i = 0; i < TI; i++) {
                const float4 u = *reinterpret_cast<const float4 *>(get + 16 * i * kChunkLd);
                const float4 v = *reinterpret_cast<const float4 *>(get + 16 * i * kChunkLd + 4);
                float e[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
                // The large limbs first: the MFMA cuts off the low bits of a
                // small C towards minus infinity when it adds large products
                // to it (small limbs first, every sum was 0.2 of its error
                // too low on average: an error that is the same in all rows,
                // which attention over many of them does not average out).
                floatx4 d[TJ];
#pragma unroll
                for (int l = 0; l < 3; l++) {
                    uint32_t packed[4];
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        packed[q] = top_halves(e[2 * q], e[2 * q + 1]);
                    const bf16x8 limb = __builtin_bit_cast(
                        bf16x8, make_uint4(packed[0], packed[1], packed[2], packed[3]));
#pragma unroll
                    for (int j = 0; j < TJ; j++) {
                        d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            limb, w[j], l > 0 ? d[j] : floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    }
                    if (l < 2) {
#pragma unroll
                        for (int q = 0; q < 8; q++)
                            e[q] -= top_limb(e[q]);
                    }
                }
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        acc[0][i][j][q] = fmaf(s[j], d[j][q], acc[0][i][j][q]);
            }
            __builtin_amdgcn_wave_barrier();
            // without this and the one on sq the compiler keeps several
            // blocks' operands at once, and spills
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) {
#pragma unroll
            for (int j = 0; j < TJ; j++)
                cur[j] = next[j];
        }
    }
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
        project_store<EPI, TJ>(f.to, seg, n, row, col, first, out);
    });
}

template <int QT, int TI, int TJ, int WK, int EPI> void launch_tile(RowGemm &f, hipStream_t stream)
{
    const int cols = 16 * TJ / (EPI == kSwiglu ? 2 : 1);
    f.tiles_m = (f.m + 16 * TI - 1) / (16 * TI);
    f.tiles_n = 0;
    for (int s = 0; s < (EPI == kQkv ? 3 : 1); s++) {
        f.tiles[s] = (f.w[s].rows + cols - 1) / cols;
        f.tiles_n += f.tiles[s];
    }
    hipLaunchKernelGGL((rowgemm_kernel<QT, TI, TJ, WK, EPI>),
                       dim3(gemm_f32_grid(f.tiles_m, f.tiles_n)), dim3(64 * WK), 0, stream, f);
    check_launch("prefill rows: projection");
}

// Rows per tile by the prompt: 16, or 32 and as many tiles as it takes (64
// rows a tile, half the waves in flight, took 2.56 ms for 64 tokens of
// TinyLlama INT4 where two tiles of 32 take 1.83). Outputs per tile by the
// launch's width, to keep every matrix over 64 workgroups and more.
template <int QT, int EPI> void launch_rows(RowGemm f, hipStream_t stream)
{
    const int n = f.w[0].rows;
    if constexpr (EPI == kAdd) {
        // prompts of more than 16 rows come here at widths below 4096 only
        n >= 4096   ? launch_tile<QT, 1, 2, 16, EPI>(f, stream)
        : f.m <= 16 ? launch_tile<QT, 1, 1, 16, EPI>(f, stream)
                    : launch_tile<QT, 2, 1, 8, EPI>(f, stream);
        return;
    }
    if constexpr (EPI == kSwiglu) {
        if (n >= 2048 && f.m <= 16) {
            launch_tile<QT, 1, 4, 8, EPI>(f, stream);
            return;
        }
    }
    f.m <= 16 ? launch_tile<QT, 1, 2, 16, EPI>(f, stream)
              : launch_tile<QT, 2, 2, 8, EPI>(f, stream);
}

template <int EPI> void launch_rows_q(const RowGemm &f, hipStream_t stream)
{
    f.w[0].type == 1 ? launch_rows<1, EPI>(f, stream) : launch_rows<0, EPI>(f, stream);
}

} // namespace

bool row_gemm_supported(const DecodeShape &s, const LayerView &w)
{
    const QMat *mats[7] = {&w.query, &w.key, &w.value, &w.output, &w.gate, &w.up, &w.down};
    for (const QMat *m : mats)
        if (m->block_size != 32 || m->cols % kRun != 0 || m->type != w.query.type)
            return false;
    return attention_f32_supported(s);
}

void launch_layer_rows(const DecodeShape &s, const LayerView &w, const float2 *rope,
                       float *k_layer, float *v_layer, const RowBuffers &b, int t,
                       hipStream_t stream)
{
    require(t >= 1 && t <= kRowGemmMax, NUT_EINVAL, "prefill rows: token count out of range");
    RowGemm f{};
    f.m = t;
    f.to = ProjectOut{b.query, rope, k_layer, v_layer, 0, s.head_dim, s.max_seq};
    f.x = b.hidden;
    f.norm_w = w.attention_norm;
    f.k = s.dim;
    f.w[0] = w.query;
    f.w[1] = w.key;
    f.w[2] = w.value;
    launch_rows_q<kQkv>(f, stream);
    launch_attention_f32(s, b.query, k_layer, v_layer, b.context, t, stream);
    f.x = b.context;
    f.w[0] = w.output;
    f.to.out = b.hidden;
    launch_rows_q<kAdd>(f, stream);
    f.x = b.hidden;
    f.norm_w = w.ffn_norm;
    f.w[0] = w.gate;
    f.w[1] = w.up;
    f.to.out = b.act;
    launch_rows_q<kSwiglu>(f, stream);
    f.x = b.act;
    f.k = s.ffn_dim;
    f.w[0] = w.down;
    f.to.out = b.hidden;
    launch_rows_q<kAdd>(f, stream);
}

} // namespace nut
