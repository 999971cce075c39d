// project.hpp — what a layer's projections become, shared by the fp32 model's
// tile (fmodel.hip) and the quantised row tile (rowgemm.hip): a lane holds TJ
// finished sums of one row (gemm_f32_reduce).
#pragma once

#include "gemm_f32.hpp"

namespace nut {

enum ProjectEpilogue {
    kAdd,    // added to the rows of `out`
    kSwiglu, // silu(gate) * up; the lane's first half are gate sums
    kQkv,    // RoPE on q and k; q rows to `out`, k and v to the cache
};

struct ProjectOut {
    float *out; // rows of n: hidden rows, activations, query rows
    const float2 *rope;
    float *k_layer, *v_layer;
    int first_pos, head_dim, max_seq;
};

// 1 / sqrt(mean of squares + 1e-5) of tile row r (src/ops.cpp:111-134) from
// the waves' shares of its squares.
template <int WK, int ROWS>
__device__ __forceinline__ float row_scale(const float (&squares)[WK][ROWS], int r, int k)
{
    float s = squares[0][r];
#pragma unroll
    for (int w = 1; w < WK; w++)
        s += squares[w][r];
    return 1.0f / sqrtf(s / float(k) + 1e-5f);
}

// Stores a lane's sums of output row `row`: its columns are first .. of n
// (segment `seg` of q, k, v), of which those before `col` belong to other
// lanes.
template <int EPI, int TJ>
__device__ __forceinline__ void project_store(const ProjectOut &f, int seg, int n, int row,
                                              int col, int first, const float (&out)[TJ])
{
    constexpr int TB = EPI == kSwiglu ? TJ / 2 : TJ;
    float vals[TB];
    float *dst;
    if constexpr (EPI == kSwiglu) {
#pragma unroll
        for (int j = 0; j < TB; j++)
            vals[j] = out[j] / (1.0f + expf(-out[j])) * out[TB + j];
        dst = f.out + size_t(row) * n + first;
    } else if constexpr (EPI == kAdd) {
        dst = f.out + size_t(row) * n + first;
#pragma unroll
        for (int j = 0; j < TB; j++)
            vals[j] = dst[j] + out[j];
    } else {
        // RoPE (rotate_vector, src/kvcache.cpp:48-59); TB, n and head_dim
        // are even, so a pair is a lane's
        static_assert(EPI != kQkv || TB % 2 == 0, "whole RoPE pairs");
        const int pos = f.first_pos + row;
        const int head = first / f.head_dim, d = first % f.head_dim;
#pragma unroll
        for (int j = 0; j < TB; j += 2) {
            float e = out[j], o = out[j + 1];
            if (seg < 2) {
                const float2 cs = f.rope[size_t(pos) * (f.head_dim / 2) + (d + j) / 2];
                const float even = e, odd = o;
                e = fmaf(even, cs.x, -(odd * cs.y));
                o = fmaf(even, cs.y, odd * cs.x);
            }
            vals[j] = e;
            vals[j + 1] = o;
        }
        // head_dim is a multiple of 4 and TB 2 or 4, first a multiple of TB:
        // a lane's columns are of one head
        dst = seg == 0 ? f.out + size_t(row) * n + first
                       : (seg == 1 ? f.k_layer : f.v_layer) +
                             (size_t(head) * f.max_seq + pos) * f.head_dim + d;
    }
    if (first == col) {
        store_u<TB>(dst, vals);
    } else {
#pragma unroll
        for (int j = 0; j < TB; j++)
            if (first + j >= col)
                dst[j] = vals[j];
    }
}

} // namespace nut
