// matvec.hip — standalone quantised and fp32 matvec kernels for gfx950.
//
// Bandwidth-bound, no MFMA. Fast layout (blocks of 32, 64, ... along whole rows): a wave
// owns R consecutive rows; lane l handles 16-byte chunks l, l + 64, ... of
// each row (32 INT4 or 16 INT8 weights, all of one block) and the R row
// sums are reduced with DPP at the end. Two variants:
//   staged  the workgroup stages x once in LDS (rows.hpp) and each lane
//           reads its x chunk from there; the first weight chunk of every
//           row is requested before the staging, so it loads meanwhile;
//   direct  each lane reads its x chunk from global memory (through L1);
//           used when x does not fit 64 KB of LDS.
// Rows that blocks straddle run in 16-weight runs (matvec_q_ragged); other
// block sizes run one row per wave, a weight per lane, from an LDS copy of x.
#include "kernels.hpp"
#include "rows.hpp"
#include "runtime.hpp"

namespace nut {

namespace {

constexpr int kThreads = kRowThreads;
constexpr int kWaves = kRowWaves;

template <int QT, int R, bool WB>
__global__ __launch_bounds__(kThreads) void matvec_q_fast(QMat m,
                                                          const float *__restrict__ x,
                                                          float *__restrict__ y)
{
    constexpr int CW = QT == 1 ? 32 : 16; // weights per 16-byte chunk
    constexpr float kBias = QT == 1 ? 8.0f : 128.0f;
    const int lane = threadIdx.x & (kWave - 1);
    const int row0 = (blockIdx.x * kWaves + threadIdx.x / kWave) * R;
    if (row0 >= m.rows)
        return; // wave-uniform
    const int row_bytes = QT == 1 ? m.cols / 2 : m.cols;
    const int chunks = row_bytes / 16;
    const int shift = WB ? scale_shift(m) : 0;
    const int blocks_per_row = m.cols >> (shift + 5);
    const uint8_t *rows[R];
    const uint16_t *scales[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int rr = min(row0 + r, m.rows - 1); // tail rows re-read the last
        rows[r] = m.data + size_t(rr) * row_bytes;
        scales[r] = m.scales + size_t(rr) * blocks_per_row;
    }
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++)
        acc[r] = 0.0f;
    for (int c = lane; c < chunks; c += kWave) {
        const int block = (QT == 1 ? c : (c >> 1)) >> shift;
        uint4 w[R];
        float s[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            w[r] = load_stream(rows[r] + 16 * c);
            s[r] = half_bits_to_float(scales[r][block]);
        }
        float xc[CW];
        const float4 *x4 = reinterpret_cast<const float4 *>(x + c * CW);
#pragma unroll
        for (int q = 0; q < CW / 4; q++) {
            const float4 v = x4[q];
            xc[4 * q] = v.x;
            xc[4 * q + 1] = v.y;
            xc[4 * q + 2] = v.z;
            xc[4 * q + 3] = v.w;
        }
        if (WB) { // see rows_matvec
            // every load before the first dot: the compiler sinks half of them
            // behind it otherwise (INT8 2000 x 15360 block 64 33 against 26 us)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < R; r++)
                acc[r] += QT == 1 ? dot_int4_scaled(w[r], xc, s[r])
                                  : dot_int8_scaled(w[r], xc, s[r]);
            continue;
        }
        float xsum = 0.0f;
#pragma unroll
        for (int i = 0; i < CW; i++)
            xsum += xc[i];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float d = QT == 1 ? dot_int4_chunk(w[r], xc) : dot_int8_chunk(w[r], xc);
            acc[r] = fmaf(s[r], d - kBias * xsum, acc[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const float v = wave_total(acc[r]);
        if (lane == 0 && row0 + r < m.rows)
            y[row0 + r] = v;
    }
}

template <int QT, int R, bool WB>
__global__ __launch_bounds__(kThreads) void matvec_q_staged(QMat m, const float *x,
                                                            float *y)
{
    extern __shared__ float xs[];
    const int row0 = (blockIdx.x * kWaves + threadIdx.x / kWave) * R;
    const uint8_t *rp[R];
    const uint16_t *sp[R];
    row_ptrs<QT, R, WB>(m, row0, 0, R, rp, sp);
    float out[R];
    rows_matvec<QT, R, WB, false>(rp, sp, m.cols, scale_shift(m), x, nullptr, row0 < m.rows, xs,
                                  nullptr, out);
    if (row0 < m.rows && (threadIdx.x & (kWave - 1)) == 0)
#pragma unroll
        for (int r = 0; r < R; r++)
            if (row0 + r < m.rows)
                y[row0 + r] = out[r];
}

// Rows that blocks straddle (block_size a power of two >= 16, any cols): a
// wave owns kRaggedRows consecutive rows; lane l handles the 16-weight runs
// l, l + 64, ... of each row, read with one load at whatever byte they begin
// (unaligned vector access is on for this target; an INT4 row that begins in
// the middle of a byte is shifted by a nibble in registers). A run lies in
// at most two blocks: the weights before the boundary take the first scale.
// Four sums a row, of four weights of each run, keep the chains no longer than
// a weight a lane made them (4096 x 255 INT4: error 7.7e-8, 8.9e-8 with one).
// The last cols % 16 weights go one to a lane. Bounded by its VALU work and
// the latency of the first loads; one weight per lane and load, as before,
// spent a 64-bit division and three loads on each: 5000 x 3001 INT4 26.4 us,
// now 8 (two matrices a pass 70.6 -> 15.8).
constexpr int kRaggedRows = 2, kRaggedThreads = 512;
constexpr int kRunLd = 20; // floats of x per run in LDS (16, padded)

struct __attribute__((packed)) Run8 {
    uint32_t w[2];
};
struct __attribute__((packed)) Run16 {
    uint32_t w[4];
};

inline size_t ragged_lds_bytes(int cols)
{
    return size_t((cols + 15) / 16) * kRunLd * sizeof(float);
}

template <int QT>
__global__ __launch_bounds__(kRaggedThreads) void matvec_q_ragged(QMat m, const float *x,
                                                                  float *y, int log_block)
{
    extern __shared__ float xs[];
    const int lane = threadIdx.x & (kWave - 1);
    const int row0 = (blockIdx.x * (kRaggedThreads / kWave) +
                      __builtin_amdgcn_readfirstlane(threadIdx.x / kWave)) *
                     kRaggedRows;
    const int runs = m.cols / 16, block = m.block_size;
    size_t base[kRaggedRows];
    int head[kRaggedRows]; // weights of the row's first block before the row
    const uint16_t *scales[kRaggedRows];
#pragma unroll
    for (int r = 0; r < kRaggedRows; r++) {
        base[r] = size_t(min(row0 + r, m.rows - 1)) * m.cols; // tail rows re-read the last
        head[r] = int(base[r] & size_t(block - 1));
        scales[r] = m.scales + (base[r] >> log_block);
    }
    struct Run {
        uint32_t w[4];
        uint32_t next; // INT4: the byte after the run's eight
        float s0, s1;
    };
    auto load = [&](int c, Run (&run)[kRaggedRows]) {
#pragma unroll
        for (int r = 0; r < kRaggedRows; r++) {
            const size_t f = base[r] + 16 * size_t(c);
            if (QT == 1) {
                const Run8 v = *reinterpret_cast<const Run8 *>(m.data + (f >> 1));
                run[r].w[0] = v.w[0];
                run[r].w[1] = v.w[1];
                // an odd start's last nibble is in the next byte
                run[r].next = (base[r] & 1) ? m.data[(f >> 1) + 8] : 0u;
            } else {
                const Run16 v = *reinterpret_cast<const Run16 *>(m.data + f);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    run[r].w[j] = v.w[j];
            }
            const int at = head[r] + 16 * c;
            run[r].s0 = half_bits_to_float(scales[r][at >> log_block]);
            run[r].s1 = half_bits_to_float(scales[r][(at + 15) >> log_block]);
        }
    };
    Run first[kRaggedRows];
    const bool any = row0 < m.rows && lane < runs;
    if (any)
        load(lane, first);
    for (int i = threadIdx.x; i < m.cols; i += kRaggedThreads)
        xs[(i >> 4) * kRunLd + (i & 15)] = x[i];
    __syncthreads();
    if (row0 >= m.rows)
        return; // wave-uniform
    float acc[kRaggedRows][4] = {};
    auto add = [&](int c, const Run (&run)[kRaggedRows]) {
        float xc[16];
        const float4 *x4 = reinterpret_cast<const float4 *>(xs + c * kRunLd);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 v = x4[q];
            xc[4 * q] = v.x;
            xc[4 * q + 1] = v.y;
            xc[4 * q + 2] = v.z;
            xc[4 * q + 3] = v.w;
        }
#pragma unroll
        for (int r = 0; r < kRaggedRows; r++) {
            // weights of the run before the block boundary
            const int before = block - ((head[r] + 16 * c) & (block - 1));
            uint32_t w[4];
            if (QT == 1) {
                w[0] = run[r].w[0];
                w[1] = run[r].w[1];
                if (base[r] & 1) { // wave-uniform
                    w[0] = w[0] >> 4 | w[1] << 28;
                    w[1] = w[1] >> 4 | run[r].next << 28;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    w[j] = run[r].w[j];
            }
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int q = QT == 1 ? int(w[i / 8] << (28 - 4 * (i % 8))) >> 28
                                      : int(w[i / 4] << (24 - 8 * (i % 4))) >> 24;
                acc[r][i / 4] =
                    fmaf(float(q) * (i < before ? run[r].s0 : run[r].s1), xc[i], acc[r][i / 4]);
            }
        }
    };
    if (any)
        add(lane, first);
    for (int c = lane + kWave; c < runs; c += kWave) {
        Run run[kRaggedRows];
        load(c, run);
        add(c, run);
    }
    const int rest = 16 * runs + lane;
    if (rest < m.cols) {
#pragma unroll
        for (int r = 0; r < kRaggedRows; r++) {
            const size_t f = base[r] + rest;
            int q;
            if (QT == 1)
                q = int(uint32_t(m.data[f >> 1]) << ((f & 1) ? 24 : 28)) >> 28;
            else
                q = int(int8_t(m.data[f]));
            const float s = half_bits_to_float(scales[r][(head[r] + rest) >> log_block]);
            acc[r][0] = fmaf(float(q) * s, xs[(rest >> 4) * kRunLd + (rest & 15)], acc[r][0]);
        }
    }
#pragma unroll
    for (int r = 0; r < kRaggedRows; r++) {
        const float v = wave_total((acc[r][0] + acc[r][1]) + (acc[r][2] + acc[r][3]));
        if (lane == 0 && row0 + r < m.rows)
            y[row0 + r] = v;
    }
}

__global__ __launch_bounds__(kThreads) void matvec_q_generic(QMat m,
                                                             const float *x,
                                                             float *y)
{
    extern __shared__ float xs[];
    for (int i = threadIdx.x; i < m.cols; i += blockDim.x)
        xs[i] = x[i];
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    for (int row = blockIdx.x * kWaves + wave; row < m.rows;
         row += gridDim.x * kWaves) {
        const float v = qrow_generic(m, row, xs);
        if (lane == 0)
            y[row] = v;
    }
}

// fp32 rows: lane l reads float4 chunks l, l+64, ... of each row.
__global__ __launch_bounds__(kThreads) void matvec_f32_kernel(
    const float *w, int rows, int cols, const float *x, float *y)
{
    extern __shared__ float xs[];
    for (int i = threadIdx.x; i < cols; i += blockDim.x)
        xs[i] = x[i];
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    for (int row = blockIdx.x * kWaves + wave; row < rows;
         row += gridDim.x * kWaves) {
        const float *wr = w + size_t(row) * cols;
        float acc = 0.0f;
        if ((cols & 3) == 0) {
            for (int c = lane; c < cols / 4; c += kWave) {
                const float4 v = reinterpret_cast<const float4 *>(wr)[c];
                const float *xc = xs + 4 * c;
                acc = fmaf(v.x, xc[0], acc);
                acc = fmaf(v.y, xc[1], acc);
                acc = fmaf(v.z, xc[2], acc);
                acc = fmaf(v.w, xc[3], acc);
            }
        } else {
            for (int c = lane; c < cols; c += kWave)
                acc = fmaf(wr[c], xs[c], acc);
        }
        acc = wave_sum(acc);
        if (lane == 0)
            y[row] = acc;
    }
}

int grid_for(int work_items)
{
    const int blocks = (work_items + kWaves - 1) / kWaves;
    return blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks);
}

} // namespace

// LDS of a kernel that stages x and its per-chunk sums (the step kernels).
size_t matvec_q_lds_bytes(const QMat &m)
{
    const int cw = chunk_weights(m.type);
    return sizeof(float) * (size_t(m.cols) + (m.cols + cw - 1) / cw);
}

template <int QT, int R>
void launch_fast(const QMat &m, const float *x, float *y, hipStream_t stream)
{
    const int waves = (m.rows + R - 1) / R;
    const int blocks = (waves + kWaves - 1) / kWaves;
    if (m.block_size == 32)
        hipLaunchKernelGGL((matvec_q_fast<QT, R, false>), dim3(blocks), dim3(kThreads), 0,
                           stream, m, x, y);
    else
        hipLaunchKernelGGL((matvec_q_fast<QT, R, true>), dim3(blocks), dim3(kThreads), 0,
                           stream, m, x, y);
}

template <int QT, int R>
void launch_staged(const QMat &m, const float *x, float *y, hipStream_t stream)
{
    const int waves = (m.rows + R - 1) / R;
    const int blocks = (waves + kWaves - 1) / kWaves;
    if (m.block_size == 32)
        hipLaunchKernelGGL((matvec_q_staged<QT, R, false>), dim3(blocks), dim3(kThreads),
                           staged_x_bytes<QT>(m.cols), stream, m, x, y);
    else
        hipLaunchKernelGGL((matvec_q_staged<QT, R, true>), dim3(blocks), dim3(kThreads),
                           staged_x_bytes<QT>(m.cols), stream, m, x, y);
}

void launch_matvec_q(const QMat &m, const float *x, float *y,
                     hipStream_t stream)
{
    // INT4 chunks need 32 floats of x per 16 bytes of weights, which keeps
    // L1 busier than HBM unless x comes from LDS; INT8 chunks need 16, and
    // below 4096 rows the staging latency costs more than it saves
    // (measured per shape with rocprofv3)
    const bool staged = m.type == 1 ? staged_x_bytes<1>(m.cols) <= 65536
                                    : m.rows >= 4096 && staged_x_bytes<0>(m.cols) <= 65536;
    // these kernels have a workgroup for every few rows, and a grid holds less
    // than 2^32 threads (32 a row); more rows go through in a loop
    const bool loop = m.rows > 1 << 26;
    if (fast_layout(m) && !loop && staged) {
        // two rows per wave, one where that leaves fewer than 256 workgroups
        if (m.rows >= 2048)
            m.type == 1 ? launch_staged<1, 2>(m, x, y, stream)
                        : launch_staged<0, 2>(m, x, y, stream);
        else
            m.type == 1 ? launch_staged<1, 1>(m, x, y, stream)
                        : launch_staged<0, 1>(m, x, y, stream);
    } else if (fast_layout(m) && !loop) {
        // rows per wave: enough waves to fill 256 CUs, as many rows in
        // flight per wave as that allows
        const int r = m.rows >= 4096 ? 4 : m.rows >= 1024 ? 2 : 1;
        if (m.type == 1)
            r == 4 ? launch_fast<1, 4>(m, x, y, stream)
                   : r == 2 ? launch_fast<1, 2>(m, x, y, stream)
                            : launch_fast<1, 1>(m, x, y, stream);
        else
            r == 4 ? launch_fast<0, 4>(m, x, y, stream)
                   : r == 2 ? launch_fast<0, 2>(m, x, y, stream)
                            : launch_fast<0, 1>(m, x, y, stream);
    } else if (!loop && m.block_size >= 16 && (m.block_size & (m.block_size - 1)) == 0 &&
               ragged_lds_bytes(m.cols) <= 65536) {
        const int log_block = __builtin_ctz(unsigned(m.block_size));
        const int per = kRaggedRows * kRaggedThreads / kWave;
        const dim3 grid((m.rows + per - 1) / per);
        if (m.type == 1)
            hipLaunchKernelGGL(matvec_q_ragged<1>, grid, dim3(kRaggedThreads),
                               ragged_lds_bytes(m.cols), stream, m, x, y, log_block);
        else
            hipLaunchKernelGGL(matvec_q_ragged<0>, grid, dim3(kRaggedThreads),
                               ragged_lds_bytes(m.cols), stream, m, x, y, log_block);
    } else {
        const size_t lds = sizeof(float) * size_t(m.cols);
        require(lds <= 64 * 1024, NUT_EINVAL,
                "quantized matvec: input dimension exceeds LDS staging");
        hipLaunchKernelGGL(matvec_q_generic, dim3(grid_for(m.rows)), dim3(kThreads),
                           lds, stream, m, x, y);
    }
    check_launch("quantized matvec");
}

void launch_matvec_f32(const float *w, int rows, int cols, const float *x,
                       float *y, hipStream_t stream)
{
    const size_t lds = sizeof(float) * size_t(cols);
    require(lds <= 64 * 1024, NUT_EINVAL,
            "threaded matvec: input dimension exceeds LDS staging");
    hipLaunchKernelGGL(matvec_f32_kernel, dim3(grid_for(rows)),
                       dim3(kThreads), lds, stream, w, rows, cols, x, y);
    check_launch("threaded matvec");
}

} // namespace nut
