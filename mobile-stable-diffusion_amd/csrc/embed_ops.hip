// Neighbours of the norm / activation path for gfx950: the Linear layers that act on
// the few rows of the time embedding (weight-streaming, one or two output columns per
// wavefront), the row softmax of the attention blocks (a row held in the registers
// of a team of lanes) and the DDIM latent update.
#include "msd_device.h"
#include "msd_internal.h"
#include "tile_transpose.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace msd {
namespace {

// ---------------------------------------------------------------------------
// y[m, n] = act_out(act_in(x)[m, k] . w[n, k]^T + bias[n]) for m <= 8 rows.
// The time is the single pass over w (n*k elements) plus launch and memory latency, so
// the kernel is built to have one latency, not two in a row: a workgroup is a single
// wavefront that owns CPW columns; lane l requests 16-byte pieces l, l+64, ... of its
// weight rows and the same pieces of every x row (a few KiB that every wavefront
// reads from cache) before it uses any of them.  No LDS, no barrier.  With SiLU on the
// input each lane activates its own x pieces, and two columns share that work.
// Each lane adds its pieces in ascending k, then the M x CPW partial sums go through
// the DPP tree, so the result does not depend on the launch shape.
// ---------------------------------------------------------------------------

template <typename T, int M, int CPW, int ROUND = 0>
__device__ __forceinline__ void linear_rows_body(const T *__restrict__ x, const T *__restrict__ w,
                                                 const float *__restrict__ bias, T *__restrict__ y,
                                                 uint32_t m, uint32_t n, uint32_t kvecs, int act_in,
                                                 int act_out, uint32_t col0) {
    constexpr int EPV = Store<T>::EPV;
    // pieces per lane per round: one round covers k = 2048 (float with more than 4 rows: 1024)
    constexpr int kLinRound = ROUND != 0 ? ROUND : (sizeof(T) == 4 && M <= 4) ? 8 : 4;
    const uint32_t lane = threadIdx.x;
    const u32x4 *xin = reinterpret_cast<const u32x4 *>(x);
    const u32x4 *win = reinterpret_cast<const u32x4 *>(w);
    float acc[CPW][M];
#pragma unroll
    for (int c = 0; c < CPW; c++)
#pragma unroll
        for (int i = 0; i < M; i++) acc[c][i] = 0.0f;
    for (uint32_t base = lane; base < kvecs; base += kWave * kLinRound) {
        u32x4 wraw[CPW][kLinRound], xraw[M][kLinRound];
#pragma unroll
        for (int u = 0; u < kLinRound; u++) {
            const uint32_t piece = min(base + u * kWave, kvecs - 1);
#pragma unroll
            for (int c = 0; c < CPW; c++)  // a column past the last re-reads the last one
                wraw[c][u] = load_stream(win + (size_t)min(col0 + c, n - 1) * kvecs + piece);
#pragma unroll
            for (int i = 0; i < M; i++)    // rows >= m repeat the last row
                xraw[i][u] = xin[(size_t)min((uint32_t)i, m - 1) * kvecs + piece];
        }
#pragma unroll
        for (int u = 0; u < kLinRound; u++) {
            if (base + u * kWave < kvecs) {
                float xf[M][EPV];
#pragma unroll
                for (int i = 0; i < M; i++) {
                    Store<T>::unpack(xraw[i][u], xf[i]);
                    if (act_in) {
#pragma unroll
                        for (int e = 0; e < EPV; e++) xf[i][e] = silu_f(xf[i][e]);
                    }
                }
#pragma unroll
                for (int c = 0; c < CPW; c++) {
                    float wf[EPV];
                    Store<T>::unpack(wraw[c][u], wf);
#pragma unroll
                    for (int i = 0; i < M; i++)
#pragma unroll
                        for (int e = 0; e < EPV; e++) acc[c][i] = fmaf(xf[i][e], wf[e], acc[c][i]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < CPW; c++) {
        float mine = 0.0f;
#pragma unroll
        for (int i = 0; i < M; i++) {
            const float total = wave_sum(acc[c][i]);
            if (lane == (uint32_t)i) mine = total;
        }
        const uint32_t col = col0 + c;
        if (lane < m && col < n) {
            float r = mine + (bias != nullptr ? bias[col] : 0.0f);
            if (act_out) r = silu_f(r);
            Store<T>::store1(y + (size_t)lane * n + col, r);
        }
    }
}

template <typename T, int M, int CPW>
__global__ __launch_bounds__(kWave) void linear_rows_kernel(
    const T *__restrict__ x, const T *__restrict__ w, const float *__restrict__ bias,
    T *__restrict__ y, uint32_t m, uint32_t n, uint32_t kvecs, int act_in, int act_out) {
    linear_rows_body<T, M, CPW>(x, w, bias, y, m, n, kvecs, act_in, act_out, blockIdx.x * CPW);
}

// Several Linear layers on the same rows x in one launch (the per-ResBlock projections of the
// time embedding all read the same [m, k] embedding): the problems' workgroups are laid end to
// end, a workgroup finds its problem by walking the table of first workgroups (at most
// kLinGroupMax entries, passed by value with the launch), then runs the same code as a single
// launch would, so each problem's result is that of its own msd_linear_rows call bit for bit.
constexpr int kLinGroupMax = 32;
struct LinearGroup {
    const void *w[kLinGroupMax];
    const float *bias[kLinGroupMax];
    void *y[kLinGroupMax];
    uint32_t n[kLinGroupMax];
    uint32_t first_block[kLinGroupMax + 1];  // first_block[count] = number of workgroups
    uint32_t count;
};

template <typename T, int M, int CPW, int ROUND = 0>
__global__ __launch_bounds__(kWave) void linear_rows_grouped_kernel(const T *__restrict__ x, LinearGroup g,
                                                                    uint32_t m, uint32_t kvecs, int act_in,
                                                                    int act_out) {
    uint32_t p = 0;
    while (p + 1 < g.count && blockIdx.x >= g.first_block[p + 1]) p++;  // uniform: scalar loop
    linear_rows_body<T, M, CPW, ROUND>(x, static_cast<const T *>(g.w[p]), g.bias[p], static_cast<T *>(g.y[p]), m,
                                g.n[p], kvecs, act_in, act_out, (blockIdx.x - g.first_block[p]) * CPW);
}

// The same for m = 3 ... 8 rows of 2-byte elements, on the matrix cores and bit for bit.  A column or a few per wavefront read
// the rows of x once per column or few, 3 to 8 times the bytes of the weights; here a workgroup of four wavefronts owns 4 CQ
// columns and reads them once for all.  The 64 lanes among which linear_rows_body deals the pieces of a row are the 16 blocks
// of four lanes of each of the four wavefronts: v_mfma_f32_4x4x1 multiplies, in every block by itself, one element of four
// columns (one a lane) with one of four rows of x (one a lane), a float32 fused multiply-add into each of the 16 sums.  So a sum
// meets the same products in the same order, of float32 values (an activated x has no fewer bits here), and the same tree
// adds the blocks.  Halves go in as the float32 they are: products of halves by a 16-bit matrix instruction, whose sums over
// 32 products are rounded in its own way, were up to 1.35 times as far from the sums in 64 bits (k = 5120).
// R pieces of every row are requested before the first is used.  Bound by the weights' bytes for three and four rows, from
// five on by conversions, SiLU and products too.  The 22 projections of a
// step, 20160 columns of k = 1280, us, a column or two per wavefront and so: 3 and 4 rows 20 / 22 with SiLU -> 12.4 / 12.8, 8 rows
// 41.5 / 42.4 -> 14.0 / 15.8 (1 row: 9.9); a single 1280-column layer, 8 rows 5.5 / 7.5 -> 4.5 / 4.7.
constexpr int kLinWgWaves = 4;
constexpr int kLinWgThreads = kLinWgWaves * kWave;
constexpr int kLinBlock = 4;                       // lanes, columns and rows of a block
constexpr int kLinBlocks = kWave / kLinBlock;      // blocks of a wavefront
constexpr int kDppRowRor8 = 0x128;  // lane i <- lane (i + 8) mod 16 inside each 16

// The value of lane ^ (1 << bit).
__device__ __forceinline__ float lane_partner(float f, int bit) {
    const int i = __float_as_int(f);
    switch (bit) {
        case 0: return dpp_move<kDppXor1>(f);
        case 1: return dpp_move<kDppXor2>(f);
        case 2: return __int_as_float(__builtin_amdgcn_ds_swizzle(i, 0x101F));
        case 3: return dpp_move<kDppRowRor8>(f);
        case 4: return __int_as_float(__builtin_amdgcn_ds_swizzle(i, 0x401F));
        default: return __shfl_xor(f, 32);
    }
}

// Sums of NV values (a power of two) over the lanes that differ in bits FIRST ... FIRST + BITS - 1.  Each step makes the
// additions of team_sum, but keeps half as many values: bit for bit the same sums.  On return v[j] of a lane is the sum of
// value (j << BITS) + those bits of the lane, of fewer values than 2^BITS that of the bits modulo NV.
template <int FIRST, int BITS, int NV>
__device__ __forceinline__ void scatter_sums(float (&v)[NV]) {
    const uint32_t lane = threadIdx.x;
#pragma unroll
    for (int bit = FIRST, n = NV; bit < FIRST + BITS; bit++) {
        if (n > 1) {
            n /= 2;
            const bool upper = (lane >> bit) & 1;
#pragma unroll
            for (int i = 0; i < NV / 2; i++) {
                if (i < n) {
                    const float mine = upper ? v[2 * i + 1] : v[2 * i], other = upper ? v[2 * i] : v[2 * i + 1];
                    v[i] = mine + lane_partner(other, bit);
                }
            }
        } else {
            v[0] += lane_partner(v[0], bit);
        }
    }
}

template <int MQ, int CQ, int R, bool ACT>
__device__ __forceinline__ void linear_quads_body(const __half *__restrict__ x, const __half *__restrict__ w,
                                                  const float *__restrict__ bias, __half *__restrict__ y, uint32_t m,
                                                  uint32_t n, uint32_t kvecs, int act_out, uint32_t col0) {
    constexpr int NV = CQ * MQ * kLinBlock;  // sums a lane takes part in
    __shared__ float parts[kLinWgWaves][NV * kLinBlock];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t block = (threadIdx.x & (kWave - 1)) / kLinBlock, i = threadIdx.x % kLinBlock;
    const u32x4 *xin = reinterpret_cast<const u32x4 *>(x), *win = reinterpret_cast<const u32x4 *>(w);
    // what this lane stores in the end
    const uint32_t t = threadIdx.x, quads = t / (kLinBlock * kLinBlock);
    const uint32_t row = kLinBlock * (quads % MQ) + i, col = col0 + kLinBlock * (quads / MQ) + t / kLinBlock % kLinBlock;
    const float b = bias != nullptr ? bias[min(col, n - 1)] : 0.0f;
    f32x4 acc[CQ][MQ];
#pragma unroll
    for (int q = 0; q < CQ; q++)
#pragma unroll
        for (int r = 0; r < MQ; r++) acc[q][r] = f32x4{0, 0, 0, 0};
    for (uint32_t base = kLinBlocks * wave; base < kvecs; base += kWave * R) {
        u32x4 wraw[CQ][R], xraw[MQ][R];
#pragma unroll
        for (int u = 0; u < R; u++) {  // (columns past the last and rows past m repeat the last one and are not stored)
            const uint32_t piece = min(base + u * kWave + block, kvecs - 1);
#pragma unroll
            for (int r = 0; r < MQ; r++) xraw[r][u] = xin[(size_t)min(kLinBlock * r + i, m - 1) * kvecs + piece];
#pragma unroll
            for (int q = 0; q < CQ; q++)
                wraw[q][u] = load_stream(win + (size_t)min(col0 + kLinBlock * q + i, n - 1) * kvecs + piece);
        }
        asm volatile("" ::: "memory");  // the loads stay in front of the branches below
#pragma unroll
        for (int u = 0; u < R; u++) {
            const uint32_t first = base + u * kWave;  // (uniform over the wavefront)
            if (first >= kvecs) break;
            if (first + kLinBlocks > kvecs) {  // a piece past the row's end counts as zeros, on both sides
                const bool have = first + block < kvecs;
                const u32x4 zero = {0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < MQ; r++) xraw[r][u] = have ? xraw[r][u] : zero;
#pragma unroll
                for (int q = 0; q < CQ; q++) wraw[q][u] = have ? wraw[q][u] : zero;
            }
            float xf[MQ][8], wf[CQ][8];
#pragma unroll
            for (int r = 0; r < MQ; r++) {
                Store<__half>::unpack(xraw[r][u], xf[r]);
                if (ACT) {
#pragma unroll
                    for (int e = 0; e < 8; e++) xf[r][e] = silu_f(xf[r][e]);
                }
            }
#pragma unroll
            for (int q = 0; q < CQ; q++) Store<__half>::unpack(wraw[q][u], wf[q]);
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
                for (int q = 0; q < CQ; q++)
#pragma unroll
                    for (int r = 0; r < MQ; r++)
                        acc[q][r] = __builtin_amdgcn_mfma_f32_4x4x1f32(wf[q][e], xf[r][e], acc[q][r], 0, 0, 0);
        }
    }
    float v[NV];  // value (q, r, j): column 4 q + j against row 4 r + i
#pragma unroll
    for (int q = 0; q < CQ; q++)
#pragma unroll
        for (int r = 0; r < MQ; r++)
#pragma unroll
            for (int j = 0; j < kLinBlock; j++) v[(q * MQ + r) * kLinBlock + j] = acc[q][r][j];
    scatter_sums<2, 4>(v);
#pragma unroll
    for (int j = 0; j < (NV + kLinBlocks - 1) / kLinBlocks; j++) {
        const uint32_t value = j * kLinBlocks + block;
        if (value < NV) parts[wave][value * kLinBlock + i] = v[j];
    }
    __syncthreads();
    if (t >= NV * kLinBlock || row >= m || col >= n) return;
    float total = (parts[0][t] + parts[1][t]) + (parts[2][t] + parts[3][t]) + b;
    if (act_out) total = silu_f(total);
    Store<__half>::store1(y + (size_t)row * n + col, total);
}

template <int MQ, int CQ, int R, bool ACT>
__global__ __launch_bounds__(kLinWgThreads, 4) void linear_quads_kernel(
    const __half *__restrict__ x, const __half *__restrict__ w, const float *__restrict__ bias, __half *__restrict__ y,
    uint32_t m, uint32_t n, uint32_t kvecs, int act_out) {
    linear_quads_body<MQ, CQ, R, ACT>(x, w, bias, y, m, n, kvecs, act_out, blockIdx.x * (kLinBlock * CQ));
}

template <int MQ, int CQ, int R, bool ACT>
__global__ __launch_bounds__(kLinWgThreads, 4) void linear_quads_grouped_kernel(const __half *__restrict__ x, LinearGroup g,
                                                                                uint32_t m, uint32_t kvecs, int act_out) {
    uint32_t p = 0;
    while (p + 1 < g.count && blockIdx.x >= g.first_block[p + 1]) p++;  // uniform: scalar loop
    linear_quads_body<MQ, CQ, R, ACT>(x, static_cast<const __half *>(g.w[p]), g.bias[p], static_cast<__half *>(g.y[p]), m,
                                      g.n[p], kvecs, act_out, (blockIdx.x - g.first_block[p]) * (kLinBlock * CQ));
}

// Large groups of 4-byte elements, 2 ... 8 rows: four wavefronts share the rows of x, activated once, in LDS, and each takes
// four columns against them.  The order of every sum is that of linear_rows_body.  Bound by the latency of its three steps
// (x to LDS, barrier, products) and, from five rows on, by the products.  The 22 projections of a step, 103 MB of
// weights, us, before with two columns per wavefront and so: 2 rows 21 - 24 -> 20, 4 rows 34 - 43 -> 24.5, 8 rows
// 53 - 59 -> 29 (1 row: 18).  Two columns instead of four 33 at 8 rows, float32 matrix products 28, with other sums.
constexpr int kSharedCols = 4;

template <int M>
__global__ __launch_bounds__(kLinWgThreads) void linear_shared_grouped_kernel(const float *__restrict__ x, LinearGroup group,
                                                                              uint32_t m, uint32_t kvecs, int act_in,
                                                                              int act_out) {
    constexpr int C = kSharedCols, ROUND = 5;
    constexpr uint32_t kChunk = ROUND * kWave;  // pieces of a row of x in LDS at a time
    __shared__ f32x4 xs[M][kChunk];
    uint32_t p = 0;
    while (p + 1 < group.count && blockIdx.x >= group.first_block[p + 1]) p++;  // uniform: scalar loop
    const u32x4 *win = static_cast<const u32x4 *>(group.w[p]);
    const float *bias = group.bias[p];
    float *y = static_cast<float *>(group.y[p]);
    const uint32_t n = group.n[p];
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const uint32_t col0 = ((blockIdx.x - group.first_block[p]) * kLinWgWaves + wave) * C;
    const uint32_t out_col = col0 + (lane % (C * M)) / M, out_row = lane % M;  // what this lane stores
    const float b = bias != nullptr ? bias[min(out_col, n - 1)] : 0.0f;
    float acc[C * M];
#pragma unroll
    for (int i = 0; i < C * M; i++) acc[i] = 0.0f;
    for (uint32_t base = 0; base < kvecs; base += kChunk) {
        u32x4 wraw[C][ROUND];
#pragma unroll
        for (int u = 0; u < ROUND; u++)
#pragma unroll
            for (int c = 0; c < C; c++)  // a column past the last re-reads the last one
                wraw[c][u] = load_stream(win + (size_t)min(col0 + c, n - 1) * kvecs + min(base + u * kWave + lane, kvecs - 1));
        const uint32_t here = min(kvecs - base, kChunk);
        if (base != 0) __syncthreads();
        for (uint32_t row = 0; row < m; row++)  // (rows from m on hold anything: their sums are not stored)
            for (uint32_t i = threadIdx.x; i < here; i += kLinWgThreads) {
                f32x4 v = reinterpret_cast<const f32x4 *>(x)[(size_t)row * kvecs + base + i];
                if (act_in) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = silu_f(v[e]);
                }
                xs[row][i] = v;
            }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < ROUND; u++) {
            if (u * kWave + lane < here) {
#pragma unroll
                for (int i = 0; i < M; i++) {
                    const f32x4 v = xs[i][u * kWave + lane];
#pragma unroll
                    for (int c = 0; c < C; c++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[c * M + i] = fmaf(v[e], __uint_as_float(wraw[c][u][e]), acc[c * M + i]);
                }
            }
        }
    }
    scatter_sums<0, 5>(acc);  // (at most 32 values: one a lane)
    float r = acc[0] + __shfl_xor(acc[0], 32);
    if (lane < C * M && out_row < m && out_col < n) {
        r += b;
        if (act_out) r = silu_f(r);
        y[(size_t)out_row * n + out_col] = r;
    }
}

constexpr int kLinThreads = 256;  // workgroup of the scalar kernel below
constexpr int kLinWaves = kLinThreads / kWave;

// Any k / alignment: x is read from global memory (it is a few KiB and stays cached).
template <typename T>
__global__ __launch_bounds__(kLinThreads) void linear_rows_generic_kernel(
    const T *__restrict__ x, const T *__restrict__ w, const float *__restrict__ bias,
    T *__restrict__ y, uint32_t m, uint32_t n, uint32_t k, int act_in, int act_out) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t col = blockIdx.x * kLinWaves + threadIdx.x / kWave;
    if (col >= n) return;
    const T *wrow = w + (size_t)col * k;
    for (uint32_t i = 0; i < m; i++) {
        float acc = 0.0f;
        for (uint32_t kk = lane; kk < k; kk += kWave) {
            float xv = Store<T>::load1(x + (size_t)i * k + kk);
            if (act_in) xv = silu_f(xv);
            acc = fmaf(xv, Store<T>::load1(wrow + kk), acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) {
            float r = acc + (bias != nullptr ? bias[col] : 0.0f);
            if (act_out) r = silu_f(r);
            Store<T>::store1(y + (size_t)i * n + col, r);
        }
    }
}

// ---------------------------------------------------------------------------
// Row softmax.  exp(x - shift) / sum, shift = the row maximum (stable) or 0 (the
// form the replaced kernel computes, which overflows above x = 88.7 exactly as it
// does).  A row lives in the registers of a team of TL lanes, VPL 16-byte vectors
// per lane: one read and one write per element.  exp goes through the hardware 2^x
// (relative error below 1.2e-7 * (1 + |x - shift| * 1.45)).
// ---------------------------------------------------------------------------
constexpr int kSmThreads = 256;
constexpr float kNegInf = -__builtin_huge_valf();

// RAGGED: rows that are no whole number of vectors or start at any element (the 18 x 14 = 252 positions of a
// deeper UNet level): the last piece of a row is cut.  Bound like the others by one read and one write, which element
// by element are eight loads and stores a lane (and three passes beyond 512 columns); softmax_dispatch says from how
// many rows on that is slower.  fp16, us, element by element and so: 16128 x 252 6.63 -> 4.66, 32256 x 252
// 10.9 -> 7.1, 65536 x 140 17.9 -> 10.2, 4000 x 1023 9.5 -> 5.2; 16128 x 256, whole vectors, takes 4.1.
// Lanes of a workgroup: long rows (a wavefront per row, 8 or 16 vectors per lane) run as single-wavefront workgroups, the shorter
// ones in workgroups of four (us, four wavefronts / two / one: fp16 5120 x 576 3.83 3.95 4.61, 24576 x 144 5.01 4.89 5.51,
// fp32 20480 x 64 3.16 3.24 3.69, 49152 x 64 5.96 6.07 5.87)
constexpr uint32_t softmax_team_lanes(int vpl, int tl) { return (tl == kWave && vpl >= 8) ? kWave : kSmThreads; }

template <typename T, int VPL, int TL, bool RAGGED>
__global__ __launch_bounds__(kSmThreads) void softmax_team_kernel(const T *x, T *y, uint32_t rows, uint32_t cols,
                                                                  int stable) {
    constexpr int EPV = Store<T>::EPV, ES = (int)sizeof(T);
    constexpr int RPW = kWave / TL;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = blockIdx.x * (softmax_team_lanes(VPL, TL) / kWave) + threadIdx.x / kWave;
    const uint32_t row = wave * RPW + lane / TL;
    const uint32_t j = lane % TL;
    const bool live = row < rows;
    const uint32_t row_vecs = RAGGED ? (cols + EPV - 1) / EPV : cols / EPV;
    const size_t row_base = (size_t)min(row, rows - 1) * cols * ES;
    const char *in = reinterpret_cast<const char *>(x) + row_base;
    char *out = reinterpret_cast<char *>(y) + row_base;
    auto left = [&](uint32_t v) { return cols - v * EPV; };  // elements of the row from vector v on
    u32x4 raw[VPL];
#pragma unroll
    for (int v = 0; v < VPL; v++) {
        const uint32_t at = min(v * TL + j, row_vecs - 1);
        raw[v] = tile_load<ES, RAGGED>(in + (size_t)at * 16, left(at));
    }
    float f[VPL][EPV];
    float mx = kNegInf;
#pragma unroll
    for (int v = 0; v < VPL; v++) {
        Store<T>::unpack(raw[v], f[v]);
        const bool have = v * TL + j < row_vecs;
#pragma unroll
        for (int e = 0; e < EPV; e++) {
            f[v][e] = (RAGGED ? (v * TL + j) * EPV + e < cols : have) ? f[v][e] : kNegInf;  // padding: exp gives 0
            mx = fmaxf(mx, f[v][e]);
        }
    }
    float shift = 0.0f;
    if (stable) {
        shift = team_max<TL>(mx);
        shift = shift == kNegInf ? 0.0f : shift;  // a row of -inf: keep the reference's 0/0
    }
    const float bias = -shift * kLog2e;
    float total = 0.0f;
#pragma unroll
    for (int v = 0; v < VPL; v++)
#pragma unroll
        for (int e = 0; e < EPV; e++) {
            f[v][e] = __builtin_amdgcn_exp2f(fmaf(f[v][e], kLog2e, bias));
            total += f[v][e];
        }
    total = team_sum<TL>(total);
    const float inv = 1.0f / total;
#pragma unroll
    for (int v = 0; v < VPL; v++) {
#pragma unroll
        for (int e = 0; e < EPV; e++) f[v][e] *= inv;
        const uint32_t at = v * TL + j;
        if (live && at < row_vecs) tile_store<ES, RAGGED>(out + (size_t)at * 16, left(at), Store<T>::pack(f[v]));
    }
}

// Rows of more than 256 vectors: the row lives in the registers of a workgroup, VPL 16-byte vectors per lane,
// one read and one write per element; the wavefronts' maxima and sums meet in LDS.  Bound by HBM, and by how many
// rows are open at once: beyond about 48 KB of them a CU, read and not yet written, more only cost time (the
// figures are at softmax_block_launch; the cause was not measured).  The launch therefore asks for LDS it does not use,
// which is what keeps workgroups off a CU.  A wavefront per row with 8 - 16 vectors a lane and workgroups of 8 a lane, both as many
// as fit, before, and so; us, TB/s: fp16 65536 x 4096 169.4 -> 168.3 (6.4), 102400 x 6400 437 -> 420 (6.2), 123904 x 7744
// 661 -> 630 (6.1), 135168 x 8448 796 -> 748 (6.1), 147456 x 9216 917 -> 899 (6.0); fp32 65536 x 4096 351 -> 335 (6.4),
// 102400 x 6400 905 -> 862 (6.1), 73728 x 9216 967 -> 906 (6.0).  A copy takes 6.4 to 6.6.
// x and y may be the same buffer: a lane stores only what it loaded itself.
constexpr int kSmBlockMaxThreads = 1024;
constexpr int kSmBlockMaxVpl = 8;

template <typename T, int VPL>
__global__ __launch_bounds__(kSmBlockMaxThreads, 4) void softmax_block_kernel(const T *x, T *y, uint32_t row_vecs,
                                                                            int stable, uint32_t nt) {
    constexpr int EPV = Store<T>::EPV;
    __shared__ float slots_max[kSmBlockMaxThreads / kWave], slots_sum[kSmBlockMaxThreads / kWave];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1), wave = tid / kWave, waves = nt / kWave;
    const size_t row_base = (size_t)blockIdx.x * row_vecs;
    const u32x4 *in = reinterpret_cast<const u32x4 *>(x) + row_base;
    u32x4 *out = reinterpret_cast<u32x4 *>(y) + row_base;
    u32x4 raw[VPL];
#pragma unroll
    for (int v = 0; v < VPL; v++) raw[v] = load_stream(in + min(v * nt + tid, row_vecs - 1));
    float f[VPL][EPV];
    float mx = kNegInf;
#pragma unroll
    for (int v = 0; v < VPL; v++) {
        Store<T>::unpack(raw[v], f[v]);
        const bool have = v * nt + tid < row_vecs;
#pragma unroll
        for (int e = 0; e < EPV; e++) {
            f[v][e] = have ? f[v][e] : kNegInf;  // padding: exp gives 0
            mx = fmaxf(mx, f[v][e]);
        }
    }
    float shift = 0.0f;
    if (stable) {
        mx = team_max<64>(mx);
        if (lane == 0) slots_max[wave] = mx;
        __syncthreads();
        shift = team_max<64>(lane < waves ? slots_max[lane] : kNegInf);
        shift = shift == kNegInf ? 0.0f : shift;  // a row of -inf: keep the reference's 0/0
    }
    const float bias = -shift * kLog2e;
    float total = 0.0f;
#pragma unroll
    for (int v = 0; v < VPL; v++)
#pragma unroll
        for (int e = 0; e < EPV; e++) {
            f[v][e] = __builtin_amdgcn_exp2f(fmaf(f[v][e], kLog2e, bias));
            total += f[v][e];
        }
    total = wave_sum(total);
    if (lane == 0) slots_sum[wave] = total;
    __syncthreads();
    const float inv = 1.0f / wave_sum(lane < waves ? slots_sum[lane] : 0.0f);
#pragma unroll
    for (int v = 0; v < VPL; v++) {
#pragma unroll
        for (int e = 0; e < EPV; e++) f[v][e] *= inv;
        if (v * nt + tid < row_vecs) store_stream(out + v * nt + tid, Store<T>::pack(f[v]));
    }
}

// Any row length / alignment: one wavefront per row, lane-strided elements, the row
// re-read from cache for each of the (up to) three passes.
template <typename T>
__global__ __launch_bounds__(kSmThreads) void softmax_generic_kernel(const T *x, T *y, uint32_t rows,
                                                                     uint32_t cols, int stable) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t row = blockIdx.x * (kSmThreads / kWave) + threadIdx.x / kWave;
    if (row >= rows) return;
    const T *in = x + (size_t)row * cols;
    T *out = y + (size_t)row * cols;
    float shift = 0.0f;
    if (stable) {
        float mx = kNegInf;
        for (uint32_t c = lane; c < cols; c += kWave) mx = fmaxf(mx, Store<T>::load1(in + c));
        mx = team_max<64>(mx);
        shift = mx == kNegInf ? 0.0f : mx;
    }
    const float bias = -shift * kLog2e;
    float total = 0.0f;
    for (uint32_t c = lane; c < cols; c += kWave)
        total += __builtin_amdgcn_exp2f(fmaf(Store<T>::load1(in + c), kLog2e, bias));
    total = wave_sum(total);
    const float inv = 1.0f / total;
    // in place: every element of the row has been read by now, and a lane rewrites only
    // the elements it reads itself in this pass
    for (uint32_t c = lane; c < cols; c += kWave) {
        const float e = __builtin_amdgcn_exp2f(fmaf(Store<T>::load1(in + c), kLog2e, bias));
        Store<T>::store1(out + c, e * inv);
    }
}

// Short rows without alignment (77 text tokens): the whole row in ITERS registers per
// lane, one read and one write per element.
template <typename T, int ITERS>
__global__ __launch_bounds__(kSmThreads) void softmax_short_kernel(const T *x, T *y, uint32_t rows,
                                                                   uint32_t cols, int stable) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t row = blockIdx.x * (kSmThreads / kWave) + threadIdx.x / kWave;
    if (row >= rows) return;
    const T *in = x + (size_t)row * cols;
    T *out = y + (size_t)row * cols;
    float f[ITERS];
    float mx = kNegInf;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const uint32_t c = lane + i * kWave;
        const float v = Store<T>::load1(in + min(c, cols - 1));
        f[i] = c < cols ? v : kNegInf;
        mx = fmaxf(mx, f[i]);
    }
    float shift = 0.0f;
    if (stable) {
        mx = team_max<64>(mx);
        shift = mx == kNegInf ? 0.0f : mx;
    }
    const float bias = -shift * kLog2e;
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        f[i] = __builtin_amdgcn_exp2f(fmaf(f[i], kLog2e, bias));
        total += f[i];
    }
    total = wave_sum(total);
    const float inv = 1.0f / total;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const uint32_t c = lane + i * kWave;
        if (c < cols) Store<T>::store1(out + c, f[i] * inv);
    }
}

// Short rows whose length is not a multiple of a 16-byte vector (77 text tokens): a
// workgroup takes RB consecutive rows (RB a multiple of 8) as one flat, 16-byte aligned
// run of memory (such a block is a whole number of vectors for any row length), moves it
// through LDS with full vectors, and a team of 4, 8 or 16 lanes per row does the arithmetic
// on the LDS copy.
constexpr uint32_t kSmFlatMaxCols = 128;  // RB = 64: 16 or 32 KiB of LDS

template <typename T, int RB, int ITERS, int TEAM>
__global__ __launch_bounds__(RB * TEAM) void softmax_flat_kernel(const T *x, T *y, uint32_t cols, int stable) {
    constexpr int EPV = Store<T>::EPV;
    constexpr int NT = RB * TEAM;
    constexpr int UN = 4;
    // [RB][cols] in the storage type: whole vectors go in and out as they are (one 16-byte LDS
    // access per vector), only the arithmetic in between touches single elements
    extern __shared__ u32x4 tile_vec[];
    T *tile = reinterpret_cast<T *>(tile_vec);
    const uint32_t block_vecs = RB * cols / EPV;
    const size_t first = (size_t)blockIdx.x * block_vecs;
    const u32x4 *in = reinterpret_cast<const u32x4 *>(x) + first;
    u32x4 *out = reinterpret_cast<u32x4 *>(y) + first;
    for (uint32_t base = threadIdx.x; base < block_vecs; base += NT * UN) {
        u32x4 raw[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) raw[u] = load_stream(in + min(base + u * NT, block_vecs - 1));
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const uint32_t v = base + u * NT;
            if (v < block_vecs) tile_vec[v] = raw[u];
        }
    }
    __syncthreads();
    // the lane's share of its row, from LDS into registers with independent reads
    T *row = tile + (threadIdx.x / TEAM) * cols;
    const uint32_t j = threadIdx.x % TEAM;
    float f[ITERS];
    float mx = kNegInf;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const uint32_t c = j + i * TEAM;
        f[i] = c < cols ? Store<T>::load1(row + c) : kNegInf;
        mx = fmaxf(mx, f[i]);
    }
    float shift = 0.0f;
    if (stable) {
        mx = team_max<TEAM>(mx);
        shift = mx == kNegInf ? 0.0f : mx;
    }
    const float bias = -shift * kLog2e;
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        f[i] = __builtin_amdgcn_exp2f(fmaf(f[i], kLog2e, bias));
        total += f[i];
    }
    total = team_sum<TEAM>(total);
    const float inv = 1.0f / total;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const uint32_t c = j + i * TEAM;
        if (c < cols) Store<T>::store1(row + c, f[i] * inv);
    }
    __syncthreads();
    for (uint32_t v = threadIdx.x; v < block_vecs; v += NT) store_stream(out + v, tile_vec[v]);
}

template <typename T, int RB, int TEAM>
void softmax_flat_launch(const T *x, T *y, uint32_t blocks, uint32_t cols, int stable, hipStream_t stream) {
    const size_t lds = (size_t)RB * cols * sizeof(T);  // a whole number of 16-byte vectors: RB is a multiple of 8
    constexpr int kFew = (80 + TEAM - 1) / TEAM, kMany = kSmFlatMaxCols / TEAM;
    if (cols <= 80)
        launch((softmax_flat_kernel<T, RB, kFew, TEAM>), dim3(blocks), dim3(RB * TEAM), lds, stream, x, y, cols, stable);
    else
        launch((softmax_flat_kernel<T, RB, kMany, TEAM>), dim3(blocks), dim3(RB * TEAM), lds, stream, x, y, cols, stable);
}

// ---------------------------------------------------------------------------
// DDIM update (eta = 0): the three float loops of the replaced host code as one pass,
// with individually rounded operations in the same order, so float32 storage gives
// the host loop's bits.
// ---------------------------------------------------------------------------
constexpr int kDdimThreads = 256;

struct DdimCoef {
    float sqrt_one_minus_at, sqrt_at, sqrt_one_minus_aprev, sqrt_aprev;
};

__device__ __forceinline__ float ddim_one(float x, float e, const DdimCoef &c) {
#pragma clang fp contract(off)  // no fused multiply-add: each product is rounded before it is added
    const float scaled = c.sqrt_one_minus_at * e;
    const float pred_x0 = (x - scaled) / c.sqrt_at;  // IEEE division (hipcc's default for float)
    const float dir_xt = c.sqrt_one_minus_aprev * e;
    const float back = c.sqrt_aprev * pred_x0;
    return back + dir_xt;
}

template <typename T>
__global__ __launch_bounds__(kDdimThreads) void ddim_update_kernel(const T *x, const T *e_t, T *x_prev, size_t n,
                                                                   int vectors, uint32_t blocks, DdimCoef c) {
    constexpr int EPV = Store<T>::EPV;
    const size_t stride = (size_t)blocks * kDdimThreads;
    const size_t first = (size_t)blockIdx.x * kDdimThreads + threadIdx.x;
    if (vectors) {
        const size_t vecs = n / EPV;
        for (size_t v = first; v < vecs; v += stride) {
            float a[EPV], b[EPV], r[EPV];
            Store<T>::unpack(reinterpret_cast<const u32x4 *>(x)[v], a);
            Store<T>::unpack(reinterpret_cast<const u32x4 *>(e_t)[v], b);
#pragma unroll
            for (int i = 0; i < EPV; i++) r[i] = ddim_one(a[i], b[i], c);
            reinterpret_cast<u32x4 *>(x_prev)[v] = Store<T>::pack(r);
        }
        for (size_t i = vecs * EPV + first; i < n; i += stride)
            Store<T>::store1(x_prev + i, ddim_one(Store<T>::load1(x + i), Store<T>::load1(e_t + i), c));
    } else {
        for (size_t i = first; i < n; i += stride)
            Store<T>::store1(x_prev + i, ddim_one(Store<T>::load1(x + i), Store<T>::load1(e_t + i), c));
    }
}

template <typename T, int M>
void linear_launch(const T *x, const T *w, const float *bias, T *y, uint32_t m, uint32_t n, uint32_t k,
                   int act_in, int act_out, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    if (act_in)  // two columns per wavefront share the activated x
        launch((linear_rows_kernel<T, M, 2>), dim3((n + 1) / 2), dim3(kWave), 0, stream, x, w, bias,
                           y, m, n, k / EPV, act_in, act_out);
    else
        launch((linear_rows_kernel<T, M, 1>), dim3(n), dim3(kWave), 0, stream, x, w, bias, y, m, n,
                           k / EPV, act_in, act_out);
}

// Three to eight rows of 2-byte elements on the matrix cores, with the bits of a column or two per wavefront: always where x is
// activated, once for four wavefronts instead of in each (us, column per wavefront and so: 64 columns of k = 320 2.97 / 2.89,
// 1280 of 320 3.52 / 3.13, 1280 of 1280 3 rows 4.92 / 3.55, 8 rows 7.60 / 4.37); else from as many columns on as fill the
// chip anyway (3 rows, k = 1280: 640 columns 3.33 / 3.51, 1280 3.95 / 3.53, 5120 6.64 / 5.57; 8 rows, 320 columns 3.78 / 3.94, 640
// 4.30 / 4.11, 1280 5.53 / 4.10, 5120 11.4 / 6.92).
template <typename T>
bool linear_takes_quads(size_t m, size_t n, int act_in) {
    return sizeof(T) == 2 && m >= 3 && (act_in || n >= (m <= 4 ? 1280u : 640u));
}

// Column quads of a workgroup: two, with three pieces of each row in flight, while the launch is short; four, with one
// piece and less of x to read and activate per column, when it lasts (us, two and four, k = 1280, with SiLU: 8192 columns 3 rows
// 7.62 / 9.24, 8 rows 9.64 / 10.8; 10240 8.39 / 9.05 and 11.1 / 11.3; 20160 13.0 / 12.8 and 18.1 / 15.8).
constexpr int linear_column_quads(size_t n) { return n >= 12288 ? 4 : 2; }

// Calls `f` with an instance's parameters: row quads, column quads, pieces in flight, SiLU on the input.
template <typename F>
void linear_quads(size_t m, size_t n, int act_in, F f) {
    auto with_rows = [&](auto cols, auto round) {
        auto with_act = [&](auto rows) {
            if (act_in) f(rows, cols, round, std::true_type{});
            else f(rows, cols, round, std::false_type{});
        };
        if (m <= 4) with_act(std::integral_constant<int, 1>{});
        else with_act(std::integral_constant<int, 2>{});
    };
    if (linear_column_quads(n) == 4) with_rows(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
    else with_rows(std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{});
}

template <typename T, int VPL, int TL, bool RAGGED>
void softmax_team_launch(const T *x, T *y, uint32_t rows, uint32_t cols, int stable, hipStream_t stream) {
    constexpr uint32_t threads = softmax_team_lanes(VPL, TL);
    constexpr uint32_t rows_per_block = (threads / kWave) * (kWave / TL);
    launch((softmax_team_kernel<T, VPL, TL, RAGGED>), dim3((rows + rows_per_block - 1) / rows_per_block),
                       dim3(threads), 0, stream, x, y, rows, cols, stable);
}

// How many rows are open at once: 48 KB of them a CU as soon as the launch fills the chip many times (us with 2, 3, 4, 5,
// 6 rows a CU: fp16 82944 x 5184 329 285 275 274 273, 147456 x 9216 899 932 929; fp32 65536 x 4096 343 335 334 336,
// 102400 x 6400 862 906); fewer rows are better served all at once (fp16 1000 x 9216, two rows a CU 10.4, no limit 7.8).
// Vectors per lane: with the limit enough wavefronts for the exponentials and no more (2 / 4 / 8 us: fp16 36864 x 2304
// 55.0 / 55.7, 82944 x 5184 275 / 275 / 493, fp32 49152 x 3072 190 / 191 / 188, 102400 x 6400 900 / 896 / 862); without,
// many short lanes (2 / 4 / 8: fp16 4096 x 4096 12.8 / 12.9 / 13.4, 1024 x 9216 8.8 / 7.4 / 10.6, 16 x 9216 2.8 / 3.0 / 4.6,
// fp32 4096 x 6400 33.7 / 35.3 / 34.8, 16 x 6400 2.5 / 2.5 / 2.7).
constexpr size_t kSmOpenBytes = 48 * 1024;
constexpr size_t kLdsPerCu = 160 * 1024, kSmMostLds = 60 * 1024;
constexpr size_t kSmLimitRounds = 16;  // the limit holds for launches of this many times the rows then in flight

template <typename T>
void softmax_block_launch(const T *x, T *y, uint32_t rows, uint32_t row_vecs, int stable, hipStream_t stream) {
    const size_t open = std::max<size_t>(kSmOpenBytes / (row_vecs * 16), 2);  // rows a CU holds: at most 11
    const bool limit = row_vecs <= 4096 && rows >= kSmLimitRounds * open * chip_info().cus;
    // one workgroup's share of the LDS, less what it has anyway: `open` of them fit a CU, one more does not
    const size_t lds = limit ? std::min(kLdsPerCu / open - 1024, kSmMostLds) : 0;
    uint32_t vpl = sizeof(T) == 2 ? (row_vecs <= (limit ? 320u : 512u) ? 2 : 4) : !limit ? 2 : row_vecs <= 1344 ? 4 : 8;
    auto lanes = [&]() { return ((row_vecs + vpl - 1) / vpl + kWave - 1) / kWave * kWave; };
    while (lanes() > (uint32_t)kSmBlockMaxThreads) vpl = vpl == 2 && sizeof(T) == 4 ? 3 : vpl < 4 ? 4 : 8;
    const dim3 block(lanes());
    auto *kernel = vpl == 8 ? softmax_block_kernel<T, 8> : vpl == 4 ? softmax_block_kernel<T, 4> : softmax_block_kernel<T, 2>;
    if (vpl == 3) kernel = softmax_block_kernel<T, sizeof(T) == 4 ? 3 : 2>;
    constexpr uint32_t kMostRows = 0xFFFFFFFFu / kSmBlockMaxThreads;  // (a grid holds less than 2^32 lanes)
    for (uint32_t done = 0; done < rows; done += kMostRows) {
        const dim3 grid(min(rows - done, kMostRows));
        const T *xs = x + (size_t)done * row_vecs * Store<T>::EPV;
        T *ys = y + (size_t)done * row_vecs * Store<T>::EPV;
        launch(kernel, grid, block, lds, stream, xs, ys, row_vecs, stable, block.x);
        if (rows - done <= kMostRows) break;
    }
}

// A row of 257 vectors up to what a wavefront's registers hold (512 of 2-byte storage, whose floats take twice the
// room, 1024 of 4-byte): a workgroup per row where the rows leave CUs idle or fill the chip many times, a wavefront per
// row between.  us, wavefront and workgroup: fp16 16 x 3072 2.67 / 2.38, 256 x 4096 3.20 / 2.91, 1024 x 3072 stable 4.15 /
// 4.32, 4096 x 2304 stable 8.88 / 9.32, 8192 x 4096 23.3 / 22.6, 36864 x 2304 55.7 / 53.4, 49152 x 3072 95.8 / 93.6, 65536 x 4096
// 169.4 / 168.3 (8192 to 131072 fp16 rows of 2056 to 4096, 192 launches: 0.96 up to 2304 columns, 0.98 - 0.99 from 3584 on, none
// slower by more than two runs differ); fp32 16 x 3072 2.58 / 2.03,
// 2048 x 4096 11.2 / 12.7, 2048 x 2304 7.14 / 8.4, 3072 x 3072 14.6 / 13.9, 8192 x 4096 44.8 / 42.1.
template <typename T>
bool softmax_wave_per_row(uint32_t rows, uint32_t row_vecs) {
    const uint32_t cus = chip_info().cus;
    return row_vecs <= 256 || (row_vecs <= (sizeof(T) == 2 ? 512u : 1024u) && rows > cus && rows < (sizeof(T) == 2 ? 32u : 12u) * cus);
}

}  // namespace

template <typename T>
int linear_rows_dispatch(const void *xv, const void *wv, const float *bias, void *yv, size_t m,
                         size_t n, size_t k, int act_in, int act_out, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const T *x = static_cast<const T *>(xv);
    const T *w = static_cast<const T *>(wv);
    T *y = static_cast<T *>(yv);
    if (m == 0 || n == 0) return MSD_OK;
    if (m > 8 || n > 0x7FFFFFFFull || k > 0x7FFFFFFFull) return MSD_ERR_INVALID_VALUE;
    const uint32_t m_pad = m <= 1 ? 1 : m <= 2 ? 2 : m <= 4 ? 4 : 8;
    const bool vectors = k != 0 && k % EPV == 0 && aligned16(x) && aligned16(w);
    if (vectors && linear_takes_quads<T>(m, n, act_in)) {
        linear_quads(m, n, act_in, [&](auto rows, auto quads, auto round, auto act) {
            launch((linear_quads_kernel<rows, quads, round, act>), dim3((uint32_t)((n + kLinBlock * quads - 1) / (kLinBlock * quads))),
                   dim3(kLinWgThreads), 0, stream, static_cast<const __half *>(xv), static_cast<const __half *>(wv), bias,
                   static_cast<__half *>(yv), (uint32_t)m, (uint32_t)n, (uint32_t)(k / EPV), act_out);
        });
    } else if (vectors) {
        switch (m_pad) {
            case 1: linear_launch<T, 1>(x, w, bias, y, (uint32_t)m, (uint32_t)n, (uint32_t)k, act_in, act_out, stream); break;
            case 2: linear_launch<T, 2>(x, w, bias, y, (uint32_t)m, (uint32_t)n, (uint32_t)k, act_in, act_out, stream); break;
            case 4: linear_launch<T, 4>(x, w, bias, y, (uint32_t)m, (uint32_t)n, (uint32_t)k, act_in, act_out, stream); break;
            default: linear_launch<T, 8>(x, w, bias, y, (uint32_t)m, (uint32_t)n, (uint32_t)k, act_in, act_out, stream); break;
        }
    } else {
        const uint32_t blocks = (uint32_t)((n + kLinWaves - 1) / kLinWaves);
        launch((linear_rows_generic_kernel<T>), dim3(blocks), dim3(kLinThreads), 0, stream, x,
                           w, bias, y, (uint32_t)m, (uint32_t)n, (uint32_t)k, act_in, act_out);
    }
    return launch_status();
}

namespace {

template <typename T, int M>
void linear_grouped_launch(const T *x, const LinearGroup &g, uint32_t m, uint32_t k, int act_in, int act_out,
                           int cpw, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const uint32_t blocks = g.first_block[g.count];
    if (cpw == 4 && k / EPV > 128 && k / EPV <= 192)  // three pieces per lane cover the row (k = 1280: 3 % faster)
        launch((linear_rows_grouped_kernel<__half, (M <= 2 ? M : 1), 4, 3>), dim3(blocks), dim3(kWave), 0,
                           stream, reinterpret_cast<const __half *>(x), g, m, k / EPV, act_in, act_out);
    else if (cpw == 4)  // (only 2-byte elements and up to two rows: see the dispatch)
        launch((linear_rows_grouped_kernel<__half, (M <= 2 ? M : 1), 4>), dim3(blocks), dim3(kWave), 0,
                           stream, reinterpret_cast<const __half *>(x), g, m, k / EPV, act_in, act_out);
    else if (cpw == 2)
        launch((linear_rows_grouped_kernel<T, M, 2>), dim3(blocks), dim3(kWave), 0, stream, x, g, m,
                           k / EPV, act_in, act_out);
    else
        launch((linear_rows_grouped_kernel<T, M, 1>), dim3(blocks), dim3(kWave), 0, stream, x, g, m,
                           k / EPV, act_in, act_out);
}

}  // namespace

template <typename T>
int linear_rows_grouped_dispatch(const void *xv, const void *const *ws, const float *const *biases,
                                 void *const *ys, const size_t *ns, size_t count, size_t m, size_t k,
                                 int act_in, int act_out, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const T *x = static_cast<const T *>(xv);
    if (m == 0 || count == 0) return MSD_OK;
    if (m > 8 || k > 0x7FFFFFFFull) return MSD_ERR_INVALID_VALUE;
    bool vectors = k != 0 && k % EPV == 0 && aligned16(x);
    for (size_t i = 0; i < count; i++) {
        if (ns[i] > 0x7FFFFFFFull) return MSD_ERR_INVALID_VALUE;
        vectors = vectors && aligned16(ws[i]);
    }
    if (!vectors) {  // odd k or alignment: one launch of the scalar kernel per problem
        for (size_t i = 0; i < count; i++) {
            const int rc = linear_rows_dispatch<T>(xv, ws[i], biases ? biases[i] : nullptr, ys[i], m, ns[i], k,
                                                   act_in, act_out, stream);
            if (rc != MSD_OK) return rc;
        }
        return MSD_OK;
    }
    const uint32_t m_pad = m <= 1 ? 1 : m <= 2 ? 2 : m <= 4 ? 4 : 8;
    // Columns per wavefront: with SiLU on the input every wavefront activates its own copy of x, so
    // columns share that work: two as in the single launch, four when the launch is large enough
    // to fill the chip anyway: fewer, longer wavefronts also stream the weights faster, with or
    // without the activation (the 22 projections of a step, 20160 columns of fp16: 15.3 us with
    // two, 12.2 us with four, 14.6 with eight; without SiLU 13.8 us with one, 11.3 with four; a
    // single 1280-column layer is slower with four, 4.25 against 3.91 us, and 4-byte elements run
    // out of registers).  The sums do not depend on it.
    size_t total_n = 0;
    for (size_t i = 0; i < count; i++) total_n += ns[i];
    const bool quads = linear_takes_quads<T>(m, total_n, act_in);
    const bool shared = sizeof(T) == 4 && m >= 2 && total_n >= 8192;  // (fewer columns leave it too few workgroups)
    const int cpw = quads ? kLinBlock * linear_column_quads(total_n) : shared ? kLinWgWaves * kSharedCols  // (columns of a workgroup)
                    : (sizeof(T) == 2 && m_pad <= 2 && total_n >= 8192) ? 4 : act_in ? 2 : 1;
    for (size_t base = 0; base < count; base += kLinGroupMax) {
        LinearGroup g;
        g.count = 0;
        uint32_t blocks = 0;
        for (size_t i = base; i < count && i < base + kLinGroupMax; i++) {
            if (ns[i] == 0) continue;
            const uint32_t slot = g.count++;
            g.w[slot] = ws[i];
            g.bias[slot] = biases ? biases[i] : nullptr;
            g.y[slot] = ys[i];
            g.n[slot] = (uint32_t)ns[i];
            g.first_block[slot] = blocks;
            blocks += (uint32_t)((ns[i] + cpw - 1) / cpw);
        }
        if (g.count == 0) continue;
        g.first_block[g.count] = blocks;
        auto rows_in_lds = [&](auto *kernel) {
            launch(kernel, dim3(blocks), dim3(kLinWgThreads), 0, stream, static_cast<const float *>(xv), g, (uint32_t)m,
                   (uint32_t)(k / EPV), act_in, act_out);
        };
        if (quads)
            linear_quads(m, total_n, act_in, [&](auto rows, auto cols, auto round, auto act) {
                launch((linear_quads_grouped_kernel<rows, cols, round, act>), dim3(blocks), dim3(kLinWgThreads), 0, stream,
                       static_cast<const __half *>(xv), g, (uint32_t)m, (uint32_t)(k / EPV), act_out);
            });
        else if (shared && m_pad == 2) rows_in_lds(linear_shared_grouped_kernel<2>);
        else if (shared && m_pad == 4) rows_in_lds(linear_shared_grouped_kernel<4>);
        else if (shared) rows_in_lds(linear_shared_grouped_kernel<8>);
        else switch (m_pad) {
            case 1: linear_grouped_launch<T, 1>(x, g, (uint32_t)m, (uint32_t)k, act_in, act_out, cpw, stream); break;
            case 2: linear_grouped_launch<T, 2>(x, g, (uint32_t)m, (uint32_t)k, act_in, act_out, cpw, stream); break;
            case 4: linear_grouped_launch<T, 4>(x, g, (uint32_t)m, (uint32_t)k, act_in, act_out, cpw, stream); break;
            default: linear_grouped_launch<T, 8>(x, g, (uint32_t)m, (uint32_t)k, act_in, act_out, cpw, stream); break;
        }
        const int rc = launch_status();
        if (rc != MSD_OK) return rc;
    }
    return MSD_OK;
}

template <typename T>
int softmax_dispatch(const void *xv, void *yv, size_t rows, size_t cols, int stable, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const T *x = static_cast<const T *>(xv);
    T *y = static_cast<T *>(yv);
    if (rows == 0 || cols == 0) return MSD_OK;
    constexpr size_t waves_per_block = kSmThreads / kWave;
    if (rows > 0x7FFFFFFFull || cols > 0x7FFFFFFFull) return MSD_ERR_INVALID_VALUE;
    const uint32_t r = (uint32_t)rows, c = (uint32_t)cols;
    const size_t row_vecs = cols / EPV;
    const bool vec_ok = cols % EPV == 0 && aligned16(x) && aligned16(y) &&
                        row_vecs <= (size_t)kSmBlockMaxThreads * kSmBlockMaxVpl;
    if (vec_ok) {
        const uint32_t rv = (uint32_t)row_vecs;
        // up to 64 vectors per row: one vector per lane on the smallest team that holds the row
        // (measured against two or four vectors per lane on smaller teams at 4 ... 32 vectors per
        // row, 2048 ... 524288 rows of fp16: never slower, 25-vector rows 71 against 109 us, 4-vector
        // rows 12.9 against 17.1, 32-vector rows 2.4 against 2.7 us at 2048 rows)
        if (!softmax_wave_per_row<T>(r, rv)) softmax_block_launch<T>(x, y, r, rv, stable, stream);
        else if (rv <= 4) softmax_team_launch<T, 1, 4, false>(x, y, r, c, stable, stream);
        else if (rv <= 8) softmax_team_launch<T, 1, 8, false>(x, y, r, c, stable, stream);
        else if (rv <= 16) softmax_team_launch<T, 1, 16, false>(x, y, r, c, stable, stream);
        else if (rv <= 32) softmax_team_launch<T, 1, 32, false>(x, y, r, c, stable, stream);
        else if (rv <= 64) softmax_team_launch<T, 1, 64, false>(x, y, r, c, stable, stream);
        else if (rv <= 128) softmax_team_launch<T, 2, 64, false>(x, y, r, c, stable, stream);
        else if (rv <= 256) softmax_team_launch<T, 4, 64, false>(x, y, r, c, stable, stream);
        else if (rv <= 512) softmax_team_launch<T, 8, 64, false>(x, y, r, c, stable, stream);
        else softmax_team_launch<T, sizeof(T) == 4 ? 16 : 8, 64, false>(x, y, r, c, stable, stream);  // (fp16: no such row)
        return launch_status();
    }
    // The flat kernel pays two barriers and two LDS round trips; below about 12000 rows the
    // row-per-wavefront kernel is quicker (3.08 against 3.10 us at 10240 x 77, 3.26 against 3.18
    // at 12288).  Lanes per row: as many as keep the launch within the 8192 wavefronts the chip
    // holds at once (a second round of wavefronts costs more than the shorter serial chain per
    // lane gains: 16 lanes per row take 4.09 us at 32768 x 77 and 7.08 at 65536, 8 lanes 4.52 and
    // 5.76); past one round 4 lanes per row are the cheapest for up to 80 columns, 8 beyond.
    // A set knob forces the flat kernel and its rows per workgroup for any size.
    const int tune_rows = g_tuning.softmax_rows.load(std::memory_order_relaxed);
    const uint32_t team = rows <= 32768 ? 16u : rows <= 65536 ? 8u : cols <= 80 ? 4u : 8u;
    // workgroups of 512 lanes up to 80 columns, of 256 beyond, and at most 64 rows
    const uint32_t lanes = cols <= 80 ? 512u : 256u;
    const uint32_t rb = tune_rows ? (uint32_t)tune_rows : lanes / team > 64u ? 64u : lanes / team;
    const bool flat_pays = tune_rows ? rows >= rb : rows >= 12288;
    if (cols <= kSmFlatMaxCols && cols >= 8 && flat_pays && aligned16(x) && aligned16(y)) {
        // whole blocks of rb rows through the flat kernel, the rest (if any) row by row below
        const uint32_t blocks = r / rb;
        switch (team * 100 + rb) {
            case 464: softmax_flat_launch<T, 64, 4>(x, y, blocks, c, stable, stream); break;
            case 432: softmax_flat_launch<T, 32, 4>(x, y, blocks, c, stable, stream); break;
            case 416: softmax_flat_launch<T, 16, 4>(x, y, blocks, c, stable, stream); break;
            case 864: softmax_flat_launch<T, 64, 8>(x, y, blocks, c, stable, stream); break;
            case 832: softmax_flat_launch<T, 32, 8>(x, y, blocks, c, stable, stream); break;
            case 816: softmax_flat_launch<T, 16, 8>(x, y, blocks, c, stable, stream); break;
            case 1664: softmax_flat_launch<T, 64, 16>(x, y, blocks, c, stable, stream); break;
            case 1632: softmax_flat_launch<T, 32, 16>(x, y, blocks, c, stable, stream); break;
            default: softmax_flat_launch<T, 16, 16>(x, y, blocks, c, stable, stream); break;
        }
        const uint32_t done = blocks * rb;
        if (done == r) return launch_status();
        x += (size_t)done * c;
        y += (size_t)done * c;
        rows -= done;
    }
    const uint32_t r_left = (uint32_t)rows;
    const dim3 grid((uint32_t)((rows + waves_per_block - 1) / waves_per_block));
    const size_t pieces = (cols + EPV - 1) / EPV;
    // Up to 512 columns, element by element or in 16-byte pieces: what the pieces save in accesses they pay in
    // latency (a cut piece is a chain of loads, and pieces that start at any element touch more lines), so they need
    // rows enough, and more of them the less their starts are aligned.  Over random shapes, pieces against elements:
    // fp16 up to 256 columns and 1000 / 4000 / 8000 / 32000 rows, odd 1.14 / 1.03 / 0.93 / 0.79, even 1.09 / 0.95 /
    // 0.86 / 0.70; fp16 beyond 256, odd and even 1.02 - 1.17 at any number of rows, multiples of four 1.04 below
    // 8000 rows and 0.96 from there on; fp32 up to 256, odd 0.99 - 1.07, even 1.03 below 6000 rows and 0.93 above,
    // beyond 256 1.01 - 1.14.
    bool pieces_pay = cols > 8 * kWave;
    if (sizeof(T) == 2)
        pieces_pay = pieces_pay || (cols <= 256 ? rows >= (cols % 2 ? 5120u : 3072u) : cols % 4 == 0 && rows >= 8192);
    else
        pieces_pay = pieces_pay || (cols <= 256 && cols % 2 == 0 && rows >= 6144);
    if (cols <= 2 * kWave) launch((softmax_short_kernel<T, 2>), grid, dim3(kSmThreads), 0, stream, x, y, r_left, c, stable);
    else if (!pieces_pay) launch((softmax_short_kernel<T, 8>), grid, dim3(kSmThreads), 0, stream, x, y, r_left, c, stable);
    else if (pieces <= 32) softmax_team_launch<T, 1, EPV == 8 ? 32 : 64, true>(x, y, r_left, c, stable, stream);  // (fp32: no such row)
    else if (pieces <= 64) softmax_team_launch<T, 1, 64, true>(x, y, r_left, c, stable, stream);
    else if (pieces <= 128) softmax_team_launch<T, 2, 64, true>(x, y, r_left, c, stable, stream);
    else if (pieces <= 256) softmax_team_launch<T, 4, 64, true>(x, y, r_left, c, stable, stream);
    else if (pieces <= 512) softmax_team_launch<T, 8, 64, true>(x, y, r_left, c, stable, stream);
    else
        launch((softmax_generic_kernel<T>), grid, dim3(kSmThreads), 0, stream, x, y, r_left, c, stable);
    return launch_status();
}

template <typename T>
int ddim_update_dispatch(const void *xv, const void *ev, void *yv, size_t n, float a_t, float a_prev,
                         float sqrt_one_minus_at, hipStream_t stream) {
    if (n == 0) return MSD_OK;
    DdimCoef c;
    c.sqrt_one_minus_at = sqrt_one_minus_at;
    c.sqrt_at = sqrtf(a_t);  // correctly rounded on the host, as in the replaced loop
    c.sqrt_one_minus_aprev = sqrtf(1.0f - a_prev);
    c.sqrt_aprev = sqrtf(a_prev);
    const int vectors = aligned16(xv) && aligned16(ev) && aligned16(yv);
    const size_t want = (n / Store<T>::EPV + kDdimThreads) / kDdimThreads;
    const uint32_t blocks = (uint32_t)(want < 4096 ? want : 4096);
    launch((ddim_update_kernel<T>), dim3(blocks), dim3(kDdimThreads), 0, stream, static_cast<const T *>(xv),
           static_cast<const T *>(ev), static_cast<T *>(yv), n, vectors, blocks, c);
    return launch_status();
}

template int linear_rows_dispatch<float>(const void *, const void *, const float *, void *, size_t, size_t, size_t, int, int, hipStream_t);
template int linear_rows_dispatch<__half>(const void *, const void *, const float *, void *, size_t, size_t, size_t, int, int, hipStream_t);
template int linear_rows_grouped_dispatch<float>(const void *, const void *const *, const float *const *, void *const *,
                                                 const size_t *, size_t, size_t, size_t, int, int, hipStream_t);
template int linear_rows_grouped_dispatch<__half>(const void *, const void *const *, const float *const *, void *const *,
                                                  const size_t *, size_t, size_t, size_t, int, int, hipStream_t);
template int softmax_dispatch<float>(const void *, void *, size_t, size_t, int, hipStream_t);
template int softmax_dispatch<__half>(const void *, void *, size_t, size_t, int, hipStream_t);
template int ddim_update_dispatch<float>(const void *, const void *, void *, size_t, float, float, float, hipStream_t);
template int ddim_update_dispatch<__half>(const void *, const void *, void *, size_t, float, float, float, hipStream_t);

}  // namespace msd
