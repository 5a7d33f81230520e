// Streaming kernels for gfx950: the GEGLU epilogue, elementwise SiLU / GELU /
// quick_GELU and the sinusoidal timestep embedding.  Flat 16-byte accesses, U
// vectors per lane with every load issued before the first use; all workgroups
// but a ragged last one run branch-free.
#include "msd_device.h"
#include "msd_internal.h"
#include "tile_transpose.h"

#include <cmath>
#include <type_traits>

namespace msd {
namespace {

constexpr int kStreamThreads = 256;
// GEGLU runs one wavefront per workgroup: with two loads and 21 VALU instructions per element
// in flight per lane, single-wavefront workgroups start and retire soonest (measured 4.5 %
// faster over the step's 16 launches than 256-lane workgroups).
constexpr int kGegluThreads = 64;
// Lanes of a workgroup of the elementwise kernels: one wavefront in launches with more wavefronts than the chip has room for
// (32 per CU), where a wavefront that starts and retires by itself keeps the launch moving through memory in order.  Shorter launches
// start sooner in workgroups of four.  Sums of two tensors gain from 22 wavefronts per CU on, where workgroups of four leave some
// CUs one more than others; passes over one tensor from 48.  us, 256 lanes and 64, at 5200 / 6144 / 9216 / 11264 / 14336
// wavefronts: fp16 add 4.16 / 4.95 / 6.37 / 7.87 / 9.23 and 4.15 / 4.62 / 6.00 / 7.31 / 8.71, copy 3.03 / 3.24 / 4.59 / 5.71 / 6.88 and
// 3.60 / 3.80 / 4.69 / 5.82 / 6.62, fp32 SiLU 3.04 / 3.24 / 4.64 / 5.87 / 6.98 and 3.66 / 3.88 / 4.84 / 5.86 / 6.76; fp16 add of 34 M
// elements 33.1 and 31.8, copy of 42 / 540 MB 15.8 / 167 and 14.5 / 163 (6.6 TB/s).
inline uint32_t stream_lanes(size_t vecs, bool two_tensors) {
    const size_t most = (two_tensors ? 22 : 48) * (size_t)kWave * chip_info().cus;
    return vecs > most ? (uint32_t)kWave : (uint32_t)kStreamThreads;
}
constexpr int kStreamUnroll = 1;  // vectors per lane of the elementwise kernels

// out[r, c] = proj[r, c] * gelu(proj[r, inner + c]); vectors never straddle a row.
// Every workgroup but the last takes the branch-free path: 2*U loads in flight
// per lane before the first use.  (Kernel arguments here are plain values, which come in scalar registers; a structure would
// be loaded from memory first, see build.py.  Recorded steps of 512 x 512, us, the division of GEGLU and of the sums, LayerNorm's
// lanes from memory and so: fp16 batch 2 739 -> 727, fp32 batch 1 750 -> 734.)
template <typename T, int U>
__global__ __launch_bounds__(kGegluThreads) void geglu_kernel(const T *__restrict__ proj,
                                                               T *__restrict__ out, uint32_t out_vecs,
                                                               uint32_t row_mul, uint32_t row_shift,
                                                               uint32_t row_vecs) {
    constexpr int EPV = Store<T>::EPV;
    const FastDiv vec_per_row{row_mul, row_shift, row_vecs};
    const u32x4 *in = reinterpret_cast<const u32x4 *>(proj);
    u32x4 *o = reinterpret_cast<u32x4 *>(out);
    const uint32_t block_base = blockIdx.x * (kGegluThreads * U);
    const uint32_t base = block_base + threadIdx.x;
    const bool full = block_base + kGegluThreads * U <= out_vecs;  // uniform
    u32x4 va[U], vb[U];
    uint32_t ovs[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t ov = base + u * kGegluThreads;
        ovs[u] = full ? ov : min(ov, out_vecs - 1);  // ragged last block re-reads the last vector
        const uint32_t r = fast_div(ovs[u], vec_per_row);
        const size_t iv = (size_t)ovs[u] + (size_t)r * vec_per_row.d;  // r*2*vpr + (ov - r*vpr)
        va[u] = load_stream(in + iv);
        vb[u] = load_stream(in + iv + vec_per_row.d);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        float a[EPV], b[EPV], r[EPV];
        Store<T>::unpack(va[u], a);
        Store<T>::unpack(vb[u], b);
#pragma unroll
        for (int e = 0; e < EPV; e++) r[e] = a[e] * gelu_erf_f(b[e]);
        const u32x4 packed = Store<T>::pack(r);
        if (full || base + u * kGegluThreads < out_vecs) store_stream(o + ovs[u], packed);
    }
}

template <typename T>
__global__ __launch_bounds__(kStreamThreads) void geglu_generic_kernel(
    const T *__restrict__ proj, T *__restrict__ out, size_t rows, size_t inner) {
    const size_t n = rows * inner;
    for (size_t i = (size_t)blockIdx.x * kStreamThreads + threadIdx.x; i < n;
         i += (size_t)gridDim.x * kStreamThreads) {
        const size_t r = i / inner, c = i - r * inner;
        const float a = Store<T>::load1(proj + r * 2 * inner + c);
        const float b = Store<T>::load1(proj + r * 2 * inner + inner + c);
        Store<T>::store1(out + i, a * gelu_erf_f(b));
    }
}

// y[i] = OP(x[i]); y may alias x: a lane reads its vectors before it writes them,
// and in the ragged last block the duplicated reads are never written back.
template <typename T, typename OP, int U, int NT>
__global__ __launch_bounds__(NT) void act_kernel(const T *x, T *y, uint32_t vecs, size_t n) {
    constexpr int EPV = Store<T>::EPV;
    const u32x4 *in = reinterpret_cast<const u32x4 *>(x);
    u32x4 *o = reinterpret_cast<u32x4 *>(y);
    const uint32_t block_base = blockIdx.x * (NT * U);
    const uint32_t base = block_base + threadIdx.x;
    const bool full = block_base + NT * U <= vecs;  // uniform
    if (vecs != 0) {
        u32x4 raw[U];
        uint32_t vs[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t v = base + u * NT;
            vs[u] = full ? v : min(v, vecs - 1);
            raw[u] = load_stream(in + vs[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            float f[EPV];
            Store<T>::unpack(raw[u], f);
#pragma unroll
            for (int e = 0; e < EPV; e++) f[e] = OP::apply(f[e]);
            const u32x4 packed = Store<T>::pack(f);
            if (full || base + u * NT < vecs) store_stream(o + vs[u], packed);
        }
    }
    // ragged tail (n % EPV elements) by the first lanes of block 0
    const size_t tail = (size_t)vecs * EPV;
    if (blockIdx.x == 0 && tail + threadIdx.x < n)
        Store<T>::store1(y + tail + threadIdx.x,
                         OP::apply(Store<T>::load1(x + tail + threadIdx.x)));
}

template <typename T, typename OP>
__global__ __launch_bounds__(kStreamThreads) void act_generic_kernel(const T *x, T *y, size_t n) {
    for (size_t i = (size_t)blockIdx.x * kStreamThreads + threadIdx.x; i < n;
         i += (size_t)gridDim.x * kStreamThreads)
        Store<T>::store1(y + i, OP::apply(Store<T>::load1(x + i)));
}

// c[i] = a[i] + b[i]  (chunk_vecs == 0), or c[i] = a[i] + b[i / chunk] with one b value per
// chunk of `chunk_vecs` vectors (the per-channel broadcast add).  c may alias a or b.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void add_kernel(const T *a, const T *b, T *c, uint32_t vecs, uint32_t chunk_mul,
                                                  uint32_t chunk_shift, uint32_t chunk_size) {
    constexpr int EPV = Store<T>::EPV;
    const FastDiv chunk_vecs{chunk_mul, chunk_shift, chunk_size};
    const uint32_t v = blockIdx.x * NT + threadIdx.x;
    if (v >= vecs) return;
    float fa[EPV], fb[EPV];
    Store<T>::unpack(load_stream(reinterpret_cast<const u32x4 *>(a) + v), fa);
    if (chunk_vecs.d == 0) {
        Store<T>::unpack(load_stream(reinterpret_cast<const u32x4 *>(b) + v), fb);
#pragma unroll
        for (int e = 0; e < EPV; e++) fa[e] += fb[e];
    } else {
        const float bv = Store<T>::load1(b + fast_div(v, chunk_vecs));
#pragma unroll
        for (int e = 0; e < EPV; e++) fa[e] += bv;
    }
    store_stream(reinterpret_cast<u32x4 *>(c) + v, Store<T>::pack(fa));
}

template <typename T>
__global__ __launch_bounds__(kStreamThreads) void add_generic_kernel(const T *a, const T *b, T *c,
                                                                     size_t n, size_t chunk_size) {
    for (size_t i = (size_t)blockIdx.x * kStreamThreads + threadIdx.x; i < n;
         i += (size_t)gridDim.x * kStreamThreads) {
        const float bv = Store<T>::load1(b + (chunk_size ? i / chunk_size : i));
        Store<T>::store1(c + i, Store<T>::load1(a + i) + bv);
    }
}

// ---------------------------------------------------------------------------
// [i, j, k] -> [i, k, j], a workgroup per 64 x 64-element tile (tile_transpose.h).
// ES = bytes per element; JFAST: consecutive workgroups take consecutive tiles of one output row.
// RAGGED: sizes that are no whole number of 16-byte pieces, or planes that are not 16-byte aligned
// (the tokens of a 9 x 7 latent); unaligned 16-byte accesses, only the pieces that a row's end cuts go
// in parts.  Against element-wise and 4-element accesses, us: fp16 32 x 63 x 1280 9.36 -> 3.37, 2 x 252 x
// 1280 2.58 -> 2.24, fp32 3 x 99 x 1280 4.56 -> 3.14; a copy of the first takes about 3.4.
// ---------------------------------------------------------------------------
template <int ES, bool JFAST, bool RAGGED>
__global__ __launch_bounds__(kTileThreads) void permute_021_words_kernel(const void *__restrict__ src,
                                                                         void *__restrict__ dst, uint32_t jsize,
                                                                         uint32_t ksize) {
    __shared__ u32x4 tile4[tile_lds_words<ES>()];
    const uint32_t k0 = (JFAST ? blockIdx.y : blockIdx.x) * kTile, j0 = (JFAST ? blockIdx.x : blockIdx.y) * kTile;
    const size_t plane = (size_t)blockIdx.z * jsize * ksize * ES;
    transpose_tile<ES, RAGGED>(static_cast<const char *>(src) + plane, static_cast<char *>(dst) + plane, jsize, ksize, j0,
                               k0, tile4, [] {}, [](uint32_t, const u32x4 &v) { return v; });
}

template <typename T>
__global__ __launch_bounds__(kStreamThreads) void permute_021_generic_kernel(
    const T *__restrict__ src, T *__restrict__ dst, size_t isize, size_t jsize, size_t ksize) {
    const size_t n = isize * jsize * ksize;
    for (size_t d = (size_t)blockIdx.x * kStreamThreads + threadIdx.x; d < n;
         d += (size_t)gridDim.x * kStreamThreads) {
        const size_t j = d % jsize, k = (d / jsize) % ksize, i = d / (jsize * ksize);
        dst[d] = src[(i * jsize + j) * ksize + k];
    }
}

// ---------------------------------------------------------------------------
// Timestep embedding
// ---------------------------------------------------------------------------
// freq_i is the float32 expression exp(neg_log_period * float(i) / float(half))
// with one rounding per operation; exp is evaluated in double and rounded once,
// which reproduces a correctly rounded float exp.  The angle float(t)*freq is a
// single float32 product; cos / sin are evaluated in double and rounded once.
template <typename T>
__global__ __launch_bounds__(256) void timestep_embedding_kernel(
    const int64_t *__restrict__ timesteps, T *__restrict__ out, uint32_t batch, uint32_t half,
    float neg_log_period) {
    const uint32_t idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= batch * half) return;
    const uint32_t b = idx / half, i = idx - b * half;
    const float z = __fdiv_rn(__fmul_rn(neg_log_period, (float)i), (float)half);
    const float freq = (float)exp((double)z);
    const float arg = __fmul_rn((float)timesteps[b], freq);
    double sn, cs;
    sincos((double)arg, &sn, &cs);
    T *row = out + (size_t)b * (2 * half);
    Store<T>::store1(row + i, (float)cs);
    Store<T>::store1(row + half + i, (float)sn);
}

// ---- streaming dispatch ----------------------------------------------------
}  // namespace

template <typename T>
int geglu_dispatch(const void *pv, void *ov, size_t rows, size_t inner, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const T *proj = static_cast<const T *>(pv);
    T *out = static_cast<T *>(ov);
    if (rows == 0 || inner == 0) return MSD_OK;
    const size_t out_vecs = rows * (inner / EPV);
    if (aligned16(proj) && aligned16(out) && inner % EPV == 0 && out_vecs < 0x7FFFFFFFull &&
        rows < 0x7FFFFFFFull) {
        const FastDiv fd = make_fast_div((uint32_t)(inner / EPV));
        // one vector per lane: these launches are short enough that a lane's dependent ALU chain
        // is on the critical path, and more, lighter wavefronts overlap it with other loads
        // (measured 9 - 30 % faster than 4 vectors per lane at every UNet shape)
        const int tune_vectors = g_tuning.geglu_vectors.load(std::memory_order_relaxed);
        const int unroll = tune_vectors ? tune_vectors : 1;
        const uint32_t ov = (uint32_t)out_vecs;
        auto blocks = [&](int u) { return (uint32_t)((out_vecs + kGegluThreads * u - 1) / (kGegluThreads * u)); };
        if (unroll == 1)
            launch((geglu_kernel<T, 1>), dim3(blocks(1)), dim3(kGegluThreads), 0, stream, proj, out, ov, fd.mul, fd.shift, fd.d);
        else if (unroll == 2)
            launch((geglu_kernel<T, 2>), dim3(blocks(2)), dim3(kGegluThreads), 0, stream, proj, out, ov, fd.mul, fd.shift, fd.d);
        else
            launch((geglu_kernel<T, 4>), dim3(blocks(4)), dim3(kGegluThreads), 0, stream, proj, out, ov, fd.mul, fd.shift, fd.d);
    } else {
        const size_t n = rows * inner;
        const size_t want = (n + kStreamThreads - 1) / kStreamThreads;
        launch((geglu_generic_kernel<T>), dim3((uint32_t)(want < 65536 ? want : 65536)),
                           dim3(kStreamThreads), 0, stream, proj, out, rows, inner);
    }
    return launch_status();
}

namespace {

template <typename T, typename OP, int NT>
void act_vectors_launch(int unroll, const T *x, T *y, uint32_t vecs, size_t n, hipStream_t stream) {
    const size_t per_block = (size_t)NT * unroll;
    const dim3 blocks(vecs ? (uint32_t)((vecs + per_block - 1) / per_block) : 1u);
    if (unroll == 4) launch((act_kernel<T, OP, 4, NT>), blocks, dim3(NT), 0, stream, x, y, vecs, n);
    else if (unroll == 2) launch((act_kernel<T, OP, 2, NT>), blocks, dim3(NT), 0, stream, x, y, vecs, n);
    else launch((act_kernel<T, OP, 1, NT>), blocks, dim3(NT), 0, stream, x, y, vecs, n);
}

template <typename T, typename OP>
int act_launch(const void *xv, void *yv, size_t n, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const T *x = static_cast<const T *>(xv);
    T *y = static_cast<T *>(yv);
    if (n == 0) return MSD_OK;
    const size_t vecs = n / EPV;
    if (aligned16(x) && aligned16(y) && vecs < 0x7FFFFFFFull) {
        const int tune_vectors = g_tuning.act_vectors.load(std::memory_order_relaxed);
        const int unroll = tune_vectors ? tune_vectors : kStreamUnroll;
        if (stream_lanes(vecs, false) == kWave) act_vectors_launch<T, OP, kWave>(unroll, x, y, (uint32_t)vecs, n, stream);
        else act_vectors_launch<T, OP, kStreamThreads>(unroll, x, y, (uint32_t)vecs, n, stream);
    } else {
        const size_t want = (n + kStreamThreads - 1) / kStreamThreads;
        launch((act_generic_kernel<T, OP>),
                           dim3((uint32_t)(want < 65536 ? want : 65536)), dim3(kStreamThreads), 0,
                           stream, x, y, n);
    }
    return launch_status();
}


}  // namespace

template <typename T>
int add_dispatch(const void *av, const void *bv, void *cv, size_t n, size_t chunk_size,
                 hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const T *a = static_cast<const T *>(av);
    const T *b = static_cast<const T *>(bv);
    T *c = static_cast<T *>(cv);
    if (n == 0) return MSD_OK;
    const bool vec_ok = aligned16(a) && aligned16(c) && n % EPV == 0 && n / EPV < 0x7FFFFFFFull &&
                        (chunk_size == 0 ? aligned16(b) : chunk_size % EPV == 0);
    if (vec_ok) {
        const uint32_t vecs = (uint32_t)(n / EPV);
        FastDiv fd = make_fast_div((uint32_t)(chunk_size / EPV));
        if (chunk_size == 0) fd.d = 0;
        const uint32_t lanes = stream_lanes(vecs, chunk_size == 0);
        auto *kernel = lanes == kWave ? add_kernel<T, kWave> : add_kernel<T, kStreamThreads>;
        launch(kernel, dim3((vecs + lanes - 1) / lanes), dim3(lanes), 0, stream, a, b, c, vecs, fd.mul, fd.shift, fd.d);
    } else {
        const size_t want = (n + kStreamThreads - 1) / kStreamThreads;
        launch((add_generic_kernel<T>), dim3((uint32_t)(want < 65536 ? want : 65536)),
                           dim3(kStreamThreads), 0, stream, a, b, c, n, chunk_size);
    }
    return launch_status();
}

template <typename TT>
int permute_021_dispatch(const void *srcv, void *dstv, size_t isize, size_t jsize, size_t ksize,
                         hipStream_t stream) {
    // pure data movement: elements are handled as raw 16- or 32-bit words
    typedef typename std::conditional<sizeof(TT) == 2, uint16_t, uint32_t>::type T;
    const T *src = static_cast<const T *>(srcv);
    T *dst = static_cast<T *>(dstv);
    if (isize * jsize * ksize == 0) return MSD_OK;
    const size_t epv = 16 / sizeof(T);
    const bool ragged = jsize % epv != 0 || ksize % epv != 0 || !aligned16(src) || !aligned16(dst);
    const dim3 tiles((uint32_t)((ksize + kTile - 1) / kTile), (uint32_t)((jsize + kTile - 1) / kTile), (uint32_t)isize);
    // Ragged, a tile costs its workgroup, its barrier and a chain of loads for each cut piece, however little of it
    // lies in the tensor: planes and rows that fill few of its 4096 elements, and small tensors, move faster element
    // by element.  us, tile against elements (elements per tile):
    //   fp16  65535 x 2 x 2 (4) 30.5 / 3.0    1778 x 3 x 300 (180) 8.2 / 6.7    6275 x 17 x 15 (255) 8.8 / 6.7
    //   fp32  5000 x 5 x 64 (320) 7.8 / 7.2   714 x 7 x 320 (448) 7.6 / 7.2, transposed 6.5 / 9.2   15 x 77 x 77 3.07 / 2.67
    // (by elements per tile, 256 Ki and more in all, tile against elements: fp16 128 - 200 1.2, 200 - 300 0.96, 350 - 400
    // 0.82; fp32 input rows longer than output rows 300 - 400 1.15, 400 - 450 1.03, 450 - 600 0.88, shorter 250 - 300
    // 1.13, 300 - 350 1.03, 350 - 400 0.92; by elements in all, 1500 and more per tile: fp16 140 - 180 Ki 0.98, 180 - 256 Ki
    // 0.90, fp32 180 - 220 Ki 1.02, 220 - 256 Ki 0.94.)  In pieces that nothing cuts, or only in halves (2-byte sides in multiples of
    // four), the tile is within 5 % of the better one or ahead at every size.
    const size_t n = isize * jsize * ksize;
    const size_t per_tile = jsize * ksize / (((jsize + kTile - 1) / kTile) * ((ksize + kTile - 1) / kTile));
    const bool halves = ragged && sizeof(T) == 2 && (jsize | ksize) % 4 == 0 &&
                        ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 7u) == 0;
    const size_t least = sizeof(T) == 2 ? 250 : jsize > ksize ? 350 : 450, least_in_all = (sizeof(T) == 2 ? 192 : 256) * 1024;
    const bool tile_pays = !ragged || halves || (per_tile >= least && n >= least_in_all);
    const bool tiled = tile_pays && isize <= 65535 && ksize <= kTileMaxSide && jsize <= kTileMaxSide &&
                       (tiles.x <= 65535 || tiles.y <= 65535);
    // Output rows shorter than input rows: consecutive workgroups take the tiles of one output
    // row, so that its 128-byte pieces are written at about the same time (batch 32, 320 x 4096
    // -> 4096 x 320, fp16: 29.9 us against 32.1 with consecutive tiles along the input rows; the
    // copy takes 29.1; the other way round nothing changes; in halves it costs up to 15 %, 695 x 368 x 452 fp16
    // 136 against 117, and gains 2 % at most).
    const bool jfast = (jsize < ksize && !halves && tiles.x <= 65535) || tiles.y > 65535;
    if (tiled) {
        constexpr int ES = (int)sizeof(T);
        auto *kernel = jfast ? (ragged ? permute_021_words_kernel<ES, true, true> : permute_021_words_kernel<ES, true, false>)
                             : (ragged ? permute_021_words_kernel<ES, false, true> : permute_021_words_kernel<ES, false, false>);
        launch(kernel, jfast ? dim3(tiles.y, tiles.x, tiles.z) : tiles, dim3(kTileThreads), 0, stream, srcv, dstv,
               (uint32_t)jsize, (uint32_t)ksize);
    } else {
        const size_t want = (n + kStreamThreads - 1) / kStreamThreads;
        launch((permute_021_generic_kernel<T>), dim3((uint32_t)(want < 65536 ? want : 65536)),
                           dim3(kStreamThreads), 0, stream, src, dst, isize, jsize, ksize);
    }
    return launch_status();
}

template <typename T>
int act_dispatch(Act op, const void *x, void *y, size_t n, hipStream_t stream) {
    switch (op) {
        case Act::Silu: return act_launch<T, OpSilu>(x, y, n, stream);
        case Act::Gelu: return act_launch<T, OpGelu>(x, y, n, stream);
        case Act::QuickGelu: return act_launch<T, OpQuickGelu>(x, y, n, stream);
        case Act::Copy: return act_launch<T, OpCopy>(x, y, n, stream);
    }
    return MSD_ERR_INVALID_VALUE;
}

template <typename T>
int temb_dispatch(const int64_t *timesteps, void *out, size_t batch, size_t dim, float max_period,
                  hipStream_t stream) {
    const uint32_t half = (uint32_t)(dim / 2);
    const uint32_t blocks = (uint32_t)((batch * half + 255) / 256);
    const float neg_log_period = -logf(max_period);  // host float log, as in the replaced host loop
    launch((timestep_embedding_kernel<T>), dim3(blocks), dim3(256), 0, stream, timesteps,
                       static_cast<T *>(out), (uint32_t)batch, half, neg_log_period);
    return launch_status();
}

template int geglu_dispatch<float>(const void *, void *, size_t, size_t, hipStream_t);
template int geglu_dispatch<__half>(const void *, void *, size_t, size_t, hipStream_t);
template int add_dispatch<float>(const void *, const void *, void *, size_t, size_t, hipStream_t);
template int add_dispatch<__half>(const void *, const void *, void *, size_t, size_t, hipStream_t);
template int permute_021_dispatch<float>(const void *, void *, size_t, size_t, size_t, hipStream_t);
template int permute_021_dispatch<__half>(const void *, void *, size_t, size_t, size_t, hipStream_t);
template int act_dispatch<float>(Act, const void *, void *, size_t, hipStream_t);
template int act_dispatch<__half>(Act, const void *, void *, size_t, hipStream_t);
template int temb_dispatch<float>(const int64_t *, void *, size_t, size_t, float, hipStream_t);
template int temb_dispatch<__half>(const int64_t *, void *, size_t, size_t, float, hipStream_t);

}  // namespace msd
