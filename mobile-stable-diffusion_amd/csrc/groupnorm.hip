// GroupNorm (+ SiLU) for gfx950.
//
// A unit is one (sample, group): ch_per_group * hw contiguous elements of an
// NCHW tensor.  A unit is cut into `split` slices, one workgroup per slice; the
// slice stays in registers as packed 16-byte vectors for the whole kernel, so
// the tensor is read from HBM once and written once.
//
//   1. every lane issues all its loads (K vectors) before the first use;
//   2. slice mean and M2 = sum (x - slice mean)^2 from one pass of sum and sum of squares
//      over the packed registers (DPP wavefront reduction, one LDS slot per wavefront), with
//      a second, centred pass when the mean is large against the spread;
//   3. split > 1: slices publish (mean, M2) as two tagged 64-bit words, poll
//      their siblings' words, and merge with Chan's formula.  The tag comes from
//      a count per unit that every slice advances by its share, so nothing is
//      reset between launches and a replayed graph works.  All traffic is
//      relaxed agent-scope atomics: no cache flushes.
//   4. y = fma(x - mean, rstd * gamma[c], beta[c]) (the mean folded into the offset when it
//      is small), optional SiLU, packed store.
//
// When the output lies apart from the input and the launch is small, whole units are instead
// shared by several workgroups (SHARED): each loads and reduces the whole unit (steps 1 and 2,
// the same bits in every one; the copies of the loads meet in the L2 of the XCD the writers are
// placed on) and does step 4 for its own part of the unit.  No step 3, nothing waits.
//
// Workgroups of one unit have adjacent block ids, so a waiter's siblings are
// normally dispatched together with it.  Nothing depends on that: every wait is
// bounded (about a millisecond of polls), and a slice whose sibling has not
// published by then computes that sibling's statistics itself from the
// sibling's part of the input, which no workgroup overwrites before it has
// seen every word of its unit.  The output is the same either way; a counter
// in the scratch records how often it happened.
#include <algorithm>
#include <type_traits>

#include "msd_device.h"
#include "msd_internal.h"
#include "tile_transpose.h"

namespace msd {

namespace {

constexpr uint32_t kGnSpinLimit = 2048;  // default poll limit: about half a microsecond per poll
// Polls that a slice waits for its own words, however short the limit for its siblings' is: some 30 ms, far more than its stores
// take.  Only another launch that overlaps this one on the same scratch, against the rules, can write over them before they are
// read; the slice then gives up on them as on a sibling's, and the kernel ends.
constexpr uint32_t kGnOwnSpinLimit = 65536;
constexpr int kGenericThreads = 256;
constexpr int kGnRedRow = 16;                // partial sums of a workgroup, one per wavefront: a row of lanes
constexpr int kGnRedSlots = 3 * kGnRedRow;   // sums, sums of squares, sums about the mean
static_assert(kGnMaxThreads / kWave <= kGnRedRow, "a row of lanes holds the wavefronts' partial sums");

// (No field that no kernel reads: what is loaded with its neighbours and not used costs a wait, for its register.)
struct GnParams {
    uint32_t vec_per_unit;   // 16-byte vectors per unit
    uint32_t vec_per_slice;  // vectors per workgroup (the last slice may be shorter)
    uint32_t split;          // workgroups per unit, power of two <= kGnMaxSplit
    uint32_t spin_limit;     // polls before a slice stops waiting for a sibling's words
    FastDiv groups;          // per sample
    float eps;
    float inv_count;         // 1 / elements per unit
    // gn_slice_kernel<..., SHARED>: several workgroups per whole unit; each loads and reduces the
    // whole unit and normalises and stores one part of it
    uint32_t part_vecs;      // vectors per part, a multiple of 64 (a wavefront is inside one part or outside)
    uint32_t hw;             // RAGGED: elements per channel
};

// The arguments that a wavefront needs before it can ask for its data are the kernels' first ones, plain values that arrive
// in scalar registers (build.py); the rest, loaded from memory, is needed when the data is on its way.  One word holds the
// logarithms of the launch's shape and its lanes.  us, structures and so: recorded steps of 512 x 512 fp16 batch 2 752 -> 739, fp32
// batch 1 762 -> 750; per launch, fp16 batch 2, in place, 640 channels at 32 x 32 4.55 -> 4.45, 1280 at 16 x 16 3.37 -> 3.22, token
// norm of those 3.29 -> 3.02 (an argument from memory in a step: 620 cycles).
// xcd_shift: the writers of a unit have block ids (1 << xcd_shift) apart: with that many XCDs they share one XCD and its L2
// (units in whole rows of that many); 0: adjacent ids.
inline uint32_t gn_shape_word(uint32_t split_shift, uint32_t writers_shift, uint32_t xcd_shift,
                                                  uint32_t threads) {
    return split_shift | writers_shift << 4 | xcd_shift << 8 | threads << 16;
}
struct GnShape {
    uint32_t split_shift, writers_shift, xcd_shift, threads;
    __device__ __forceinline__ explicit GnShape(uint32_t word)
        : split_shift(word & 15u), writers_shift(word >> 4 & 15u), xcd_shift(word >> 8 & 255u), threads(word >> 16) {}
};

// Sum over the workgroup (blockDim.x / 64 wavefronts); one barrier.
__device__ __forceinline__ float block_sum_rt(float v, float *slots) {
    const float w = wave_sum(v);
    const uint32_t nw = blockDim.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) slots[threadIdx.x / kWave] = w;
    __syncthreads();
    float t = 0.0f;
    for (uint32_t i = 0; i < nw; i++) t += slots[i];
    return t;
}

__device__ __forceinline__ unsigned long long tagged(uint32_t tag, float v) {
    return ((unsigned long long)tag << 32) | (unsigned long long)__float_as_uint(v);
}

// What a launch's tag on a unit comes from, the same for all its slices: by one lane at kernel start each slice adds its share of
// kGnMaxSplit to the unit's count, and what it finds there, divided by kGnMaxSplit, is the number of launches before.  The shares
// of a launch sum to exactly kGnMaxSplit, whatever its split, and a slice that has not added its own finds less than that on top,
// however late it starts; nothing is left to do at the end.  After launches that overlapped on one scratch, which the rules
// forbid, the count is a multiple of kGnMaxSplit again and no tag that they left in the slots is above its launches: those
// that follow in order are not affected.
// (The index is a vector register to the compiler, which otherwise adds for all lanes at once and waits for the answer on the spot;
// and the answer stays whole until the statistics are there: with one half of it unused the next loads waited for its register.)
// us per launch, in place, a launch count that the last slice to finish advances / a tag per slice kept in its own slot, which
// an overlap could set apart for good / so: fp16 320 channels at 64 x 64 batch 2 5.97 / 4.91 / 4.92, 640 7.12 / 6.37 / 6.35, fp32 320
// batch 1 5.83 / 5.01 / 5.02, 960 batch 2 11.72 / 10.79 / 10.82; sixteen units' counts in a line: fp16 960 batch 1 5.70 -> 6.25.
__device__ __forceinline__ unsigned long long gn_exchange_enter(const GnExchange &scratch, uint32_t split, uint32_t unit) {
    uint32_t index = unit * kGnCountStride;
    asm volatile("" : "+v"(index));
    const unsigned long long share = kGnMaxSplit >> __builtin_ctz(split);
    return __hip_atomic_fetch_add(scratch.counts + index, share, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Merges the slices of one unit.  Called by every lane of the workgroup with the slice's
// (mean, M2); `count` is what lane 0 got from gn_exchange_enter at kernel start.  On return
// stats[0] = mean and stats[1] = 1/sqrt(var + eps) of the whole unit, in LDS, after a barrier.
// Slice l covers vectors [l * vec_per_slice, min(vec_per_unit, (l + 1) * vec_per_slice)).
// `read(l, i)` returns vector i of slice l as the statistics see it (after the optional addend);
// it is only used when slice l has not published within the poll limit.
template <typename T, typename Params, typename Reader>
__device__ __forceinline__ void gn_exchange(const GnExchange &scratch, const Params &p, uint32_t unit,
                                            uint32_t slice, unsigned long long count, float slice_mean,
                                            float slice_m2, float *stats, Reader read) {
    constexpr int EPV = Store<T>::EPV;
    const uint32_t tid = threadIdx.x;
    unsigned long long *slot_mean = scratch.slot_mean + (size_t)unit * kGnMaxSplit;
    unsigned long long *slot_m2 = scratch.slot_m2 + (size_t)unit * kGnMaxSplit;
    if (tid < kWave) {  // wavefront 0 owns the exchange; lane 0 holds the count
        const uint32_t tag = (uint32_t)__builtin_amdgcn_readfirstlane((int)(count / kGnMaxSplit)) + 1u;
        if (tid == 0) {
            __hip_atomic_store(slot_mean + slice, tagged(tag, slice_mean), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(slot_m2 + slice, tagged(tag, slice_m2), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        // lane l waits for slice l
        float m_l = 0.0f, q_l = 0.0f, n_l = 0.0f;
        bool ok = true;
        if (tid < p.split) {
            unsigned long long wm, wq;
            uint32_t polls = 0;
            // A slice does not give up on its own words: they arrive without anybody's help, and
            // having read them back is what lets it store output (see below).
            const uint32_t limit = tid == slice ? max(kGnOwnSpinLimit, p.spin_limit) : p.spin_limit;
            do {
                wm = __hip_atomic_load(slot_mean + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                wq = __hip_atomic_load(slot_m2 + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = (uint32_t)(wm >> 32) == tag && (uint32_t)(wq >> 32) == tag;
                if (!ok) __builtin_amdgcn_s_sleep(1);
            } while (!ok && ++polls < limit);
            m_l = __uint_as_float((uint32_t)wm);
            q_l = __uint_as_float((uint32_t)wq);
            const uint32_t b = tid * p.vec_per_slice;
            const uint32_t e = min(p.vec_per_unit, b + p.vec_per_slice);
            n_l = (float)((e - b) * EPV);
        }
        // Slices that have not published (not dispatched yet, or starved): this wavefront
        // computes their (mean, M2) from their part of the input, two passes.  A slice stores
        // output only after it has read back every word of its unit from the memory side, its
        // own included, so what is read here is still input unless the sibling published in the
        // meantime - then its words are at the memory side before its first output store
        // leaves, and they win when they are read again after the passes.  That second read
        // must not start before the passes' loads have returned: the wait below stops the
        // memory pipeline, and as a compiler barrier the compiler, from moving it ahead.
        unsigned long long missing = __builtin_amdgcn_ballot_w64(!ok);
        if (missing != 0) {  // uniform over the wavefront
            while (missing != 0) {
                const uint32_t s = (uint32_t)__builtin_ctzll(missing);
                missing &= missing - 1;
                const uint32_t b = s * p.vec_per_slice;
                const uint32_t n = min(p.vec_per_unit, b + p.vec_per_slice) - b;
                float sum = 0.0f;
                for (uint32_t i = tid; i < n; i += kWave) {
                    float f[EPV];
                    Store<T>::unpack(read(s, i), f);
#pragma unroll
                    for (int e = 0; e < EPV; e++) sum += f[e];
                }
                const float mean_s = wave_sum(sum) / (float)(n * EPV);
                float q = 0.0f;
                for (uint32_t i = tid; i < n; i += kWave) {
                    float f[EPV];
                    Store<T>::unpack(read(s, i), f);
#pragma unroll
                    for (int e = 0; e < EPV; e++) {
                        const float d = f[e] - mean_s;
                        q = fmaf(d, d, q);
                    }
                }
                const float m2_s = wave_sum(q);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (tid == s) {
                    const unsigned long long wm =
                        __hip_atomic_load(slot_mean + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const unsigned long long wq =
                        __hip_atomic_load(slot_m2 + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const bool late = (uint32_t)(wm >> 32) == tag && (uint32_t)(wq >> 32) == tag;
                    m_l = late ? __uint_as_float((uint32_t)wm) : mean_s;
                    q_l = late ? __uint_as_float((uint32_t)wq) : m2_s;
                }
            }
            if (tid == 0)
                __hip_atomic_fetch_add(scratch.fallbacks, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // Chan: mean = sum n_l mean_l / n ; M2 = sum M2_l + sum n_l (mean_l - mean)^2
        const float total_mean = wave_sum(m_l * n_l) * p.inv_count;
        const float dm = m_l - total_mean;
        const float m2 = wave_sum(fmaf(n_l * dm, dm, q_l));
        if (tid == 0) {
            stats[0] = total_mean;
            stats[1] = __builtin_amdgcn_rsqf(m2 * p.inv_count + p.eps);
        }
    }
    __syncthreads();
}

// Sum and sum of squares of a packed vector, accumulated in float32.  Half storage uses
// v_dot2_f32_f16 (both products of a register pair are exact in float32 and are added to a
// float32 accumulator; subnormal halves count), so the statistics never need an unpacked copy
// of the slice.  Two accumulator pairs (even / odd registers) halve the dependent chains.
template <typename T>
struct Moments;
template <>
struct Moments<float> {
    static __device__ __forceinline__ void add(const u32x4 &v, float (&s)[2], float (&q)[2]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float f = __uint_as_float(v[i]);
            s[i & 1] += f;
            q[i & 1] = fmaf(f, f, q[i & 1]);
        }
    }
};
template <>
struct Moments<__half> {
    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ void add(const u32x4 &v, float (&s)[2], float (&q)[2]) {
        const half2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t w = v[i];
            const half2_t h = *reinterpret_cast<const half2_t *>(&w);
            s[i & 1] = __builtin_amdgcn_fdot2(h, ones, s[i & 1], false);
            q[i & 1] = __builtin_amdgcn_fdot2(h, h, q[i & 1], false);
        }
    }
};

// |mean| <= 2 sigma: the slice's M2 may be taken from the raw moments (relative error
// below 1e-6); otherwise it is recomputed about the mean (a second pass over the registers)
constexpr float kGnFastMoments = 4.0f;
// |mean| <= 4 sigma of the whole unit: the epilogue may fold the mean into the offset
constexpr float kGnFoldMean = 16.0f;

// Mean and M2 = sum (x - mean)^2 of the workgroup's slice, held as K packed vectors per lane
// (vector k of lane t is element k * nt + t of the slice, nt the workgroup's lanes; the first n_valid count, the
// registers of the others hold zeros).  One pass gives sum and sum of squares (wavefront
// reduction by DPP, the wavefronts' partial sums meet once in LDS, every wavefront adds them
// in the same order).  M2 = sum x^2 - n mean^2 is kept when it is well conditioned; when the
// mean is large against the spread (or the slice is constant) a second pass over the registers
// sums (x - mean)^2 instead, so the result is as accurate as a two-pass variance either way.
// The choice is the same in every wavefront: they all hold bit-identical sums.
// Between the last load's return and the first store this is the launch's critical path: the two sums
// are reduced together (one value per lane after the first half of the steps), a wavefront's pair takes one LDS access each way,
// the at most 16 partial sums meet in one row of lanes, and the mean is a product with the reciprocal of the count, which
// is there before the loads return, corrected once by the remainder (Markstein's division: the bits of the quotient, but
// for subnormal ones; NaN instead of an infinity where the sum has overflowed, where the output is NaN with either).  us per launch at
// batch 2, six LDS swizzles one after the other and a division, and so: fp16 320 channels at 64 x 64 5.19 -> 4.94, in place 5.93 ->
// 5.76, 640 at 32 x 32 3.92 -> 3.74, in place 4.76 -> 4.59, 1280 at 8 x 8 2.65 -> 2.50; fp32 640 at 32 x 32 in place 5.58 -> 5.29.
template <typename T, int K, bool FULL>
__device__ __forceinline__ void gn_slice_stats(u32x4 (&raw)[K], uint32_t n_valid, uint32_t nt, float *red,
                                               float &slice_mean, float &slice_m2) {
    constexpr int EPV = Store<T>::EPV;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t nw = nt / kWave;
    const float count = (float)(n_valid * EPV);
    float inv = 1.0f / count;
    asm volatile("" : "+v"(inv));  // (computed here, while the loads are in flight)
    float s[2] = {0.0f, 0.0f}, q[2] = {0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < K; k++) Moments<T>::add(raw[k], s, q);
    const float wave_sums = wave_sum_of_two(s[0] + s[1], q[0] + q[1]);
    if (lane % kGnRedRow == 0 && lane < 2 * kGnRedRow) red[lane + tid / kWave] = wave_sums;
    __syncthreads();
    const bool entry = lane % kGnRedRow < nw;
    const float sums = team_sum<kGnRedRow>(entry ? red[lane % (2 * kGnRedRow)] : 0.0f);
    const float sum_x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sums), 0));
    const float sum_xx = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sums), kGnRedRow));
    const float quotient = sum_x * inv;
    slice_mean = fmaf(fmaf(-quotient, count, sum_x), inv, quotient);
    slice_m2 = sum_xx - sum_x * slice_mean;
    // n mean^2 <= kappa M2; false also for a negative or NaN M2
    if (!(sum_x * slice_mean <= kGnFastMoments * slice_m2)) {  // uniform over the workgroup
        float c = 0.0f;
#pragma unroll
        for (int k = 0; k < K; k++) {
            float f[EPV];
            forget(raw[k]);  // unpack here, not once for every later use (the copies would not fit)
            Store<T>::unpack(raw[k], f);
            float ck = 0.0f;
#pragma unroll
            for (int e = 0; e < EPV; e++) {
                const float d = f[e] - slice_mean;
                ck = fmaf(d, d, ck);
            }
            if (!FULL) ck = (k * nt + tid < n_valid) ? ck : 0.0f;
            c += ck;
            // one vector at a time: unpacked copies of the whole slice would not fit the registers
            __builtin_amdgcn_sched_barrier(0);
        }
        const float wave_c = wave_sum(c);
        float *red_c = red + 2 * kGnRedRow;
        if (lane == 0) red_c[tid / kWave] = wave_c;
        __syncthreads();
        slice_m2 = wave_sum(lane < nw ? red_c[lane] : 0.0f);
    }
}

// Where a vector that may cross from one channel into the next (hw not a multiple of a vector, but
// at least one) lies: its first element's channel inside the group, and how many of its elements,
// from the first on, belong to that channel (all of them: EPV or more).
struct GnStraddle {
    uint32_t channel, first;
};
template <int EPV>
__device__ __forceinline__ GnStraddle gn_straddle(uint32_t v, const FastDiv &hw) {
    const uint32_t c = fast_div(v * EPV, hw);
    return GnStraddle{c, (c + 1) * hw.d - v * EPV};
}

// FULL: every lane owns exactly K vectors (no masking anywhere).  RAGGED: hw is not a multiple of a
// vector (deeper UNet levels of images that are not square powers of two: 9 x 7, 18 x 14), so
// a vector may hold the end of one channel and the start of the next; each element then picks one
// of two affine pairs (two selects per element, hidden like the rest of the epilogue).  Such shapes
// used to take the general kernel, whose three passes in single elements are a latency chain.  us
// per launch, before and now: fp16 batch 2, 2560 channels at 9 x 7 10.1 -> 2.9, in place 14.1 -> 3.8;
// 1280 at 18 x 14 17.9 -> 2.9, in place 25.3 -> 4.4; batch 16, 640 at 18 x 14 10.7 -> 4.7; fp32 batch 4,
// 2560 at 11 x 9 15.9 -> 3.4.
template <typename T, int K, bool SILU, bool FULL, bool SHARED, bool RAGGED, bool EARLY>
__device__ __forceinline__ void gn_body(const T *x, const T *chunk, T *y,
                                        const float *__restrict__ gamma,
                                        const float *__restrict__ beta, const GnExchange &scratch,
                                        const GnParams &p, uint32_t nt, uint32_t vec_per_unit, uint32_t unit, uint32_t slice,
                                        uint32_t part, uint32_t v_begin, uint32_t v_end, uint32_t ch_per_group,
                                        const FastDiv &hw_vec, float *red, float *stats, float2 *aff) {
    constexpr int EPV = Store<T>::EPV;
    const uint32_t tid = threadIdx.x;
    const u32x4 *xin = reinterpret_cast<const u32x4 *>(x) + (size_t)unit * vec_per_unit;

    // ---- the slice goes into registers.  Lanes past the end of a ragged slice re-read its
    // last vector (a valid address) and are masked later: no load sits behind a branch.
    u32x4 raw[K];
    // Index of a lane's k-th vector inside the unit, and its address.  Both are recomputed
    // from the lane number wherever they are needed (a few instructions) instead of being kept
    // in registers per vector; `lane_again()` returns the lane number as a value the compiler
    // cannot tie to earlier computations, so it cannot decide otherwise.
    auto lane_again = [&]() {
        uint32_t t = tid;
        asm volatile("" : "+v"(t));
        return t;
    };
    auto vidx = [&](int k, uint32_t t) {
        const uint32_t v = v_begin + k * nt + t;
        return FULL ? v : min(v, v_end - 1);
    };
    auto have = [&](int k, uint32_t t) { return FULL || v_begin + k * nt + t < v_end; };
    // the address: a base that is the same for the whole workgroup (scalar registers) plus a
    // lane offset, which for a full slice is the same for every k
    auto at = [&](auto *base, int k, uint32_t t) {
        using Byte = std::conditional_t<std::is_const<std::remove_pointer_t<decltype(base)>>::value, const char, char>;
        const uint32_t offset = vidx(k, t) * (uint32_t)sizeof(u32x4);  // a unit is smaller than 4 GiB (host)
        return reinterpret_cast<decltype(base)>(reinterpret_cast<Byte *>(base) + offset);
    };
#pragma unroll
    for (int k = 0; k < K; k++) raw[k] = load_stream(at(xin, k, tid));
    // optional per-(sample, channel) addend applied before the statistics (the reference's
    // chunkwise_add pass): the sum replaces the slice in registers, rounded to the storage
    // type exactly as a separate add kernel would have stored it
    struct Addend {
        T first, second;  // of a vector's channel, RAGGED of the two it may hold
    };
    auto addend_of = [&](uint32_t v) {
        const T *cb = chunk + (size_t)unit * ch_per_group;  // the unit's channels
        if (!RAGGED) {
            const T c = cb[fast_div(v, hw_vec)];
            return Addend{c, c};
        }
        const uint32_t c = gn_straddle<EPV>(v, hw_vec).channel;
        return Addend{cb[c], cb[min(c + 1, ch_per_group - 1)]};
    };
    auto plus = [&](const u32x4 &raw_v, uint32_t v, const Addend &addend) {
        const float c0 = Store<T>::load1(&addend.first), c1 = Store<T>::load1(&addend.second);
        const uint32_t first = RAGGED ? gn_straddle<EPV>(v, hw_vec).first : EPV;
        float f[EPV];
        Store<T>::unpack(raw_v, f);
#pragma unroll
        for (int e = 0; e < EPV; e++) f[e] += !RAGGED || (uint32_t)e < first ? c0 : c1;
        return Store<T>::pack(f);
    };
    // Everything is requested before anything is waited for, in the order in which it is needed (loads return in order): data,
    // addends, then gamma and beta (us per launch with addends, fp16 batch 2, one after the other and so: 640 channels at 32 x 32
    // 4.63 -> 4.47, 1280 at 16 x 16 3.51 -> 3.40; recorded step of 512 x 512 727 -> 721).  Six vectors per lane request
    // gamma and beta when the data is there: only launches of several workgroups per CU have that many, and twelve more requests a
    // lane in front of the other wavefronts' data cost them 10 % (us, everything early and so: fp16 640 channels at 600 positions
    // batch 32, no SiLU, 9.70 -> 8.71, fp32 at 300 9.84 -> 8.63, 320 at 9216 batch 3 13.1 -> 12.2, batch 2 8.96 -> 9.16; with the
    // addends late too 960 at 784 batch 12 9.07 -> 9.22).  Long slices request
    // their addends when they have the data: K more registers, and their launches are long enough to hide it (fp32 128
    // channels at 512 x 512, three passes of a decoder block 152.7 us, with everything early 153.5).
    constexpr bool kPrefetchAffine = !RAGGED && K <= kGnPrefetchAffineK, kEarly = kPrefetchAffine && EARLY;
    Addend addend[kPrefetchAffine ? K : 1];
    if (kPrefetchAffine && chunk != nullptr) {  // uniform
#pragma unroll
        for (int k = 0; k < K; k++) addend[kPrefetchAffine ? k : 0] = addend_of(vidx(k, tid));
    }
    // What follows waits for the arguments in memory: the compiler neither moves it up nor, as new values to it, shares it
    // with another branch in front of the loads.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+s"(unit), "+s"(part));
    u32x4 *yout = reinterpret_cast<u32x4 *>(y) + (size_t)unit * vec_per_unit;
    const uint32_t ch0 = (unit - fast_div(unit, p.groups) * p.groups.d) * ch_per_group;
    // per-vector channel affine.  Up to six vectors per lane: fetched into registers up front,
    // while the data is in flight.  More: the group's gamma and beta go to LDS once (they are
    // there after the barrier of the statistics) and the epilogue reads each vector's pair one
    // vector ahead, so a lane's registers hold little besides its packed slice.
    float ga[kPrefetchAffine ? K : 1], be[kPrefetchAffine ? K : 1];
    auto fetch_affine = [&]() {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t c = ch0 + fast_div(vidx(k, tid), hw_vec);
            ga[kPrefetchAffine ? k : 0] = gamma[c];
            be[kPrefetchAffine ? k : 0] = beta[c];
        }
    };
    if (kEarly) {
        fetch_affine();
        __builtin_amdgcn_sched_barrier(0);
    }
    // The count is asked for behind what is waited for first.  Up to five vectors a lane that is everything (recorded step of
    // 512 x 512, fp32, in front of gamma and beta / so: 728 / 726 us).  Slices of twelve and more put gamma and beta into LDS in front of
    // the sums and would wait for the count with them; they ask for it after that, and their sums take long enough for it to
    // arrive (us, in front / so: fp32 128 channels at 512 x 512, 16 vectors, 45.35 / 45.13, fp16 22.61 / 22.41; those of ten would
    // lose: fp32 320 at 64 x 64 batch 8 13.5 / 13.9).
    constexpr bool kLong = K >= 12;
    unsigned long long count = 0;
    if (!kLong && !SHARED && p.split > 1 && tid == 0) count = gn_exchange_enter(scratch, p.split, unit);
    if (chunk != nullptr) {  // uniform
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t v = vidx(k, tid);
            raw[k] = plus(raw[k], v, kPrefetchAffine ? addend[kPrefetchAffine ? k : 0] : addend_of(v));
        }
    }
    if (!FULL) {  // registers of lanes past the end of a ragged slice hold zeros from here on
#pragma unroll
        for (int k = 0; k < K; k++) {
            const bool mine = have(k, tid);
#pragma unroll
            for (int i = 0; i < 4; i++) raw[k][i] = mine ? raw[k][i] : 0u;
        }
    }
    if (kPrefetchAffine && !kEarly) fetch_affine();
    if (!kPrefetchAffine) {
        for (uint32_t c = tid; c < ch_per_group; c += nt) {  // ch_per_group <= kGnLdsChannels (host)
            aff[c] = make_float2(gamma[ch0 + c], beta[ch0 + c]);
        }
    }

    if (kLong && !SHARED && p.split > 1 && tid == 0) count = gn_exchange_enter(scratch, p.split, unit);

    float slice_mean, slice_m2;
    gn_slice_stats<T, K, FULL>(raw, v_end - v_begin, nt, red, slice_mean, slice_m2);

    float mean, rstd;
    if (SHARED || p.split == 1) {
        mean = slice_mean;
        rstd = __builtin_amdgcn_rsqf(slice_m2 * p.inv_count + p.eps);
    } else {
        // vector i of slice l as the statistics see it (input plus the optional addend)
        auto read = [&](uint32_t l, uint32_t i) {
            const uint32_t v = l * p.vec_per_slice + i;
            u32x4 r = xin[v];
            if (chunk != nullptr) r = plus(r, v, addend_of(v));
            return r;
        };
        gn_exchange<T>(scratch, p, unit, slice, count, slice_mean, slice_m2, stats, read);
        mean = stats[0];
        rstd = stats[1];
    }

    // ---- normalise from registers, per-channel affine, optional SiLU.  When the unit's mean is
    // within four standard deviations of zero it is folded into the offset,
    // y = fma(x, a, beta - mean a) (one operation per element, error a few 1e-7 at most);
    // otherwise y = fma(x - mean, a, beta), which stays exact for |mean| >> sigma.
    auto epilogue = [&](auto fold_tag) {
        constexpr bool kFold = decltype(fold_tag)::value;
        float g_next = 0.0f, b_next = 0.0f;
        if (!kPrefetchAffine && !RAGGED) {
            const uint32_t c = fast_div(vidx(0, lane_again()), hw_vec);
            const float2 gb = aff[c];  // one 8-byte LDS read
            g_next = gb.x;
            b_next = gb.y;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            float g_k, b_k;
            if (RAGGED) {
                g_k = b_k = 0.0f;  // (two pairs per vector, read below)
            } else if (kPrefetchAffine) {
                g_k = ga[kPrefetchAffine ? k : 0];
                b_k = be[kPrefetchAffine ? k : 0];
            } else {
                g_k = g_next;
                b_k = b_next;
                if (k + 1 < K) {  // the next vector's pair: its LDS latency passes under this vector's work
                    const uint32_t c = fast_div(vidx(k + 1, lane_again()), hw_vec);
                    const float2 gb = aff[c];
                    g_next = gb.x;
                    b_next = gb.y;
                }
            }
            // several writers per unit: this one normalises and stores the vectors of its part
            // only; a wavefront is inside a part or outside it as a whole
            if (SHARED) {  // (decided per wavefront: a scalar branch)
                const uint32_t first = __builtin_amdgcn_readfirstlane(vidx(k, lane_again()));
                if (first - part * p.part_vecs >= p.part_vecs) continue;
            }
            float f[EPV];
            if (RAGGED) {
                const GnStraddle at_v = gn_straddle<EPV>(vidx(k, lane_again()), hw_vec);
                const float2 gb0 = aff[at_v.channel];
                const float2 gb1 = aff[min(at_v.channel + 1, ch_per_group - 1)];
                const float a0 = rstd * gb0.x, a1 = rstd * gb1.x;
                const float b0 = kFold ? fmaf(-mean, a0, gb0.y) : gb0.y, b1 = kFold ? fmaf(-mean, a1, gb1.y) : gb1.y;
                forget(raw[k]);  // unpack here, one vector at a time
                Store<T>::unpack(raw[k], f);
#pragma unroll
                for (int e = 0; e < EPV; e++) {
                    const bool in0 = (uint32_t)e < at_v.first;
                    const float t = fmaf(kFold ? f[e] : f[e] - mean, in0 ? a0 : a1, in0 ? b0 : b1);
                    f[e] = SILU ? silu_f(t) : t;
                }
            } else {
                const float a = rstd * g_k;
                const float b_fold = fmaf(-mean, a, b_k);
                forget(raw[k]);  // unpack here, one vector at a time
                Store<T>::unpack(raw[k], f);
#pragma unroll
                for (int e = 0; e < EPV; e++) {
                    const float t = kFold ? fmaf(f[e], a, b_fold) : fmaf(f[e] - mean, a, b_k);
                    f[e] = SILU ? silu_f(t) : t;
                }
            }
            const u32x4 packed = Store<T>::pack(f);
            const uint32_t t = lane_again();
            if (have(k, t)) store_stream(at(yout, k, t), packed);
            // the scheduler must not start unpacking the next vectors before this one is stored:
            // eight elements are enough independent work, and the slice stays packed until used
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (mean * mean * (rstd * rstd) <= kGnFoldMean)  // uniform over the workgroup
        epilogue(std::true_type{});
    else
        epilogue(std::false_type{});
}

// Up to six vectors per lane (four for float storage) the kernel fits 64 registers: eight
// wavefronts per SIMD, so two 1024-lane workgroups share a CU and one loads while the other
// computes (what large batches need).
// EARLY: gamma and beta are requested in front of the wait for the data (gn_body).
template <typename T, int K, bool SILU, bool SHARED, bool RAGGED, bool EARLY = K <= kGnEarlyK>
__global__ __launch_bounds__(kGnMaxThreads, (K <= (sizeof(T) == 2 ? 6 : 4) ? 8 : 4)) void gn_slice_kernel(
    const T *x, uint32_t vec_per_unit, uint32_t vec_per_slice, uint32_t shape, const T *chunk, uint32_t hw_mul,
    uint32_t hw_shift, uint32_t ch_per_group, const float *__restrict__ gamma, const float *__restrict__ beta, T *y,
    GnExchange scratch, GnParams p) {
    __shared__ float red[kGnRedSlots];
    __shared__ float stats[2];
    __shared__ float2 aff[!RAGGED && K <= kGnPrefetchAffineK ? 1 : kGnLdsChannels];  // (gamma, beta) of the group's channels
    const GnShape of(shape);
    const FastDiv hw_vec{hw_mul, hw_shift, RAGGED ? p.hw : 0};
    uint32_t unit, slice, part;
    if (SHARED) {  // whole units, `writers` workgroups each
        const uint32_t j = blockIdx.x >> of.xcd_shift;
        part = j & ((1u << of.writers_shift) - 1u);
        unit = ((j >> of.writers_shift) << of.xcd_shift) + (blockIdx.x & ((1u << of.xcd_shift) - 1u));
        slice = 0;
    } else {
        unit = blockIdx.x >> of.split_shift;
        slice = blockIdx.x & ((1u << of.split_shift) - 1u);
        part = 0;
    }
    const uint32_t v_begin = slice * vec_per_slice;
    const uint32_t v_end = min(vec_per_unit, v_begin + vec_per_slice);
    // uniform over the workgroup; the largest K is only launched on slices it fits exactly
    if (K == kGnMaxK || v_end - v_begin == K * of.threads)
        gn_body<T, K, SILU, true, SHARED, RAGGED, EARLY>(x, chunk, y, gamma, beta, scratch, p, of.threads, vec_per_unit, unit, slice, part,
                                          v_begin, v_end, ch_per_group, hw_vec, red, stats, aff);
    else
        gn_body<T, K, SILU, false, SHARED, RAGGED, EARLY>(x, chunk, y, gamma, beta, scratch, p, of.threads, vec_per_unit, unit, slice, part,
                                           v_begin, v_end, ch_per_group, hw_vec, red, stats, aff);
}

// Any shape or alignment (units that are no whole number of vectors, channels of less than a vector, many
// units of a few vectors): one workgroup per unit, three passes over global memory with scalar accesses (the
// second and third pass hit in cache for UNet-sized units).
template <typename T, bool SILU>
__global__ __launch_bounds__(kGenericThreads) void gn_generic_kernel(
    const T *x, const T *chunk, T *y, const float *__restrict__ gamma,
    const float *__restrict__ beta, uint32_t unit_size, uint32_t hw, uint32_t groups,
    uint32_t ch_per_group, float eps) {
    __shared__ float red_a[kGenericThreads / kWave];
    __shared__ float red_b[kGenericThreads / kWave];
    const uint32_t unit = blockIdx.x;
    const T *xin = x + (size_t)unit * unit_size;
    T *yout = y + (size_t)unit * unit_size;
    const uint32_t ch0 = (unit % groups) * ch_per_group;
    const T *cb = chunk ? chunk + (size_t)(unit / groups) * (groups * ch_per_group) + ch0 : nullptr;
    // element i of the unit, with the optional addend, rounded to the storage type
    auto value = [&](uint32_t i) {
        float v = Store<T>::load1(xin + i);
        if (cb) v = round_to_storage<T>(v + Store<T>::load1(cb + i / hw));
        return v;
    };
    float s = 0.0f;
    for (uint32_t i = threadIdx.x; i < unit_size; i += kGenericThreads) s += value(i);
    const float mean = block_sum_rt(s, red_a) / (float)unit_size;
    float q = 0.0f;
    for (uint32_t i = threadIdx.x; i < unit_size; i += kGenericThreads) {
        const float d = value(i) - mean;
        q = fmaf(d, d, q);
    }
    const float rstd = 1.0f / sqrtf(block_sum_rt(q, red_b) / (float)unit_size + eps);
    // every lane re-reads only elements it writes itself, so y may alias x
    for (uint32_t i = threadIdx.x; i < unit_size; i += kGenericThreads) {
        const uint32_t c = ch0 + i / hw;
        const float t = fmaf(value(i) - mean, rstd * gamma[c], beta[c]);
        Store<T>::store1(yout + i, SILU ? silu_f(t) : t);
    }
}

// ---------------------------------------------------------------------------
// GroupNorm with a token-major store: y[b, p, c] = GroupNorm(x)[b, c, p].
// Replaces GroupNorm followed by the (0, 2, 1) permute that turns NCHW into tokens.
// A slice is all channels of the group over a range of positions, so that for each position
// the slice owns one contiguous run of ch_per_group outputs; normalised values go through
// LDS ([channel][position], 16-byte padded pitch) and leave as 4-byte stores that walk those
// runs.  Statistics and the exchange between slices are those of gn_slice_kernel.
// ---------------------------------------------------------------------------
struct GnTokParams {
    uint32_t ch_per_group;
    // as in GnParams, for gn_exchange; vec_per_slice = ch_per_group * position vectors per slice, vec_per_unit = that * split
    uint32_t vec_per_unit, vec_per_slice, split, spin_limit;
    float eps, inv_count;
    FastDiv row_dwords;   // 4-byte words per output run: ch_per_group * sizeof(T) / 4
    uint32_t hw;          // positions per sample
    uint32_t channels;
    uint32_t pitch;       // LDS elements between channels: positions per slice + 16 bytes
};

template <typename T, int K>
__global__ __launch_bounds__(kGnMaxThreads) void gn_tokens_kernel(
    const T *__restrict__ x, uint32_t vec_per_unit, uint32_t nvec, uint32_t pos_mul, uint32_t pos_shift, uint32_t pvs,
    uint32_t hw_vec, uint32_t combos_mul, uint32_t combos_shift, uint32_t combos, uint32_t groups, uint32_t shape,
    T *__restrict__ y, const float *__restrict__ gamma, const float *__restrict__ beta, GnExchange scratch, GnTokParams q) {
    constexpr int EPV = Store<T>::EPV;
    extern __shared__ u32x4 lds_vec[];
    __shared__ float red[kGnRedSlots];
    __shared__ float stats[2];
    const GnTokParams &p = q;
    const GnShape of(shape);
    const FastDiv pos_vecs{pos_mul, pos_shift, pvs};
    const uint32_t tid = threadIdx.x;
    const uint32_t nt = of.threads;
    // block id = group * (batch * split) + sample * split + slice: the workgroups that write
    // pieces of the same output lines (all groups of one sample and position range) have ids
    // that differ by multiples of batch * split, so with workgroups dealt round-robin to the
    // 8 XCDs they meet in one L2 when that product is a multiple of 8 (batch 2 x 4 slices);
    // the slices of a unit stay adjacent
    const uint32_t group = fast_div(blockIdx.x, FastDiv{combos_mul, combos_shift, combos});
    const uint32_t combo = blockIdx.x - group * combos;
    const uint32_t sample = combo >> of.split_shift;
    const uint32_t unit = sample * groups + group;
    const uint32_t slice = combo & ((1u << of.split_shift) - 1u);
    const u32x4 *xin = reinterpret_cast<const u32x4 *>(x) + (size_t)unit * vec_per_unit;

    // lane-local vector -> (channel of the group, position vector of the slice)
    u32x4 raw[K];
    uint32_t cl[K], pv[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint32_t vl = min(k * nt + tid, nvec - 1);  // ragged tail re-reads the last vector
        cl[k] = fast_div(vl, pos_vecs);
        pv[k] = vl - cl[k] * pvs;
        raw[k] = load_stream(xin + (size_t)cl[k] * hw_vec + slice * pvs + pv[k]);
        const bool have = k * nt + tid < nvec;  // lanes past the end hold zeros (the statistics rely on it)
#pragma unroll
        for (int i = 0; i < 4; i++) raw[k][i] = have ? raw[k][i] : 0u;
    }
    __builtin_amdgcn_sched_barrier(0);  // (what follows waits for the arguments in memory)
    unsigned long long count = 0;
    if (p.split > 1 && tid == 0) count = gn_exchange_enter(scratch, p.split, unit);
    const uint32_t ch0 = group * q.ch_per_group;

    float slice_mean, slice_m2;
    gn_slice_stats<T, K, false>(raw, nvec, nt, red, slice_mean, slice_m2);

    float mean, rstd;
    if (p.split == 1) {
        mean = slice_mean;
        rstd = __builtin_amdgcn_rsqf(slice_m2 * p.inv_count + p.eps);
    } else {
        // vector i of slice l: channel i / pos_vecs of the group, position vector i % pos_vecs
        auto read = [&](uint32_t l, uint32_t i) {
            const uint32_t c = fast_div(i, pos_vecs);
            return xin[(size_t)c * hw_vec + l * pvs + (i - c * pvs)];
        };
        gn_exchange<T>(scratch, p, unit, slice, count, slice_mean, slice_m2, stats, read);
        mean = stats[0];
        rstd = stats[1];
    }

    // ---- normalise into LDS as [channel][position]
    T *lds = reinterpret_cast<T *>(lds_vec);
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (k * nt + tid < nvec) {
            const float a = rstd * gamma[ch0 + cl[k]];
            const float b = beta[ch0 + cl[k]];
            float f[EPV];
            Store<T>::unpack(raw[k], f);
#pragma unroll
            for (int e = 0; e < EPV; e++) f[e] = fmaf(f[e] - mean, a, b);
            *reinterpret_cast<u32x4 *>(lds + (size_t)cl[k] * q.pitch + pv[k] * EPV) = Store<T>::pack(f);
        }
    }
    __syncthreads();

    // ---- token-major store: for each position of the slice one run of ch_per_group values
    const uint32_t rows = pvs * EPV;                         // positions in the slice
    const uint32_t words = rows * q.row_dwords.d;            // 4-byte words to write
    const size_t first = ((size_t)sample * q.hw + (size_t)slice * rows) * q.channels + ch0;
    uint32_t *out = reinterpret_cast<uint32_t *>(y + first);
    const uint32_t row_stride = q.channels * sizeof(T) / 4;  // words between positions
    for (uint32_t i = tid; i < words; i += nt) {
        const uint32_t r = fast_div(i, q.row_dwords);
        const uint32_t c = i - r * q.row_dwords.d;
        uint32_t w;
        if (sizeof(T) == 2) {
            const uint16_t lo = reinterpret_cast<const uint16_t *>(lds)[(2 * c) * q.pitch + r];
            const uint16_t hi = reinterpret_cast<const uint16_t *>(lds)[(2 * c + 1) * q.pitch + r];
            w = (uint32_t)lo | ((uint32_t)hi << 16);
        } else {
            w = reinterpret_cast<const uint32_t *>(lds)[c * q.pitch + r];
        }
        out[(size_t)r * row_stride + c] = w;
    }
}

// The token-major norm for units that stay whole: `writers` workgroups (one or several) per unit, each of which loads
// and reduces all of it and stores its own part, all channels of the group over a range of positions (several writers: as
// in gn_slice_kernel<..., SHARED>, nothing is exchanged).  What a part needs goes to LDS as it was loaded, before the
// statistics are there, so one barrier covers both; it is normalised on the way out, by lanes that keep to their channels.
// An XCD takes units_per_xcd units in a row: what the writers of a unit load meets in its L2, and so do the pieces of an
// output line (ch_per_group elements each) that neighbouring groups store; with units dealt to the XCDs in turn a line
// went to memory in several.  KiB written (WRITE_SIZE), units in turn and so, which is the output's size: fp16 batch 2, 640
// channels at 32 x 32 4096 / 2560, at 36 x 28 4048 / 2520, 1280 at 16 x 16 1536 / 1280; fp32 640 at 32 x 32 6144 / 5120.
// RAGGED: hw is no whole number of vectors, a vector may cross from one channel into the next; LDS then holds the whole unit
// as it lies in memory.
struct GnTokUnitParams {
    FastDiv groups;          // per sample
    uint32_t ch_per_group, channels, hw;
    uint32_t part_pos;       // positions of a part; of the last one what is left
    uint32_t pitch;          // LDS elements between channels
    uint32_t row_step;       // positions that the workgroup stores at a time
    FastDiv hw_vec;          // vectors per channel (not RAGGED)
    FastDiv row_dwords;      // 4-byte words per output run: ch_per_group * sizeof(T) / 4
    float eps, inv_count;
};

// What a lane stores: always the same 4 bytes of an output run (its channels), of every row_step-th position.
// Stores of 4 bytes: 8 and 16 bytes at a time read LDS with more bank conflicts (us with 16 / 8 / 4 bytes, fp16 batch 2: 1280
// channels at 16 x 16 4.2 / - / 3.7, 640 at 32 x 32 - / 4.9 / 4.7).
template <typename T>
struct GnTokStore {
    static constexpr int N = 4 / (int)sizeof(T);  // channels per store
    uint32_t row0, c0, ch0, sample;
    float g[N], b[N];

    __device__ __forceinline__ GnTokStore(uint32_t unit, const GnTokUnitParams &q) {
        row0 = fast_div(threadIdx.x, q.row_dwords);
        c0 = (threadIdx.x - row0 * q.row_dwords.d) * N;
        sample = fast_div(unit, q.groups);
        ch0 = (unit - sample * q.groups.d) * q.ch_per_group + c0;
    }

    __device__ __forceinline__ void fetch(const float *gamma, const float *beta) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            g[i] = gamma[ch0 + i];
            b[i] = beta[ch0 + i];
        }
    }

    __device__ __forceinline__ void operator()(const T *lds, T *y, uint32_t pos0, uint32_t rows, float mean, float rstd,
                                               const GnTokUnitParams &q) const {
        if (row0 >= q.row_step) return;
        float a[N];
#pragma unroll
        for (int i = 0; i < N; i++) a[i] = rstd * g[i];
        T *out = y + ((size_t)sample * q.hw + pos0) * q.channels + ch0;
        const T *in = lds + c0 * q.pitch;
#pragma unroll 4
        for (uint32_t r = row0; r < rows; r += q.row_step) {
            float f[N];
#pragma unroll
            for (int i = 0; i < N; i++) f[i] = fmaf(Store<T>::load1(in + i * q.pitch + r) - mean, a[i], b[i]);
            uint32_t w;
            if constexpr (sizeof(T) == 2) {
                const __half2 h = __floats2half2_rn(f[0], f[N - 1]);
                w = *reinterpret_cast<const uint32_t *>(&h);
            } else {
                w = __float_as_uint(f[0]);
            }
            *reinterpret_cast<uint32_t *>(out + (size_t)r * q.channels) = w;
        }
    }
};

template <typename T, int K, bool RAGGED, bool EARLY>
__global__ __launch_bounds__(kGnMaxThreads) void gn_tokens_unit_kernel(
    const T *__restrict__ x, uint32_t nvec, uint32_t units_per_xcd, uint32_t shape, T *__restrict__ y,
    const float *__restrict__ gamma, const float *__restrict__ beta, GnTokUnitParams q) {
    constexpr int EPV = Store<T>::EPV;
    extern __shared__ u32x4 lds_vec[];
    __shared__ float red[kGnRedSlots];
    const GnShape of(shape);
    const uint32_t tid = threadIdx.x, nt = of.threads;
    const uint32_t of_xcd = blockIdx.x >> of.xcd_shift;
    const uint32_t part = of_xcd & ((1u << of.writers_shift) - 1u);
    const uint32_t unit = (blockIdx.x & ((1u << of.xcd_shift) - 1u)) * units_per_xcd + (of_xcd >> of.writers_shift);
    const u32x4 *xin = reinterpret_cast<const u32x4 *>(x) + (size_t)unit * nvec;
    T *lds = reinterpret_cast<T *>(lds_vec);
    u32x4 raw[K];
#pragma unroll
    for (int k = 0; k < K; k++) raw[k] = load_stream(xin + min(k * nt + tid, nvec - 1));  // ragged tail: the last vector again
    __builtin_amdgcn_sched_barrier(0);  // (loads return in order: the data does not wait for gamma and beta)
    const uint32_t pos0 = part * q.part_pos, rows = min(q.part_pos, q.hw - pos0);
    GnTokStore<T> store(unit, q);
    if (EARLY) store.fetch(gamma, beta);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint32_t v = k * nt + tid;
        const bool have = v < nvec;
        if (RAGGED) {
            if (have) lds_vec[v] = raw[k];
        } else {
            const uint32_t c = fast_div(v, q.hw_vec), p = (v - c * q.hw_vec.d) * EPV - pos0;
            if (have && p < rows) *reinterpret_cast<u32x4 *>(lds + c * q.pitch + p) = raw[k];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) raw[k][i] = have ? raw[k][i] : 0u;  // (the statistics rely on it)
    }
    float mean, m2;
    gn_slice_stats<T, K, false>(raw, nvec, nt, red, mean, m2);  // (its barrier covers the tile)
    const float rstd = __builtin_amdgcn_rsqf(m2 * q.inv_count + q.eps);
    if (!EARLY) store.fetch(gamma, beta);
    store(RAGGED ? lds + pos0 : lds, y, pos0, rows, mean, rstd, q);
}

// Any shape: one workgroup per unit, three passes, element-wise scattered stores.
template <typename T>
__global__ __launch_bounds__(kGenericThreads) void gn_tokens_generic_kernel(
    const T *__restrict__ x, T *__restrict__ y, const float *__restrict__ gamma,
    const float *__restrict__ beta, uint32_t unit_size, uint32_t hw, uint32_t groups,
    uint32_t ch_per_group, float eps) {
    __shared__ float red_a[kGenericThreads / kWave];
    __shared__ float red_b[kGenericThreads / kWave];
    const uint32_t unit = blockIdx.x;
    const T *xin = x + (size_t)unit * unit_size;
    float s = 0.0f;
    for (uint32_t i = threadIdx.x; i < unit_size; i += kGenericThreads) s += Store<T>::load1(xin + i);
    const float mean = block_sum_rt(s, red_a) / (float)unit_size;
    float m2 = 0.0f;
    for (uint32_t i = threadIdx.x; i < unit_size; i += kGenericThreads) {
        const float d = Store<T>::load1(xin + i) - mean;
        m2 = fmaf(d, d, m2);
    }
    const float rstd = 1.0f / sqrtf(block_sum_rt(m2, red_b) / (float)unit_size + eps);
    const uint32_t ch0 = (unit % groups) * ch_per_group;
    const uint32_t channels = groups * ch_per_group;
    T *yout = y + (size_t)(unit / groups) * hw * channels;
    for (uint32_t i = threadIdx.x; i < unit_size; i += kGenericThreads) {
        const uint32_t c = ch0 + i / hw, pos = i % hw;
        const float t = fmaf(Store<T>::load1(xin + i) - mean, rstd * gamma[c], beta[c]);
        Store<T>::store1(yout + (size_t)pos * channels + c, t);
    }
}

// ---------------------------------------------------------------------------
// The same in two launches: gn_stats_kernel leaves (mean, M2) of every slice of every unit in the
// scratch, gn_tokens_apply_kernel transposes 64 x 64 tiles (tile_transpose.h) and normalises them on
// the way.  The second launch reads x again, from the caches.  Takes every unit that is a whole number of
// vectors, whatever its rows are: fp16 batch 2, 1280 channels at 18 x 14 27.2 -> 5.8 us, at 9 x 7 7.9 -> 5.3, at
// 22 x 18 44.1 -> 6.4 (before: one workgroup per unit, three passes in single elements).
// ---------------------------------------------------------------------------
constexpr int kStatsThreads = 256;
constexpr int kStatsUnroll = 4;  // vectors per lane in flight

// (mean, M2) of one slice per workgroup.  Bound by the read of x.  Plain loads: the next launch wants
// the lines in the caches.
template <typename T>
__global__ __launch_bounds__(kStatsThreads) void gn_stats_kernel(const T *__restrict__ x, uint32_t vec_per_unit,
                                                                 uint32_t vec_per_slice, uint32_t slices_mul,
                                                                 uint32_t slices_shift, uint32_t slices,
                                                                 float2 *__restrict__ partials) {
    constexpr int EPV = Store<T>::EPV;
    __shared__ float2 red[kStatsThreads / kWave];
    __shared__ float red_c[kStatsThreads / kWave];
    const uint32_t unit = fast_div(blockIdx.x, FastDiv{slices_mul, slices_shift, slices});
    const uint32_t slice = blockIdx.x - unit * slices;
    const uint32_t begin = slice * vec_per_slice;
    const uint32_t n = min(vec_per_unit, begin + vec_per_slice) - begin;
    const u32x4 *in = reinterpret_cast<const u32x4 *>(x) + (size_t)unit * vec_per_unit + begin;
    // every vector of the slice that is this lane's, kStatsUnroll requested at a time; what lies past
    // the end re-reads the last vector and counts as `past`
    auto for_each = [&](const u32x4 &past, auto use) {
        for (uint32_t base = threadIdx.x; base < n; base += kStatsThreads * kStatsUnroll) {
            u32x4 raw[kStatsUnroll];
#pragma unroll
            for (int u = 0; u < kStatsUnroll; u++) raw[u] = in[min(base + u * kStatsThreads, n - 1)];
#pragma unroll
            for (int u = 0; u < kStatsUnroll; u++) use(base + u * kStatsThreads < n ? raw[u] : past);
        }
    };
    float s[2] = {0.0f, 0.0f}, q[2] = {0.0f, 0.0f};
    for_each(u32x4{0, 0, 0, 0}, [&](const u32x4 &v) { Moments<T>::add(v, s, q); });
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const float sums = wave_sum_of_two(s[0] + s[1], q[0] + q[1]);
    if (lane % kGnRedRow == 0 && lane < 2 * kGnRedRow) reinterpret_cast<float *>(&red[wave])[lane / kGnRedRow] = sums;
    __syncthreads();
    float sum_x = 0.0f, sum_xx = 0.0f;
#pragma unroll
    for (int i = 0; i < kStatsThreads / kWave; i++) {
        sum_x += red[i].x;
        sum_xx += red[i].y;
    }
    const float mean = sum_x / (float)(n * EPV);
    float m2 = sum_xx - sum_x * mean;
    // as in gn_slice_stats: when the mean is large against the spread, a second pass about the mean
    if (!(sum_x * mean <= kGnFastMoments * m2)) {  // uniform over the workgroup
        float c = 0.0f;
        for (uint32_t i = threadIdx.x; i < n; i += kStatsThreads) {
            float f[EPV];
            Store<T>::unpack(in[i], f);
#pragma unroll
            for (int e = 0; e < EPV; e++) {
                const float d = f[e] - mean;
                c = fmaf(d, d, c);
            }
        }
        const float wave_c = wave_sum(c);
        if (lane == 0) red_c[wave] = wave_c;
        __syncthreads();
        m2 = 0.0f;
#pragma unroll
        for (int i = 0; i < kStatsThreads / kWave; i++) m2 += red_c[i];
    }
    if (threadIdx.x == 0) partials[(size_t)unit * kGnStatSlices + slice] = make_float2(mean, m2);
}

// (no field that the kernel does not read: see GnParams)
struct GnApplyParams {
    uint32_t vec_per_unit, vec_per_slice;  // of the statistics
    float eps, inv_count;
};

// JFAST, RAGGED: as in permute_021_words_kernel.
// LINES: the rows of x are whole cache lines.  Otherwise every tile shares lines of x with the tiles beside it, two of three in
// fp16: the tiles of a row then run one after the other on one XCD (each takes a run of the plane's tiles, row by
// row), and their loads leave the lines in its caches.  All tiles of tensors of 10 - 30 MB are in flight at once and ask for what they
// share at the same time, from other XCDs and past the caches otherwise.  us, both launches, in the order of the blocks with streaming
// loads / so: fp32 1280 channels at 2800 positions batch 2 18.95 / 15.75, 640 at 9072 16.5 / 13.4, fp16 1280 at 5600 12.2 / 9.2,
// 640 at 9896 batch 2 19.1 / 15.0, 960 at 2460 batch 16 (no whole vectors) 52.5 / 43.9; over 100 random shapes 0.86.  Rows of
// whole lines: fp16 1280 at 256 batch 39 14.5 / 15.5, 320 at 64 x 64 batch 16 21.4 / 22.6.
template <typename T, bool JFAST, bool RAGGED, bool LINES>
__global__ __launch_bounds__(kTileThreads) void gn_tokens_apply_kernel(
    const T *__restrict__ x, uint32_t channels, uint32_t hw, const float2 *__restrict__ partials, uint32_t groups,
    uint32_t cpg_mul, uint32_t cpg_shift, uint32_t slices_and_xcd_shift, const float *__restrict__ gamma,
    const float *__restrict__ beta, T *__restrict__ y, GnApplyParams p) {
    const uint32_t slices = slices_and_xcd_shift & 255u;
    constexpr int ES = (int)sizeof(T), EPV = Store<T>::EPV;
    constexpr uint32_t kTeam = kTileThreads / kTile;  // lanes that merge one channel's statistics
    __shared__ u32x4 tile4[tile_lds_words<ES>()];
    __shared__ float4 affine[kTile];  // (mean, rstd * gamma, beta) of the tile's channels
    uint32_t kt = JFAST ? blockIdx.y : blockIdx.x, jt = JFAST ? blockIdx.x : blockIdx.y;
    if (!LINES) {  // block ids go to the XCDs in turn
        const uint32_t nj = (channels + kTile - 1) / kTile, nk = (hw + kTile - 1) / kTile, xcd_shift = slices_and_xcd_shift >> 8;
        const uint32_t id = JFAST ? kt * nj + jt : jt * nk + kt;
        const uint32_t xcd = id & ((1u << xcd_shift) - 1u), tiles = nj * nk;
        const uint32_t tile = xcd * (tiles >> xcd_shift) + min(xcd, tiles & ((1u << xcd_shift) - 1u)) + (id >> xcd_shift);
        jt = tile / nk;
        kt = tile - jt * nk;
    }
    const uint32_t k0 = kt * kTile, j0 = jt * kTile;
    const size_t plane = (size_t)blockIdx.z * channels * hw;
    // Chan's formula over the unit's slices, by the four lanes of a channel
    auto ready = [&]() {
        const uint32_t j = threadIdx.x / kTeam, lane = threadIdx.x % kTeam;
        const uint32_t c = min(j0 + j, channels - 1);
        const float g = gamma[c], b = beta[c];
        const float2 *of_unit = partials + (size_t)(blockIdx.z * groups + fast_div(c, FastDiv{cpg_mul, cpg_shift, 0})) * kGnStatSlices;
        float n_l[kGnStatSlices / kTeam];
        float2 part[kGnStatSlices / kTeam];
#pragma unroll
        for (uint32_t i = 0; i < kGnStatSlices / kTeam; i++) {
            const uint32_t l = lane + i * kTeam;
            part[i] = of_unit[l < slices ? l : 0];
        }
        // (all of them are requested before the first is used: left to itself the compiler puts each behind a branch on
        // its slice and waits for one after the other.  us, the token norm of 320 channels at 64 x 64, fp16 batch 2: 6.52 -> 6.45)
        asm volatile("" : : "s"(y));  // (an argument in memory: loaded here, not when the first store wants it)
#pragma unroll
        for (uint32_t i = 0; i < kGnStatSlices / kTeam; i++) asm volatile("" : "+v"(part[i].x), "+v"(part[i].y));
        float weighted = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < kGnStatSlices / kTeam; i++) {
            const uint32_t l = lane + i * kTeam;
            const bool have = l < slices;
            const uint32_t begin = l * p.vec_per_slice;
            n_l[i] = have ? (float)((min(p.vec_per_unit, begin + p.vec_per_slice) - begin) * EPV) : 0.0f;
            weighted = have ? fmaf(part[i].x, n_l[i], weighted) : weighted;
        }
        const float mean = team_sum<kTeam>(weighted) * p.inv_count;
        float m2 = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < kGnStatSlices / kTeam; i++) {
            const float d = part[i].x - mean;
            if (lane + i * kTeam < slices) m2 += fmaf(n_l[i] * d, d, part[i].y);
        }
        const float rstd = __builtin_amdgcn_rsqf(team_sum<kTeam>(m2) * p.inv_count + p.eps);
        if (lane == 0) affine[j] = make_float4(mean, rstd * g, b, 0.0f);
        __syncthreads();
    };
    auto normalise = [&](uint32_t row, const u32x4 &v) {
        const float4 a = affine[row];
        float f[EPV];
        Store<T>::unpack(v, f);
#pragma unroll
        for (int e = 0; e < EPV; e++) f[e] = fmaf(f[e] - a.x, a.y, a.z);
        return Store<T>::pack(f);
    };
    transpose_tile<ES, RAGGED, !LINES>(reinterpret_cast<const char *>(x + plane), reinterpret_cast<char *>(y + plane), channels,
                               hw, j0, k0, tile4, ready, normalise);
}

// ---------------------------------------------------------------------------
// Host: launches (the plan comes from gn_plan.hip)
// ---------------------------------------------------------------------------
// log2 of the distance between the block ids of a unit's writers: the XCD count when the
// workgroups of a launch are dealt to a power-of-two number of XCDs in turn and the units come
// in whole rows of that many (the writers then share an XCD), else 0 (adjacent ids).
inline uint32_t gn_xcd_shift(const Chip &chip, bool shared, size_t units) {
    if (!shared || chip.xcds <= 1 || (chip.xcds & (chip.xcds - 1)) != 0 || units % chip.xcds != 0) return 0;
    return (uint32_t)__builtin_ctz(chip.xcds);
}

// The leading plain arguments of gn_slice_kernel beside those of GnParams.
struct GnGeometry {
    uint32_t blocks, threads, shape, ch_per_group;
    uint32_t per_cu;  // workgroups, rounded down
    FastDiv hw;  // vectors per channel (RAGGED: elements per channel)
};

template <typename T, int K, bool RAGGED>
void gn_launch_k(bool silu, bool shared, const GnGeometry &g, hipStream_t stream, const T *x,
                 const T *chunk, T *y, const float *gamma, const float *beta, const GnScratch &sc,
                 const GnParams &p) {
    if (K <= kGnSharedMaxK && shared) {
        constexpr int KS = K <= kGnSharedMaxK ? K : 1;  // (larger K never get here: no such instances)
        launch((silu ? gn_slice_kernel<T, KS, true, true, RAGGED> : gn_slice_kernel<T, KS, false, true, RAGGED>),
               dim3(g.blocks), dim3(g.threads), 0, stream, x, p.vec_per_unit, p.vec_per_slice, g.shape, chunk, g.hw.mul,
               g.hw.shift, g.ch_per_group, gamma, beta, y, sc, p);
    } else {
        auto *kernel = silu ? gn_slice_kernel<T, K, true, false, RAGGED> : gn_slice_kernel<T, K, false, false, RAGGED>;
        if constexpr (sizeof(T) == 4 && K <= kGnEarlyK && !RAGGED) {
            // Float slices of launches with several workgroups per CU ask for gamma and beta behind the data (see gn_body): us, early /
            // so, two per CU 192 channels at 752 positions batch 17 (three vectors) 5.68 / 4.95, 256 at 800 batch 16 (four) 5.98 / 5.35, 384
            // at 704 batch 18 (five) 8.81 / 8.41; six 256 at 304 batch 48 6.41 / 5.92, 512 at 192 batch 60 9.53 / 8.90; against it three
            // per CU 128 at 568 batch 24 (three) 4.01 / 4.10, two 128 at 824 batch 16 (two) 4.02 / 4.09.  (Half slices of as many: 0.95
            // to 1.03 of the early ones.)
            if (g.per_cu >= (K >= 3 ? 2u : 4u)) kernel = silu ? gn_slice_kernel<T, K, true, false, RAGGED, false> : gn_slice_kernel<T, K, false, false, RAGGED, false>;
        }
        launch(kernel, dim3(g.blocks), dim3(g.threads), 0, stream, x, p.vec_per_unit, p.vec_per_slice, g.shape, chunk, g.hw.mul,
               g.hw.shift, g.ch_per_group, gamma, beta, y, sc, p);
    }
}

template <typename T, bool RAGGED>
int gn_launch(uint32_t k, bool silu, bool shared, const GnGeometry &g, hipStream_t stream, const T *x,
              const T *chunk, T *y, const float *gamma, const float *beta, const GnScratch &sc, const GnParams &p) {
    switch (k) {
        case 1: gn_launch_k<T, 1, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 2: gn_launch_k<T, 2, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 3: gn_launch_k<T, 3, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 4: gn_launch_k<T, 4, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 5: gn_launch_k<T, 5, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 6: gn_launch_k<T, 6, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 8: gn_launch_k<T, 8, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 10: gn_launch_k<T, 10, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 12: gn_launch_k<T, 12, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 16: gn_launch_k<T, 16, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        case 20: gn_launch_k<T, 20, RAGGED>(silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p); break;
        default: return MSD_ERR_INVALID_VALUE;  // not a K the kernels are built for: a planning error
    }
    return launch_status();
}

template <typename T>
int gn_generic(bool silu, const T *x, const T *chunk, T *y, const float *gamma, const float *beta,
               size_t units, size_t unit_size, size_t hw, size_t groups, size_t cpg, float eps,
               hipStream_t stream) {
    launch((silu ? gn_generic_kernel<T, true> : gn_generic_kernel<T, false>),
                       dim3((uint32_t)units), dim3(kGenericThreads), 0, stream, x, chunk, y, gamma, beta,
                       (uint32_t)unit_size, (uint32_t)hw, (uint32_t)groups, (uint32_t)cpg, eps);
    return launch_status();
}

}  // namespace

template <typename T>
int gn_dispatch(const void *xv, const void *chunkv, void *yv, const float *gamma, const float *beta,
                size_t batch, size_t channels, size_t hw, size_t groups, float eps, bool silu,
                const GnScratch *fixed, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    const int tune_spin = g_tuning.gn_spin_limit.load(std::memory_order_relaxed);
    const T *x = static_cast<const T *>(xv);
    const T *chunk = static_cast<const T *>(chunkv);
    T *y = static_cast<T *>(yv);
    const size_t cpg = channels / groups;
    const size_t unit_size = cpg * hw;
    const size_t units = batch * groups;
    if (units == 0 || unit_size == 0) return MSD_OK;
    if (units > 0x7FFFFFFFull || unit_size > 0x7FFFFFFFull) return MSD_ERR_INVALID_VALUE;
    if (fixed != nullptr && units > fixed->units) return MSD_ERR_SCRATCH_LIMIT;
    // several workgroups may share a unit only if none of them can store into what another still
    // loads: the output must lie apart from the input
    const char *xb = reinterpret_cast<const char *>(x), *yb = reinterpret_cast<const char *>(y);
    const size_t bytes = units * unit_size * sizeof(T);
    const bool apart = xb + bytes <= yb || yb + bytes <= xb;
    const bool ragged = hw % EPV != 0;
    auto decide = [&](size_t max_units) {
        return gn_decide(sizeof(T), batch, channels, hw, groups, aligned16(x) && aligned16(y), max_units, apart);
    };
    GnDecision d = decide(fixed != nullptr ? fixed->units : kGnMaxUnits);
    GnScratch sc{};
    // Channels of no whole vectors go without scratch where there is none to take: in whole units, or
    // (units that no workgroup holds) through the general kernel
    if (ragged && fixed == nullptr && d.split > 1 && !optional_scratch(stream, &sc)) d = decide(0);
    if (d.split == 0)
        return gn_generic<T>(silu, x, chunk, y, gamma, beta, units, unit_size, hw, groups, cpg, eps, stream);

    const uint32_t split = d.split;
    GnParams p;
    p.vec_per_unit = (uint32_t)(unit_size / EPV);
    p.vec_per_slice = d.vec_per_slice;
    p.split = split;
    p.groups = make_fast_div((uint32_t)groups);
    p.hw = (uint32_t)hw;
    p.eps = eps;
    p.inv_count = 1.0f / (float)unit_size;
    p.spin_limit = tune_spin > 0 ? (uint32_t)tune_spin : kGnSpinLimit;
    const bool shared = d.writers > 1;
    p.part_vecs = (uint32_t)((((p.vec_per_unit + d.writers - 1) / d.writers + kWave - 1) / kWave) * kWave);
    const Chip chip = chip_info();
    const size_t blocks = units * split * d.writers;
    const GnGeometry g{(uint32_t)blocks, d.threads,
                       gn_shape_word((uint32_t)__builtin_ctz(split), (uint32_t)__builtin_ctz(d.writers),
                                     gn_xcd_shift(chip, shared, units), d.threads),
                       (uint32_t)cpg, (uint32_t)(blocks / chip.cus), make_fast_div((uint32_t)(ragged ? hw : hw / EPV))};

    if (fixed != nullptr) {
        sc = *fixed;
    } else if (split > 1 && !ragged) {
        const hipError_t err = get_scratch(stream, &sc);
        if (err != hipSuccess) return (int)err;
    }
    if (ragged)
        return gn_launch<T, true>(d.k, silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p);
    return gn_launch<T, false>(d.k, silu, shared, g, stream, x, chunk, y, gamma, beta, sc, p);
}

template int gn_dispatch<float>(const void *, const void *, void *, const float *, const float *,
                                size_t, size_t, size_t, size_t, float, bool, const GnScratch *, hipStream_t);
template int gn_dispatch<__half>(const void *, const void *, void *, const float *, const float *,
                                 size_t, size_t, size_t, size_t, float, bool, const GnScratch *, hipStream_t);

namespace {

// How gn_tokens_unit_kernel takes a shape (k == 0: not at all).
struct GnTokUnitPlan {
    uint32_t writers, threads, k;
    bool ragged;
    uint32_t part_pos, pitch;
    size_t lds;
    bool early;
};

constexpr size_t kGnTokMaxLds = 60 * 1024;

// When gn_tokens_unit_kernel requests gamma and beta (EARLY): with the data, so that they have arrived when the sums have, except in large
// launches of many workgroups or of several writers per unit.  There the time is the memory's, and stores that start that much
// earlier, while other workgroups still load, cost more than the wait (us, behind the sums / with the data: fp16 batch 2 1280
// channels at 8 x 8 2.70 / 2.51, at 16 x 16 3.56 / 3.27, batch 16 2560 at 320 positions 13.2 / 12.7; fp32 512 at 784 batch 24
// 13.9 / 17.6, 640 at 784 batch 12, two writers, 10.9 / 13.4, fp16 1280 at 324 batch 48 19.6 / 23.2, 2560 at 380 batch 24
// 26.1 / 24.4; just over two workgroups per CU 512 at 792 batch 18 12.1 / 15.2, fp16 960 at 840 batch 19 17.7 / 21.5, fp32 640 at 700
// batch 19 22.3 / 21.4.  With the data over behind the sums, means over 146 random shapes: up to two workgroups per CU, one
// writer, 0.98, more of them and 16 MB or more 1.03, below that 0.99).
inline bool gn_tokens_early_affine(const Chip &chip, size_t bytes, size_t blocks, uint32_t writers) {
    return bytes < (size_t)16 << 20 || (writers == 1 && blocks <= 2 * (size_t)chip.cus);
}

template <typename T>
GnTokUnitPlan gn_tokens_unit_plan(const Chip &chip, size_t units, size_t cpg, size_t hw, int tune_writers) {
    constexpr size_t EPV = Store<T>::EPV;
    const size_t unit_size = cpg * hw, run = cpg * sizeof(T);
    GnTokUnitPlan pl{1, 0, 0, hw % EPV != 0, 0, 0, 0, false};
    if (unit_size % EPV != 0 || run % 4 != 0 || units > 0x7FFFFFFFull / 16) return pl;
    // as many writers as give the chip a workgroup per CU; they must share an XCD (gn_auto_writers)
    const bool may_share = (chip.xcds & (chip.xcds - 1)) == 0 && units % chip.xcds == 0;
    uint32_t w = tune_writers > 0 ? (uint32_t)tune_writers : 1;
    if (tune_writers == 0 && may_share)
        while (w < 8 && units * w * 2 <= chip.cus) w *= 2;
    auto cut = [&](uint32_t parts) {
        const size_t vecs = (hw / EPV + parts - 1) / parts;  // per channel and part
        pl.writers = parts;
        pl.part_pos = (uint32_t)(pl.ragged ? (hw + parts - 1) / parts : vecs * EPV);
        pl.pitch = (uint32_t)(pl.ragged ? hw : vecs * EPV + EPV);
        pl.lds = (cpg * pl.pitch * sizeof(T) + 15) / 16 * 16;
    };
    cut(w);
    while (!pl.ragged && tune_writers == 0 && may_share && pl.lds > kGnTokMaxLds && pl.writers < 8) cut(pl.writers * 2);
    while (pl.writers > 1 && (size_t)(pl.writers - 1) * pl.part_pos >= hw) cut(pl.writers / 2);  // no empty part
    if (pl.lds > kGnTokMaxLds) return pl;
    const uint32_t max_k = sizeof(T) == 4 ? 10 : kGnMaxRaggedK;
    // (writers that a knob asks for get the lanes of a launch with a workgroup per CU)
    const size_t blocks = tune_writers > 0 ? std::min(units * pl.writers, (size_t)chip.cus) : units * pl.writers;
    const GnThreads t = gn_threads_for(chip, sizeof(T), (uint32_t)(unit_size / EPV), 1, blocks, max_k, false, pl.writers > 1);
    pl.threads = t.threads;
    pl.k = t.threads < run / 4 ? 0 : (uint32_t)t.k;  // (a lane per word of an output run)
    pl.early = gn_tokens_early_affine(chip, units * unit_size * sizeof(T), units * pl.writers, pl.writers);
    return pl;
}

template <typename T, int K>
void gn_tokens_unit_launch(const GnTokUnitPlan &pl, uint32_t xcd_shift, uint32_t units, uint32_t vec_per_unit, hipStream_t stream,
                           const T *x, T *y, const float *gamma, const float *beta, const GnTokUnitParams &q) {
    const uint32_t blocks = units * pl.writers, units_per_xcd = units >> xcd_shift;
    auto *kernel = pl.early ? (pl.ragged ? gn_tokens_unit_kernel<T, K, true, true> : gn_tokens_unit_kernel<T, K, false, true>)
                            : (pl.ragged ? gn_tokens_unit_kernel<T, K, true, false> : gn_tokens_unit_kernel<T, K, false, false>);
    launch(kernel, dim3(blocks), dim3(pl.threads), pl.lds, stream, x, vec_per_unit, units_per_xcd,
           gn_shape_word(0, (uint32_t)__builtin_ctz(pl.writers), xcd_shift, pl.threads), y, gamma, beta, q);
}

template <typename T>
int gn_tokens_unit(const GnTokUnitPlan &pl, const Chip &chip, const T *x, T *y, const float *gamma, const float *beta,
                   size_t units, size_t channels, size_t hw, size_t groups, float eps, hipStream_t stream) {
    constexpr uint32_t EPV = Store<T>::EPV;
    const size_t cpg = channels / groups, unit_size = cpg * hw;
    const uint32_t vec_per_unit = (uint32_t)(unit_size / EPV), xcd_shift = gn_xcd_shift(chip, true, units);
    GnTokUnitParams q;
    q.groups = make_fast_div((uint32_t)groups);
    q.ch_per_group = (uint32_t)cpg;
    q.channels = (uint32_t)channels;
    q.hw = (uint32_t)hw;
    q.part_pos = pl.part_pos;
    q.pitch = pl.pitch;
    q.hw_vec = make_fast_div(pl.ragged ? 1u : (uint32_t)hw / EPV);
    q.row_dwords = make_fast_div((uint32_t)(cpg * sizeof(T) / 4));
    q.row_step = pl.threads / q.row_dwords.d;
    q.eps = eps;
    q.inv_count = 1.0f / (float)unit_size;
    switch (pl.k) {
        case 1: gn_tokens_unit_launch<T, 1>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 2: gn_tokens_unit_launch<T, 2>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 3: gn_tokens_unit_launch<T, 3>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 4: gn_tokens_unit_launch<T, 4>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 5: gn_tokens_unit_launch<T, 5>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 6: gn_tokens_unit_launch<T, 6>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 8: gn_tokens_unit_launch<T, 8>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        case 10: gn_tokens_unit_launch<T, 10>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q); break;
        default:  // (12, 16: 2-byte elements only, see max_k)
            if constexpr (sizeof(T) == 2) {
                if (pl.k == 12)
                    gn_tokens_unit_launch<T, 12>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q);
                else
                    gn_tokens_unit_launch<T, 16>(pl, xcd_shift, (uint32_t)units, vec_per_unit, stream, x, y, gamma, beta, q);
            }
    }
    return launch_status();
}

template <typename T, int K>
void gn_tokens_launch(uint32_t blocks, uint32_t threads, size_t lds_bytes, hipStream_t stream,
                      const T *x, T *y, const float *gamma, const float *beta, const GnScratch &sc,
                      const GnTokParams &q, uint32_t groups, uint32_t hw_vec, const FastDiv &pos_vecs, const FastDiv &combos) {
    launch((gn_tokens_kernel<T, K>), dim3(blocks), dim3(threads), lds_bytes, stream, x, q.vec_per_unit, q.vec_per_slice,
           pos_vecs.mul, pos_vecs.shift, pos_vecs.d, hw_vec, combos.mul, combos.shift, combos.d, groups,
           gn_shape_word((uint32_t)__builtin_ctz(q.split), 0, 0, threads), y, gamma, beta, sc, q);
}

// Whether gn_tokens_unit_kernel is the better one launch for a shape it can take: its units are loaded once per writer and
// held by one workgroup, so they may be the longer the fewer there are.  us, the kernels below (slices with an exchange, or
// one workgroup per unit and 4 K positions; two launches for `halves`) and this one: fp16 640 channels, batch 2, at 24 x 24
// 4.9 / 3.8, 36 x 28 7.2 / 4.6, 40 x 40 6.8 / 5.5, batch 8 at 32 x 32 8.9 / 7.9; 1280 at 18 x 14 batch 2 5.6 / 3.7, 8 8.0 / 5.3, at
// 24 x 24 batch 2 6.4 / 5.0; fp32 640 at 32 x 32 batch 2 6.5 / 5.7, 16 24.3 / 22.6, 1280 at 18 x 14 batch 2 7.8 / 4.4.
// Above the limits (ratio of this one to the others over 8000 random shapes, by KB a unit): up to half a unit per CU 128: 0.96,
// 136: 1.01, 152: 1.03; up to one 104: 0.83, 112: 0.88, 120: 1.1 - 1.3; more 64: 0.95, 72: 1.0, 80: 1.0, 88: 1.1.
// Ragged planes: the 2-byte ones whose rows are whole halves of a vector.  The others keep the two launches: 2 x 1280 x 63
// takes 5.1 us in them and would take 2.7 in one, but for which odd planes that holds has not been measured.  Short runs of many units not (128 channels at 5732 batch 10 13.9 / 18.6).
inline bool gn_tokens_stays_whole(const Chip &chip, size_t elt, size_t units, size_t unit_size, size_t cpg, size_t hw) {
    if (hw * elt % 16 != 0 && (elt != 2 || hw % 4 != 0 || (cpg * elt < 40 && units > chip.cus))) return false;
    const size_t limit = units * 2 <= chip.cus ? 128 : units <= chip.cus ? 112 : 72;
    return unit_size * elt <= limit * 1024;
}

// Where the one-launch kernel can run, two launches (1.5 - 2 us more for the smallest tensors) pay when
//   - its stores are short runs (cpg elements, at most 40 bytes, that must meet in the L2) and its units
//     are long enough to be cut (us, before and now: 320 channels at 64 x 64 fp16 batch 2 8.08 -> 7.48, 16
//     35.7 -> 23.6; 640 at 40 x 40 batch 8 12.7 -> 11.4; at 32 x 32 the one launch keeps 9.2 against 9.8), or
//     divide so badly that it gets less than half a workgroup per CU (320 at 40 x 40 batch 2 7.41 -> 6.13; shorter
//     ones keep the one launch: 640 at 432 positions batch 1 3.95 against 4.89);
//   - the tensor is large, so that LDS and registers leave it too few workgroups in flight (fp16 640 at
//     32 x 32 batch 32 27.5 -> 23.4, fp32 320 at 64 x 64 batch 16 61.3 -> 42.7; a copy takes 15.7 and 29; below
//     24 MiB the one launch wins, fp32 640 at 32 x 32 batch 8 12.6 against 13.4).  Not where its workgroups are a
//     whole number per CU, few enough to be in flight at once (fp16 1280 at 2560 positions batch 6, three per CU,
//     19.3 against 24.6; fp32 2560 at 640 batch 6, 16.8 against 21.2) and cut the rows at whole 32 bytes (fp16 1920
//     at 4032 batch 2 in parts of 504 positions 33.1, two launches 18.0), nor where rows are no whole number of
//     lines, which tiles of 64 positions then share (fp16 640 at 36 x 28 batch 32 23.4 against 30.0).
// Both need positions that fill the tiles (fp32 1280 at 288 positions, 4.5 tiles, batch 23 14.2 against 20.7).
// Over 2800 random shapes of 1280 and more elements per unit what this takes is 0.955 of the one launch on average;
// 23 are more than 1.1 times it (to 1.29: fp16 640 at 1232 batch 16 18.9 against 14.6).
inline bool gn_tokens_prefers_two(const Chip &chip, size_t elt, size_t unit_size, size_t units, size_t cpg, size_t hw,
                                  size_t blocks, size_t part_vecs, bool whole) {
    const size_t tiled = (hw + kTile - 1) / kTile * kTile, bytes = units * unit_size * elt;
    if (hw * 16 < tiled * 15) return false;
    if (cpg * elt <= 40)
        return unit_size > 20480 || (!whole && unit_size >= 12288 && blocks * 2 < chip.cus) || bytes >= (size_t)24 << 20;
    if (bytes < (size_t)24 << 20 || hw * elt % 128 != 0) return false;
    const size_t rounds = (blocks + chip.cus - 1) / chip.cus;
    return rounds * 2 > 3 * elt || blocks * 100 <= rounds * chip.cus * 97 || part_vecs % 2 != 0 ||
           (elt == 4 && unit_size > 160000);
}

// The two launches; false where their preconditions do not hold or there is no memory for the partials,
// neither the caller's nor scratch of the stream (nothing has been launched then: the other kernels take
// over).  All launches on one stream, of either element type, share its scratch: the lock keeps another
// thread's pair from coming between.
template <typename T>
bool gn_tokens_two_launches(const T *x, T *y, const float *gamma, const float *beta, size_t batch, size_t channels,
                            size_t hw, size_t groups, float eps, float2 *partials, hipStream_t stream, int *status) {
    constexpr size_t EPV = Store<T>::EPV;
    const size_t cpg = channels / groups, unit_size = cpg * hw, units = batch * groups;
    const dim3 tiles((uint32_t)((hw + kTile - 1) / kTile), (uint32_t)((channels + kTile - 1) / kTile), (uint32_t)batch);
    if (!aligned16(x) || unit_size % EPV != 0 || units > kGnMaxUnits || hw > kTileMaxSide || channels > kTileMaxSide ||
        (tiles.x > 65535 && tiles.y > 65535))
        return false;
    std::unique_lock<std::mutex> lock;
    if (partials == nullptr) {
        GnScratch sc;
        if (!optional_scratch(stream, &sc)) return false;
        partials = sc.partials;
        lock = std::unique_lock<std::mutex>(partials_lock(sc));
    }
    GnApplyParams p;
    p.vec_per_unit = (uint32_t)(unit_size / EPV);
    const Chip chip = chip_info();
    // slices of at most 2048 vectors, shorter (two per lane at least) while the chip has less than two
    // workgroups per CU
    uint32_t slices = 1;
    while (slices < kGnStatSlices && ((units * slices < 2 * (size_t)chip.cus && p.vec_per_unit >= slices * 2 * kStatsThreads) ||
                                      p.vec_per_unit > slices * 2048))
        slices *= 2;
    p.vec_per_slice = (p.vec_per_unit + slices - 1) / slices;
    slices = (p.vec_per_unit + p.vec_per_slice - 1) / p.vec_per_slice;  // (no empty slice)
    const FastDiv by_slices = make_fast_div(slices), by_cpg = make_fast_div((uint32_t)cpg);
    p.eps = eps;
    p.inv_count = 1.0f / (float)unit_size;
    const bool ragged = channels % EPV != 0 || hw % EPV != 0 || !aligned16(y);
    const bool jfast = (channels < hw && tiles.x <= 65535) || tiles.y > 65535;
    const bool lines = !ragged && hw * sizeof(T) % kCacheLine == 0 && reinterpret_cast<uintptr_t>(x) % kCacheLine == 0;
    auto *apply = jfast ? (ragged  ? gn_tokens_apply_kernel<T, true, true, false>
                           : lines ? gn_tokens_apply_kernel<T, true, false, true>
                                   : gn_tokens_apply_kernel<T, true, false, false>)
                        : (ragged  ? gn_tokens_apply_kernel<T, false, true, false>
                           : lines ? gn_tokens_apply_kernel<T, false, false, true>
                                   : gn_tokens_apply_kernel<T, false, false, false>);
    const bool pow2_xcds = (chip.xcds & (chip.xcds - 1)) == 0;
    const uint32_t xcd_shift = pow2_xcds ? (uint32_t)__builtin_ctz(chip.xcds) : 0;
    launch((gn_stats_kernel<T>), dim3((uint32_t)(units * slices)), dim3(kStatsThreads), 0, stream, x, p.vec_per_unit,
           p.vec_per_slice, by_slices.mul, by_slices.shift, slices, partials);
    launch(apply, jfast ? dim3(tiles.y, tiles.x, tiles.z) : tiles, dim3(kTileThreads), 0, stream, x, (uint32_t)channels,
           (uint32_t)hw, partials, (uint32_t)groups, by_cpg.mul, by_cpg.shift, slices | xcd_shift << 8, gamma, beta, y, p);
    *status = launch_status();
    return true;
}

}  // namespace

template <typename T>
int gn_tokens_dispatch(const void *xv, void *yv, const float *gamma, const float *beta, size_t batch,
                       size_t channels, size_t hw, size_t groups, float eps, float2 *partials, hipStream_t stream) {
    constexpr int EPV = Store<T>::EPV;
    constexpr uint32_t kMaxK = sizeof(T) == 4 ? 10 : kGnMaxRaggedK;
    const T *x = static_cast<const T *>(xv);
    T *y = static_cast<T *>(yv);
    const size_t cpg = channels / groups;
    const size_t unit_size = cpg * hw;
    const size_t units = batch * groups;
    if (units == 0 || unit_size == 0) return MSD_OK;
    if (units > 0x7FFFFFFFull || unit_size > 0x7FFFFFFFull) return MSD_ERR_INVALID_VALUE;
    // what the one-launch kernel below does not take: the two launches, or the scalar kernel
    // (short units of small tensors, or of planes much narrower than a tile: one short launch instead of two.  us, one
    // and two: fp16 1 x 320 x 36 3.4 / 5.1, 64 x 2560 x 4 4.5 / 8.3, 22 x 2560 x 10 4.8 / 6.4, 8 x 960 x 28
    // 4.3 / 5.1, 166 x 256 x 79 22.8 / 10.6, 2 x 1280 x 63 7.9 / 5.3.  Over 3100 random shapes 6 are more than 1.1
    // times the one launch, none more than 1.2.)
    auto generic = [&]() {
        int status = MSD_OK;
        const bool pays = unit_size >= 1280 || (unit_size >= 256 && hw >= 24 && units * unit_size >= 400000);
        if (pays &&
            gn_tokens_two_launches<T>(x, y, gamma, beta, batch, channels, hw, groups, eps, partials, stream, &status))
            return status;
        launch((gn_tokens_generic_kernel<T>), dim3((uint32_t)units), dim3(kGenericThreads), 0,
                           stream, x, y, gamma, beta, (uint32_t)unit_size, (uint32_t)hw, (uint32_t)groups,
                           (uint32_t)cpg, eps);
        return launch_status();
    };
    const Chip chip = chip_info();
    const int tune_split = g_tuning.gn_split.load(std::memory_order_relaxed);
    const int tune_writers = g_tuning.gn_writers.load(std::memory_order_relaxed);
    const bool words_ok = aligned16(x) && (reinterpret_cast<uintptr_t>(y) & 3u) == 0;
    // whole units, unless a knob asks for slices (or for what one writer does without sharing: slices)
    GnTokUnitPlan unit{};
    if (words_ok && tune_split <= 1 && tune_writers != 1) unit = gn_tokens_unit_plan<T>(chip, units, cpg, hw, tune_writers);
    const bool whole = unit.k != 0 && (tune_writers > 1 || tune_split == 1 || gn_tokens_stays_whole(chip, sizeof(T), units, unit_size, cpg, hw));
    auto in_one = [&]() { return gn_tokens_unit<T>(unit, chip, x, y, gamma, beta, units, channels, hw, groups, eps, stream); };
    const bool vector_ok = words_ok && hw % EPV == 0 && (cpg * sizeof(T)) % 4 == 0 && (channels * sizeof(T)) % 4 == 0;
    if (whole && (!vector_ok || tune_writers > 1 || tune_split == 1)) return in_one();
    if (!vector_ok) return generic();
    const size_t hw_vec = hw / EPV;
    // slices cut the positions: the split must divide them, fit the registers and the LDS.
    // Cut earlier than gn_dispatch does: the block layout puts the workgroups that write pieces
    // of the same output lines on one XCD when batch * split is a multiple of the XCD count, which
    // is worth more than the exchange costs from 16 Ki elements on.  With half a workgroup per CU
    // or more, units stay whole or (exactly half) go in two; four slices otherwise, eight when
    // even that leaves a quarter of the chip idle and a slice keeps 4 Ki elements.
    uint32_t want = 1;
    if (unit_size > 16384) {
        want = units * 2 > chip.cus ? 1 : units * 2 == chip.cus ? 2 : 4;
        if (units * 16 < 3 * (size_t)chip.cus && unit_size >= 32768) want = 8;
    }
    const int tune_spin = g_tuning.gn_spin_limit.load(std::memory_order_relaxed);
    if (tune_split > 0) want = (uint32_t)tune_split;
    uint32_t split = 0;
    for (uint32_t s = 1; s <= kGnMaxSplit; s *= 2) {
        if (hw_vec % s != 0) break;
        const size_t nvec = cpg * (hw_vec / s);
        const size_t lds = cpg * (hw / s + 16 / sizeof(T)) * sizeof(T);
        if (nvec > (size_t)kGnMaxThreads * kMaxK || lds > kGnTokMaxLds) continue;
        split = s;
        if (s >= want) break;
    }
    if (split == 0 || (split > 1 && units > kGnMaxUnits)) return whole ? in_one() : generic();

    GnTokParams q;
    const size_t pvs = hw_vec / split;  // position vectors of a slice
    const size_t nvec = cpg * pvs;
    q.ch_per_group = (uint32_t)cpg;
    q.vec_per_unit = (uint32_t)(cpg * hw_vec);
    q.vec_per_slice = (uint32_t)nvec;
    q.split = split;
    q.eps = eps;
    q.inv_count = 1.0f / (float)unit_size;
    q.spin_limit = tune_spin > 0 ? (uint32_t)tune_spin : kGnSpinLimit;
    const FastDiv pos_vecs = make_fast_div((uint32_t)pvs), combos = make_fast_div((uint32_t)(batch * split));  // ((sample, slice) pairs)
    q.row_dwords = make_fast_div((uint32_t)(cpg * sizeof(T) / 4));
    q.hw = (uint32_t)hw;
    q.channels = (uint32_t)channels;
    q.pitch = (uint32_t)(pvs * EPV + 16 / sizeof(T));
    const size_t lds_bytes = cpg * q.pitch * sizeof(T);
    const GnThreads pl = gn_threads_for(chip, sizeof(T), (uint32_t)nvec, split, units * split, kMaxK, false, false);
    if (pl.k == 0) return whole ? in_one() : generic();
    const uint32_t blocks = (uint32_t)(units * split);
    if (tune_split == 0 && tune_writers == 0 &&
        gn_tokens_prefers_two(chip, sizeof(T), unit_size, units, cpg, hw, blocks, pvs, whole)) {
        int status = MSD_OK;
        if (gn_tokens_two_launches<T>(x, y, gamma, beta, batch, channels, hw, groups, eps, partials, stream, &status)) return status;
    }
    if (whole) return in_one();
    GnScratch sc{};
    if (split > 1) {
        const hipError_t err = get_scratch(stream, &sc);
        if (err != hipSuccess) return (int)err;
    }
    const uint32_t threads = pl.threads;
    switch (pl.k) {
        case 1: gn_tokens_launch<T, 1>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 2: gn_tokens_launch<T, 2>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 3: gn_tokens_launch<T, 3>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 4: gn_tokens_launch<T, 4>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 5: gn_tokens_launch<T, 5>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 6: gn_tokens_launch<T, 6>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 8: gn_tokens_launch<T, 8>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        case 10: gn_tokens_launch<T, 10>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos); break;
        default:  // (12, 16: 2-byte elements only, see kMaxK)
            if constexpr (sizeof(T) == 2) {
                if (pl.k == 12)
                    gn_tokens_launch<T, 12>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos);
                else
                    gn_tokens_launch<T, 16>(blocks, threads, lds_bytes, stream, x, y, gamma, beta, sc, q, (uint32_t)groups, (uint32_t)hw_vec, pos_vecs, combos);
            }
    }
    return launch_status();
}

template int gn_tokens_dispatch<float>(const void *, void *, const float *, const float *, size_t, size_t,
                                       size_t, size_t, float, float2 *, hipStream_t);
template int gn_tokens_dispatch<__half>(const void *, void *, const float *, const float *, size_t, size_t,
                                        size_t, size_t, float, float2 *, hipStream_t);

}  // namespace msd
