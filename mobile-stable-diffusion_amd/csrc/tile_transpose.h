// [j, k] -> [k, j] of one 64 x 64-element tile by a workgroup of 256 lanes: the body of the stand-alone
// permute and of the token-major GroupNorm's second launch.
//
// Both global sides use 16-byte accesses; the LDS tile of 32-bit words is written transposed: word w
// of tile row k belongs to output row k (one 4-byte element, or the 2-byte elements of input rows 2w
// and 2w + 1 at column k, paired in registers after the load).  Inside a tile row the aligned groups
// of four words are permuted by an XOR with a number taken from the row index, chosen so that the 32
// lanes of a half wavefront, which write one column each (8 rows a fixed distance apart x 4 adjacent
// words), fall on 32 different banks, while a lane's four output words stay adjacent and aligned: the
// read side is one 16-byte LDS access per piece, and the eight lanes that read one tile row together
// take eight different groups.
#pragma once

#include "msd_device.h"

namespace msd {

constexpr int kTile = 64;
constexpr size_t kCacheLine = 128;
constexpr int kTileThreads = 256;
// Most positions along a side: a grid holds less than 2^32 lanes in a dimension.
constexpr size_t kTileMaxSide = 0xFFFFFFFFull / kTileThreads * kTile;

// LDS of a tile, in 16-byte words.
template <int ES>
constexpr uint32_t tile_lds_words() {
    return kTile * (kTile * ES / 4) / 4;
}

// 2, 4, 8 or 16 bytes at any element boundary: the memory pipeline takes such accesses as they are.
template <typename W>
__device__ __forceinline__ W load_any(const char *at) {
    W w;
    __builtin_memcpy(&w, at, sizeof(W));
    return w;
}
template <typename W>
__device__ __forceinline__ void store_any(char *at, W w) {
    __builtin_memcpy(at, &w, sizeof(W));
}

// The piece (16 / ES elements) at `at` of a row with `left` elements from there on; what lies past the
// row's end is not read.  RAGGED: pieces may start at any element and may be cut by the row's end.
// KEEP: the lines stay in the caches, for the pieces beside this one.
template <int ES, bool RAGGED, bool KEEP = false>
__device__ __forceinline__ u32x4 tile_load(const char *at, uint32_t left) {
    if constexpr (!RAGGED && KEEP) return *reinterpret_cast<const u32x4 *>(at);
    if constexpr (!RAGGED) return load_stream(reinterpret_cast<const u32x4 *>(at));
    if (left >= 16 / ES) return load_any<u32x4>(at);
    uint32_t w0 = 0, w1 = 0, w2 = 0, w3 = 0;
    const uint32_t bytes = left * ES;  // 2 ... 14
    if (bytes & 8) {
        w0 = load_any<uint32_t>(at);
        w1 = load_any<uint32_t>(at + 4);
    }
    if (bytes & 4) {
        const uint32_t w = load_any<uint32_t>(at + (bytes & 8));
        w0 = bytes & 8 ? w0 : w;
        w2 = w;
    }
    if (ES == 2 && (bytes & 2)) {
        const uint32_t w = load_any<uint16_t>(at + (bytes & 12)), word = bytes >> 2;
        w0 = word == 0 ? w : w0;
        w1 = word == 1 ? w : w1;
        w2 = word == 2 ? w : w2;
        w3 = w;
    }
    return u32x4{w0, w1, w2, w3};
}
template <int ES, bool RAGGED>
__device__ __forceinline__ void tile_store(char *at, uint32_t left, const u32x4 &v) {
    if constexpr (!RAGGED) {
        store_stream(reinterpret_cast<u32x4 *>(at), v);
        return;
    }
    if (left >= 16 / ES) {
        store_any<u32x4>(at, v);
        return;
    }
    const uint32_t bytes = left * ES;
    if (bytes & 8) {
        store_any<uint32_t>(at, v[0]);
        store_any<uint32_t>(at + 4, v[1]);
    }
    if (bytes & 4) store_any<uint32_t>(at + (bytes & 8), bytes & 8 ? v[2] : v[0]);
    if (ES == 2 && (bytes & 2)) {
        const uint32_t word = bytes >> 2;
        store_any<uint16_t>(at + (bytes & 12), (uint16_t)(word == 0 ? v[0] : word == 1 ? v[1] : word == 2 ? v[2] : v[3]));
    }
}

// in: the [jsize, ksize] plane, out: the [ksize, jsize] plane, ES bytes per element; the tile starts at
// (j0, k0).  Without RAGGED jsize and ksize are multiples of 16 / ES and both planes are 16-byte
// aligned (a piece is all inside the tensor or all outside).  ready() runs between the loads and their
// first use, by every lane (KEEP: see tile_load); map(row, piece) returns the piece of tile row `row` (channel j0 + row) as
// it is to be stored.
template <int ES, bool RAGGED, bool KEEP = false, typename Ready, typename Map>
__device__ __forceinline__ void transpose_tile(const char *in, char *out, uint32_t jsize, uint32_t ksize, uint32_t j0,
                                               uint32_t k0, u32x4 *tile4, Ready ready, Map map) {
    constexpr uint32_t kWords = kTile * ES / 4;      // 32-bit words per output row of the tile: 32 or 64
    constexpr uint32_t kRowShift = ES == 4 ? 2 : 3;  // tile rows one lane writes: 4 or 8
    uint32_t *tile = reinterpret_cast<uint32_t *>(tile4);
    // word `col` of tile row `row` lives at this index
    auto at = [](uint32_t row, uint32_t col) { return row * kWords + (col ^ (((row >> kRowShift) & 7u) << 2)); };
    const uint32_t t = threadIdx.x;
    if constexpr (ES == 4) {
        // a lane loads elements k .. k+3 of one input row, four times: 8 lanes cover 32 columns,
        // the passes take the two column halves of the tile and the two halves of its rows.  All
        // loads leave before the first LDS write (a piece outside the tensor re-reads the plane's
        // first piece instead of sitting behind a branch).
        const uint32_t kq = (t & 7) * 4, jr = t >> 3;
        u32x4 v[4];
#pragma unroll
        for (int pass = 0; pass < 4; pass++) {
            const uint32_t k = k0 + kq + 32 * (pass & 1), j = j0 + jr + 32 * (pass >> 1);
            const bool inside = j < jsize && k < ksize;
            const size_t from = inside ? ((size_t)j * ksize + k) * 4 : 0;
            v[pass] = tile_load<ES, RAGGED, KEEP>(in + from, inside ? ksize - k : 0);
        }
        ready();
#pragma unroll
        for (int pass = 0; pass < 4; pass++) {
            const uint32_t kl = kq + 32 * (pass & 1), jl = jr + 32 * (pass >> 1);
            if (j0 + jl < jsize && k0 + kl < ksize) {
                const u32x4 w = map(jl, v[pass]);
#pragma unroll
                for (int e = 0; e < 4; e++) tile[at(kl + e, jl)] = w[e];
            }
        }
    } else {
        // a lane loads elements k .. k+7 of input rows j and j+1 and pairs them by column
        const uint32_t kq = (t & 7) * 8, jw = t >> 3;  // jw: word of the output rows, 0 .. 31
        const uint32_t j = j0 + 2 * jw, k = k0 + kq;
        const bool inside = j < jsize && k < ksize;
        u32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
        if (inside) {
            a = tile_load<ES, RAGGED, KEEP>(in + ((size_t)j * ksize + k) * 2, ksize - k);
            // (without RAGGED jsize is even; an odd one's last row pairs with itself)
            const uint32_t second = RAGGED ? min(j + 1, jsize - 1) : j + 1;
            b = tile_load<ES, RAGGED, KEEP>(in + ((size_t)second * ksize + k) * 2, ksize - k);
        }
        ready();
        if (inside) {
            const u32x4 pa = map(2 * jw, a), pb = map(2 * jw + 1, b);
#pragma unroll
            for (int w = 0; w < 4; w++) {
                tile[at(kq + 2 * w, jw)] = (pa[w] & 0xffffu) | (pb[w] << 16);
                tile[at(kq + 2 * w + 1, jw)] = (pa[w] >> 16) | (pb[w] & 0xffff0000u);
            }
        }
    }
    __syncthreads();
    // a lane stores 16-byte pieces (four words) of output rows; all LDS reads come first
    constexpr uint32_t kPieces = kWords / 4;                   // pieces per output row of the tile: 8 or 16
    constexpr uint32_t kRowsPerPass = kTileThreads / kPieces;  // 32 or 16
    constexpr uint32_t kPasses = kTile / kRowsPerPass;
    const uint32_t wq = (t % kPieces) * 4, kr = t / kPieces;
    u32x4 w[kPasses];
#pragma unroll
    for (uint32_t pass = 0; pass < kPasses; pass++)  // (pieces outside the tensor are read but never stored)
        w[pass] = tile4[at(kr + pass * kRowsPerPass, wq) / 4];
#pragma unroll
    for (uint32_t pass = 0; pass < kPasses; pass++) {
        const uint32_t k = k0 + kr + pass * kRowsPerPass, j = j0 + wq * (4 / ES);
        if (k < ksize && j < jsize) tile_store<ES, RAGGED>(out + ((size_t)k * jsize + j) * ES, jsize - j, w[pass]);
    }
}

}  // namespace msd
