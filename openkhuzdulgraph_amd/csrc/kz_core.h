// Core bitmap of a forward graph: the adjacency of its `size` highest ids as
// bit rows in HBM, so that the rows a clique root needs among those ids are
// gathered bit by bit instead of streaming and hashing whole lists.
//
// After degree orientation the lists concentrate on the highest ids: on
// RMAT-22 (edge factor 16) the top 32 K of 2.4 M ids hold 79 % of the list
// entries and 88 % of the candidate pairs (i, j) of all roots, and a root has
// fewer pairs (7.2 G in all) than its candidates' lists have entries (28.9 G,
// of which 10.9 G were streamed and 1.2 G candidates searched without the
// core).  A row of a root is one load per 64 candidates: lane j reads the word
// that holds its candidate's bit, a compare puts the row's 64-bit word in a
// scalar pair.  That is about 6 VALU instructions per 64 pairs against 25 per
// streamed id, no hash and no LDS atomics, and the lanes share cache lines
// because the candidates are sorted.  RMAT-24 4-cliques 180.2 -> 76.4 ms a
// count (roots of 512-1024 candidates 52.0 -> 13.6, 128-512 71.1 -> 30.2, hub
// rows 17.5 -> 7.7, wave bucket 22.5 -> 12.2).  The 128-512 bucket is now
// bound by lines: 1.8 G of them in 30 ms, 7.6 TB/s with 6 % L2 hits.
//
// Layout: core vertices are numbered downwards, r(x) = n - 1 - x, so forward
// neighbours have smaller numbers: row r holds bits [0, r) in 128-byte lines,
// rows one after another (core_line).  The hottest columns, the highest ids,
// share each row's first lines.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kz_kernels.h"

namespace kz {

constexpr uint32_t kCoreMax = 1u << 20;  // a row under construction fits LDS (128 KB)

// 128-byte lines before row r.
__host__ __device__ inline uint32_t core_line(uint32_t r) {
    const uint32_t t = r ? r - 1 : 0u, q = t >> 10;
    return ((q * (q + 1)) << 9) + (t & 1023u) * (q + 1);
}
// Bytes of a core of `size` rows.  Lanes whose candidate is not above the
// row's vertex may read past a row's end (their bit is masked): up to
// size / 8 bytes past the last row.
inline uint64_t core_alloc_bytes(uint32_t size) {
    return 128ull * core_line(size) + (uint64_t(size) / 8 + 256) / 128 * 128;
}

// Number of a core vertex, held inside the core for ids below it.
__device__ __forceinline__ uint32_t core_num(uint32_t x, uint32_t n1, uint32_t size) {
    const uint32_t r = n1 - x;
    return r < size ? r : size - 1;
}

// The word at byte `off` of the row starting at `line`.
__device__ __forceinline__ uint32_t core_word(const uint32_t* bm, uint32_t line, uint32_t off) {
    const char* row = reinterpret_cast<const char*>(bm) + (uint64_t(line) << 7);
    return *(const KZ_GLOBAL_AS uint32_t*)(row + off);
}
// The same for a wave-uniform line: the row's address stays scalar (hidden
// from the compiler, which would otherwise add 64-bit row offsets to a vector
// address for every load).
__device__ __forceinline__ uint32_t core_word_uniform(const uint32_t* bm, uint32_t line, uint32_t off) {
    uint64_t row = reinterpret_cast<uint64_t>(bm) + (uint64_t(line) << 7);
    asm("" : "+s"(row));
    return *(const KZ_GLOBAL_AS uint32_t*)(reinterpret_cast<const KZ_GLOBAL_AS char*>(row) + off);
}

// old with lane l's value replaced by v (l, v wave-uniform): v_writelane_b32,
// which has no builtin of its own.
__device__ uint32_t lane_write(uint32_t v, uint32_t l, uint32_t old) __asm("llvm.amdgcn.writelane.i32");

// Rows [i0, i0 + 32) x candidates [64 kk, 64 kk + 64) of a root's DAG from
// the core: calls put(i, word) on lane i - i0 for each row i in [lo, d) with
// word kk of row i (bits j > i only).  at(i) is the root's i-th list entry
// (ids from index lo on are in the core).  Row addresses are scalar, the
// lane's offset the same for every row, 16 gathers in flight.  Wave-wide.
template <class At, class Put>
__device__ __forceinline__ void core_tile(const uint32_t* bm, uint32_t n1, uint32_t size, uint32_t d, uint32_t lo,
                                          uint32_t i0, uint32_t kk, At&& at, Put&& put) {
    constexpr int kBatch = 16;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t j = 64 * kk + lane;
    const uint32_t xr = core_num(at(j < d ? j : d - 1), n1, size);
    const uint32_t off = (xr >> 5) << 2, bit = 1u << (xr & 31u);
    const uint32_t i = i0 + (lane & 31u);
    const uint32_t ic = i < lo ? lo : i < d ? i : d - 1;
    const uint32_t line = core_line(core_num(at(ic), n1, size));
    uint32_t wl = 0, wh = 0;
    auto rows = [&](auto diag) {
#pragma unroll
        for (int b = 0; b < 32; b += kBatch) {
            uint32_t v[kBatch];
#pragma unroll
            for (int r = 0; r < kBatch; ++r) {
                uint32_t o = off;
                // lanes not above the row read its first word, not a cold line
                if constexpr (decltype(diag)::value) o = j > i0 + uint32_t(b + r) ? off : 0u;
                v[r] = core_word_uniform(bm, wave_lane(line, uint32_t(b + r)), o);
            }
#pragma unroll
            for (int r = 0; r < kBatch; ++r) {
                const unsigned long long m = __builtin_amdgcn_ballot_w64((v[r] & bit) != 0u);
                wl = lane_write(uint32_t(m), uint32_t(b + r), wl);
                wh = lane_write(uint32_t(m >> 32), uint32_t(b + r), wh);
            }
        }
    };
    if (64 * kk < i0 + 32) rows(std::true_type{});
    else rows(std::false_type{});
    unsigned long long w = (static_cast<unsigned long long>(wh) << 32) | wl;
    if (i >= 64 * kk) w &= i - 64 * kk >= 63 ? 0ull : ~0ull << (i - 64 * kk + 1);
    if (d - 64 * kk < 64) w &= (1ull << (d - 64 * kk)) - 1;
    if (lane < 32 && i >= lo && i < d) put(i, w);
}

// Core rows of a short root, c <= 64 / S core candidates at list indices k0
// .. k0 + c - 1 (lane l holds the core number `xr` and row line of list entry
// l): S rows share a load, 64 / S lanes each, so a root of 8 candidates takes
// one load.  Returns lane l's row word (bit j: list index j; 0 below k0).
template <int S>
__device__ __forceinline__ unsigned long long core_rows_short(const uint32_t* bm, uint32_t xr, uint32_t line,
                                                              uint32_t k0, uint32_t c) {
    constexpr uint32_t W = 64 / S;
    constexpr uint32_t Q = W / S;  // loads for W rows
    constexpr uint32_t B = Q < 4 ? Q : 4;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t seg = lane / W, cj = lane % W;
    const uint32_t xj = __shfl(xr, int((k0 + cj) & 63u));
    const uint32_t off = (xj >> 5) << 2, bit = 1u << (xj & 31u);
    const uint32_t mine = lane - k0;  // this lane's row, for lane >= k0
    unsigned long long w = 0;
    for (uint32_t q0 = 0; q0 * S + 1 < c; q0 += B) {
        uint32_t v[B];
        bool use[B];
#pragma unroll
        for (uint32_t q = 0; q < B; ++q) {
            const uint32_t ri = (q0 + q) * S + seg;
            use[q] = (cj > ri) & (cj < c);
            const uint32_t ln = __shfl(line, int((k0 + (ri < c ? ri : c - 1)) & 63u));
            v[q] = core_word(bm, ln, use[q] ? off : 0u);
        }
#pragma unroll
        for (uint32_t q = 0; q < B; ++q) {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(use[q] & ((v[q] & bit) != 0u));
            if (lane >= k0 && mine / S == q0 + q) w = ((m >> (W * (mine % S))) & ((1ull << W) - 1)) << k0;
        }
    }
    return w;
}

// Index of the first list entry in the core (entries >= base), d if none.
// L in LDS; wave-uniform.
__device__ __forceinline__ uint32_t core_first(const uint32_t* L, uint32_t d, uint32_t base) {
    const uint32_t lane = threadIdx.x & 63;
    uint32_t lo = 0, hi = d;  // the answer is in [lo, hi]
    while (hi > lo) {
        const uint32_t step = (hi - lo + 63) >> 6;
        const uint32_t i = lo + lane * step;
        const uint32_t c = uint32_t(__popcll(__ballot(i < hi && L[i < hi ? i : hi - 1] < base)));
        if (c == 0) return lo;
        lo += (c - 1) * step + 1;
        hi = hi < lo + step - 1 ? hi : lo + step - 1;
    }
    return lo;
}

}  // namespace kz
