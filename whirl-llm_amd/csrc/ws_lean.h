// The lean single-sweep sampler for gfx950: one workgroup of 1024 threads (sixteen wave64s, four per SIMD) per row,
// for batches with at least one row per compute unit. It answers the rows most requests are made of - fp32
// logits of any length and address, a closed filter without a top-k (top-p and / or min-p), the inverse-CDF draw - and
// hands every other row (and every row on which one of its own checks fails) to the three-pass code of ws_sample.h
// inside the same launch. Results are those of ws_sample.h's single-sweep kernel: the same bins, the same histogram
// words, the same decision rules (src/sampling/sampler.cpp:15-78, :118-131) and margins.
//
// What is different from that kernel, and why:
//   * every token's bin is remembered as eight of its bits, four tokens per register (of 163840 tokens 40 registers instead of 160): a
//     scan for the tokens of a few bins tests four tokens with three instructions per bin; a token of another bin with
//     the same bits is found as well and dropped when its logit has been read again. The registers this frees let the
//     first two batches of the row travel while phase 0 builds its tables, and four waves per SIMD hide the tail's
//     latencies.
//   * the histogram is scanned four consecutive bins per thread, the cuts' and the draw's bins are found by all threads
//     at once (every thread tests the bins it has just scanned), and one wave works out what follows from the answers.
//   * the candidates - the tokens of those bins, 4096 a row at most - are put in their exact order (logit descending,
//     id ascending) by a bucket sort of their 64-bit keys whose buckets follow the keys that are there, thousands of
//     equal logits included; a block-wide scan of their masses in that order settles the cuts and the draw.
// Rows that end inside a vector, or begin off one, go the same way: their vectors are read where they lie (row_vector, part_vector), at no cost to the
// others (256 aligned rows of 151936 47.5 us before and 46.9 after: fewer scalar registers spilled). What three sweeps took of them: see plan_batch.
#pragma once
#include <type_traits>

#include "ws_sample.h"

#ifndef WS_LEAN_EARLY
#define WS_LEAN_EARLY 4  // batches binned before the history ids are looked at
#endif

namespace ws {

// Registers of the bin cache a thread, four tokens each: builds for rows of up to 32768, 49152, 65536, 98304, 155648, 163840 and 262144
// tokens, and a row gets the shortest that holds it. The loads past a row's end are asked for like the others - they may not lie behind a branch -, 64
// lanes at one address each: a row of 25000 tokens waited 8 K clocks of 46 K for them in the build of 40 (us, that one and its own: 54 rows of 25792 20.1 / 17.3, 34 of
// 35392 24.3 / 20.5, 256 of 32000 with 1000 ids 26.5 / 21.6, 200 of 50257 27.9 / 24.3, 100 of 98304 30.9 / 29.0). The longest, of whose 128 registers the cache and a scan's finds are 96,
// spills 71 (masked 73), still far from the two more sweeps that such rows took (ws_abi.hip); the masked one of 8, whose batches are all early ones, spills 17.
// The classes of the longer rows lie closer together than what a launch varies by (256 rows, the build of 38 and the next one: of 151936 40.5 / 41.1, of 140000 level; against one of 32, which
// there is not: of 98312 31.8 / 30.7, of 120000 34.6 / 33.6, of 131072 38.7 / 36.0, masked 38.0 / 40.6).
constexpr int kLeanRegs[] = {8, 12, 16, 24, 38, 40, 64};
constexpr int kLeanLooks = 64;  // from here on finds are looked at before they are listed, when they are too many
constexpr int kLeanBatch = 2;   // 128-bit loads per thread and batch
constexpr uint32_t kLeanBuckets = 128u;   // words of the finish's tables in LeanShared
constexpr uint32_t kLeanMaxList = 4096u;  // candidates of a row's ranges together: what the sort's 32 KiB hold
// The bins the cut and the draw can fall in: as many as have eight different cache bytes, sixteen at most.
constexpr uint32_t kLeanMaxBins = 16u;
// A token's coordinate is measured from where ws_sample.h measures it, an anchor this many units of the exponent above the largest of the row's first tokens;
// the bins begin kLeanRoom of them, four units, above the anchor, where coordinates are below zero. The room is for peaked rows: with logits of sigma 4 at T = 0.5
// the maximum of 151936 tokens lies 4.8 units above that of the first 8192 on average, and more than 8 on a quarter of the rows. (Measured from
// the first bin, tokens four to eight units below the head's largest have a bit less of their coordinate in 32 bits, and the mass that is taken from it has too. Rms error
// of a normaliser against 64 bits, in 1e-8, from the first bin / from the anchor / ws_sample.h: 50257 tokens of N(0, 3) at T = 0.6 14.3 / 9.4 / 9.4,
// 151937 of raised tokens 8.5 / 4.9 / 4.9, Zipfian 7.4 / 5.4 / 5.4; the sweep takes the same instructions either way.)
constexpr float kLeanAbove = 8.f;
constexpr int kLeanRoom = 256;
// A row whose maximum lies above the first bin is swept once more, from its maximum down (lean_rest): a second sweep where three would be made. Up to
// this far above the anchor, that is: a maximum further up is a lone token with next to no mass below it, and such a row is handed back. (us, handed back / swept once more: ten rows
// of 256 of 151937 with sigma / T = 8 95 / 67, 86 of 256 of raised tokens at T = 0.6 100 / 62, 18 of 256 of 50257 54 / 42. More room for the bins instead would take
// masses from coordinates of up to 1024, at a fourth of their precision.)
constexpr int kLeanFar = 1536;
// A range may span this many bins when few of them hold a token (the draw's range on a peaked row: two tokens fifty
// bins apart); its bins then share the range's eight slots of the sort in order, several to a slot.
constexpr uint32_t kLeanWide = 1024u;
// The first bin of this kernel's tail, 48 units of the exponent below the first bin: the last 1024 bins, one to a thread,
// take the tokens below that and the masked-out ones. (A scan of the bin cache for a bin finds the tokens of the tail
// bins with the same cached bits as well: spread over 1024 bins, a 256th of the tail's tokens at most. In 64 bins a
// row with nine tokens in ten masked out had up to a sixteenth of them found with every bin it asked for.)
constexpr int kLeanTail = 3072;

// A token's height, bin_coord's coordinate with its sign turned round: what is above the anchor is above zero. What lies beyond the bins is put at their ends,
// NaN at `low`, a negative number (of three values with a NaN among them the instruction takes the smallest).
__device__ __forceinline__ float lean_height(float aq, float c64, float x, float low) {
    return __builtin_amdgcn_fmed3f(__fmaf_rn(x, c64, -aq), low, static_cast<float>(kLeanRoom));
}
// its bin, counted from the anchor's: -kLeanRoom is the first (a floor and a conversion would be two instructions)
__device__ __forceinline__ int lean_bin(float height) {
    int b;
    asm("v_cvt_flr_i32_f32 %0, -%1" : "=v"(b) : "v"(height));
    return b;
}
// the same, and the histogram's word; at_anchor: the anchor's. (In one block: behind a written-out instruction the compiler puts a pause before the next that
// reads its result.)
typedef __attribute__((address_space(3))) uint64_t* LeanWord;
__device__ __forceinline__ int lean_bin(float height, LeanWord at_anchor, LeanWord& word) {
    int b;
    asm("v_cvt_flr_i32_f32 %0, -%2\n\tv_lshl_add_u32 %1, %0, 3, %3" : "=&v"(b), "=v"(word) : "v"(height), "v"(at_anchor));
    return b;
}

#ifdef WS_PHASE_TIMERS
#define WSL_FAIL(code)                                                                                   \
    do {                                                                                                 \
        if (threadIdx.x == 0 && A.entropy) A.entropy[row * 32 + 28] = (code) + 100.0 * sel_dbg(S);       \
        if (threadIdx.x == 0) S.top = __uint_as_float(0x7fc00000u);                                      \
        return false;                                                                                    \
    } while (0)
#define WSL_MARK(k)                                                \
    do {                                                           \
        if (threadIdx.x == 0) S.marks[(k)] = clock64() - wsl_t0;   \
    } while (0)
#else
#define WSL_FAIL(code)                                                 \
    do {                                                               \
        if (threadIdx.x == 0u) S.top = __uint_as_float(0x7fc00000u);   \
        return false;                                                  \
    } while (0)
#define WSL_MARK(k) \
    do {            \
    } while (0)
#endif

// The cached bytes of masked-out tokens. All of a thread's lie in one bin of the tail, and where that bin's byte was one of those asked for, four threads found
// every masked-out token they had, one after the other: 20 us of a row of 151936 with five tokens in six masked out. So each of a thread's tokens
// gets a byte of its own (register c, token e): what is asked for finds no more of them than of any other tokens, and they are dropped like those.
constexpr uint32_t lean_other_byte(int c) {
    uint32_t k = 0;
    for (int e = 0; e < 4; ++e) k |= ((static_cast<uint32_t>(c) * 4u + static_cast<uint32_t>(e)) * 101u & 0xffu) << (8 * e);
    return k;
}
// all ones in byte e where bit e of `out` is set
__device__ __forceinline__ uint32_t masked_bytes(int32_t out) {
    const uint32_t m0 = static_cast<uint32_t>((out << 31) >> 31), m1 = static_cast<uint32_t>((out << 30) >> 31), m2 = static_cast<uint32_t>((out << 29) >> 31),
                   m3 = static_cast<uint32_t>((out << 28) >> 31);
    return __builtin_amdgcn_perm(m3, m2, 0x04000c0cu) | __builtin_amdgcn_perm(m1, m0, 0x0c0c0400u);
}

// bit 7 of every byte of y that equals the byte c4 repeats (and, possibly, of a byte above such a byte: a token found that
// way is dropped when its logit has been read again)
__device__ __forceinline__ uint32_t bytes_equal(uint32_t y, uint32_t c4) {
    const uint32_t x = y ^ c4;
    return (x - 0x01010101u) & ~x;
}

template <int NT>
__device__ __forceinline__ uint32_t lean_flags(uint32_t y, const uint32_t (&c4)[4]) {
    uint32_t f = bytes_equal(y, c4[0]);
    if (NT > 1) f |= bytes_equal(y, c4[1]);
    if (NT > 2) f |= bytes_equal(y, c4[2]);
    if (NT > 3) f |= bytes_equal(y, c4[3]);
    return f;
}

// What a thread's scan of its bin cache found: per group of 8 registers (32 tokens) the first two tokens whose cached byte
// equals one of the bytes asked for, with their logits requested right there (the loads travel while the scan goes on).
template <int NREG>
struct LeanHits {
    static constexpr int kGroups = (NREG + 7) / 8;  // (the last may have fewer than eight registers)
    uint32_t idx[2 * kGroups];   // token index, 0xffffffff = none
    uint32_t bits[2 * kGroups];  // its logit as loaded
};

// A third token of a group and beyond goes to list[] as (token | kListNeedsLoad, 0), one LDS atomic each (rare). With
// TO_LIST every find goes there (a second round of bytes). V: the row's tokens.
// wanted(logit bits): only such a find goes to the list, with its logit (nullptr: as above).
template <int NT, bool TO_LIST, int NREG, class WANTED = std::nullptr_t>
__device__ __forceinline__ void lean_scan(const uint32_t (&cache)[NREG], const uint32_t (&c4)[4], const void* __restrict__ xg, LeanHits<NREG>& H,
                                          uint2* list, uint32_t* n_list, uint32_t cap, uint32_t V, WANTED&& wanted = nullptr) {
    constexpr bool LOOK = !std::is_same_v<std::decay_t<WANTED>, std::nullptr_t>;
    constexpr int kGroups = LeanHits<NREG>::kGroups;
    const uint32_t t = threadIdx.x, nv = V >> 2;  // (whole vectors; of the one that the row may end in only the row's tokens are looked at)
    auto logit_bits = [&](uint32_t i) {
        return static_cast<const uint32_t*>(xg)[i];
    };
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        // where the row ends is looked at per group, uniformly: a group past the row is skipped, the one group the end
        // falls in masks its finds, the others need no test
        uint32_t acc = 0;
        const uint32_t g_lo = static_cast<uint32_t>(g * 8) * WS_BLOCK;
        if (g_lo + 8u * WS_BLOCK <= nv) {
#pragma unroll
            for (int r = 0; r < 8 && g * 8 + r < NREG; ++r)  // bit 8 e + r: token e of register r
                acc = ((lean_flags<NT>(cache[g * 8 + r], c4) >> (7 - r)) & (0x01010101u << r)) | acc;
        } else if (g_lo * 4u < V) {
#pragma unroll
            for (int r = 0; r < 8 && g * 8 + r < NREG; ++r) {
                const uint32_t j = g_lo + static_cast<uint32_t>(r) * WS_BLOCK + t;
                const uint32_t keep = (j < nv ? 0x01010101u : (j == nv ? 0x00010101u >> (8u * (3u - (V & 3u))) : 0u)) << r;
                acc = ((lean_flags<NT>(cache[g * 8 + r], c4) >> (7 - r)) & keep) | acc;
            }
        }
        auto token_of = [&](uint32_t bit) {
            const uint32_t reg = static_cast<uint32_t>(g * 8) + (bit & 7u);
            return ((reg * WS_BLOCK + t) << 2) + (bit >> 3);
        };
        if (!TO_LIST) {
            H.idx[g] = H.idx[kGroups + g] = 0xffffffffu;
            H.bits[g] = H.bits[kGroups + g] = 0u;
            if (acc) {
                const uint32_t i = token_of(static_cast<uint32_t>(__ffs(acc)) - 1u);
                acc &= acc - 1u;
                H.idx[g] = i;
                H.bits[g] = logit_bits(i);
            }
            if (acc) {
                const uint32_t i = token_of(static_cast<uint32_t>(__ffs(acc)) - 1u);
                acc &= acc - 1u;
                H.idx[kGroups + g] = i;
                H.bits[kGroups + g] = logit_bits(i);
            }
        }
        while (acc) {
            const uint32_t i = token_of(static_cast<uint32_t>(__ffs(acc)) - 1u);
            acc &= acc - 1u;
            uint32_t bits = 0u;
            if constexpr (LOOK) {
                bits = logit_bits(i);
                if (!wanted(bits)) continue;
            }
            const uint32_t slot = atomicAdd(n_list, 1u);
            if (slot < cap) list[slot] = make_uint2(LOOK ? i : i | kListNeedsLoad, bits);
        }
    }
}

// exp(-a) for 0 <= a < 63 from the tables exp(-b / 64) (s_exp: kExpHi, then kExpLo) and a polynomial on the remaining
// [0, 1/64): a few units in the last place, a fifth of the instructions of the library's exp
__device__ __forceinline__ double exp_neg(double a, const double* s_exp) {
    const double t64 = a * 64.0;
    if (!(t64 >= 0.0 && t64 < 4032.0)) return exp(-a);
    const uint32_t n = static_cast<uint32_t>(t64);
    const double r = a - static_cast<double>(n) * (1.0 / 64.0);
    double p = 1.0 / 720.0;
    p = fma(p, -r, 1.0 / 120.0);
    p = fma(p, -r, 1.0 / 24.0);
    p = fma(p, -r, 1.0 / 6.0);
    p = fma(p, -r, 0.5);
    p = fma(p, -r, 1.0);
    p = fma(p, -r, 1.0);
    return s_exp[n >> 6] * s_exp[64u + (n & 63u)] * p;
}

// e^-a, of either sign: 2^k e^r with |r| <= ln 2 / 2, the series to r^13 (0.9 units in the last place at most over 2e7 arguments; a quarter of the library's instructions).
// The reduction is Cody and Waite's, with ln 2 in the two parts that Sun's public fdlibm (e_exp.c) gives it.
__device__ __forceinline__ double code_exp(double a) {
    const double k = __builtin_rint(a * -1.44269504088896340736);
    double r = fma(k, -6.93147180369123816490e-01, -a);
    r = fma(k, -1.90821492927058770002e-10, r);
    double p = 1.0 / 6227020800.0;
    p = fma(p, r, 1.0 / 479001600.0);
    p = fma(p, r, 1.0 / 39916800.0);
    p = fma(p, r, 1.0 / 3628800.0);
    p = fma(p, r, 1.0 / 362880.0);
    p = fma(p, r, 1.0 / 40320.0);
    p = fma(p, r, 1.0 / 5040.0);
    p = fma(p, r, 1.0 / 720.0);
    p = fma(p, r, 1.0 / 120.0);
    p = fma(p, r, 1.0 / 24.0);
    p = fma(p, r, 1.0 / 6.0);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return __builtin_amdgcn_ldexp(p, static_cast<int>(k));
}
// the same of any a that is not below zero (2^30 e-folds and more would not fit the exponent's integer). NaN, which an infinite inverse temperature makes of
// the maximum's own distance, counts as no mass: such a row's probability is 0 / 0, NaN all the same
__device__ __forceinline__ double exp_down(double a) { return code_exp(fmin(a, 1e6)); }

// One of four values by number. The values come in as arguments, every one of them read before the choice: a chain
// of conditional reads of an array's elements is turned into one read at a computed index, and the array into memory.
template <typename T>
__device__ __forceinline__ T pick4(uint32_t k, T a0, T a1, T a2, T a3) {
    const T lo = k & 1u ? a1 : a0, hi = k & 1u ? a3 : a2;
    return k & 2u ? hi : lo;
}

// Sorts the n (<= kShortCap) different 64-bit keys keys[0 .. n) in LDS into descending order. bucket_of(key) in [0, nb)
// (nb: 64 or 512; bcnt, bstart: nb words of LDS each, 16-byte aligned) must not rise along that order (equal for keys it cannot tell apart): a key's place is the start of its bucket plus
// the number of larger keys among the bucket's members, which it reads after all keys have been laid out bucket by
// bucket - a few dozen reads a key where a full comparison sort takes dozens of barriers. Every thread calls it.
template <class B>
__device__ __forceinline__ void bucket_sort_desc(uint64_t* keys, uint32_t n, uint32_t* bcnt, uint32_t* bstart, uint32_t nb, B&& bucket_of) {
    constexpr uint32_t K = kShortCap / WS_BLOCK;
    const uint32_t t = threadIdx.x;
    uint64_t key[K];
    uint32_t bk[K], pos[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n) key[k] = k * WS_BLOCK + t < n ? keys[k * WS_BLOCK + t] : 0ull;  // (uniform: rounds past the list issue nothing)
    for (uint32_t i = t; i < nb; i += WS_BLOCK) bcnt[i] = 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n && k * WS_BLOCK + t < n) {
            bk[k] = min(nb - 1u, bucket_of(key[k]));
            pos[k] = atomicAdd(&bcnt[bk[k]], 1u);
        }
    __syncthreads();
    if (t < 64u) {  // one wave: one or eight consecutive counts a lane
        if (nb == 64u) {
            const uint32_t c = bcnt[t];
            bstart[t] = wave_incl_scan(c) - c;
        } else {
            const uint4 a = *reinterpret_cast<const uint4*>(&bcnt[t * 8u]), b = *reinterpret_cast<const uint4*>(&bcnt[t * 8u + 4u]);
            const uint32_t sa = a.x + a.y + a.z + a.w, sum = sa + b.x + b.y + b.z + b.w;
            const uint32_t run = wave_incl_scan(sum) - sum, mid = run + sa;
            *reinterpret_cast<uint4*>(&bstart[t * 8u]) = make_uint4(run, run + a.x, run + a.x + a.y, run + a.x + a.y + a.z);
            *reinterpret_cast<uint4*>(&bstart[t * 8u + 4u]) = make_uint4(mid, mid + b.x, mid + b.x + b.y, mid + b.x + b.y + b.z);
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n && k * WS_BLOCK + t < n) keys[bstart[bk[k]] + pos[k]] = key[k];
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n && k * WS_BLOCK + t < n) {
            const uint32_t b0 = bstart[bk[k]], c = bcnt[bk[k]];
            uint32_t above = 0;
            for (uint32_t i = 0; i < c; i += 4u) {  // four reads on their way together
                uint64_t o[4];
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) o[q] = keys[b0 + min(i + q, c - 1u)];
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) above += (i + q < c && o[q] > key[k]) ? 1u : 0u;
            }
            pos[k] = b0 + above;
        }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n && k * WS_BLOCK + t < n) keys[pos[k]] = key[k];
    __syncthreads();
}

// Every one of a row's parameters with one scalar load, all asked for together and waited for once. (Written as plain reads
// they become vector loads, each behind the test of its pointer and each waited for on its own: a dozen trips to memory one
// after the other.) An absent array is read at the kernel's argument segment instead and the value dropped.
// args: the kernel's argument segment.
typedef const __attribute__((address_space(4))) BatchArgs* LeanArgPtr;
__device__ __forceinline__ LeanRowParams load_row_params(const BatchArgs& A, const uint32_t row, const LeanArgPtr args) {
    LeanRowParams P;
    const uint64_t dummy = reinterpret_cast<uint64_t>(args);
    auto at = [&](const void* base, uint64_t byte_off) { return base ? reinterpret_cast<uint64_t>(base) + byte_off : dummy; };
    const uint64_t r4 = static_cast<uint64_t>(row) * 4u, r8 = static_cast<uint64_t>(row) * 8u;
    const uint64_t p_inv_t = at(A.inv_t, r4), p_top_k = at(A.top_k, r4), p_race = at(A.race, r4), p_top_p = at(A.top_p, r8), p_min_p = at(A.min_p, r8);
    // (the history's length: its own array, or else the next row's offset - which an offsets array with lengths beside it need not have)
    const uint64_t p_hoff = at(A.hist ? A.hist_off : nullptr, r4);
    const uint64_t p_hlen = A.hist ? (A.hist_len ? at(A.hist_len, r4) : at(A.hist_off, r4 + 4u)) : dummy;
    const uint64_t p_boff = at(A.bias_ids ? A.bias_off : nullptr, r4), p_seed = at(A.seed, r8), p_step = at(A.step, r8);
    const uint64_t p_rep = at(A.rep, r4), p_pres = at(A.pres, r4), p_freq = at(A.freq, r4);
    uint32_t v_inv_t, v_top_k, v_race, v_hoff, v_hlen, v_rep, v_pres, v_freq;
    uint64_t v_top_p, v_min_p, v_boff, v_seed, v_step;
    asm volatile(
        "s_load_dword %0, %13, 0x0\n\t"
        "s_load_dword %1, %14, 0x0\n\t"
        "s_load_dword %2, %15, 0x0\n\t"
        "s_load_dwordx2 %3, %16, 0x0\n\t"
        "s_load_dwordx2 %4, %17, 0x0\n\t"
        "s_load_dword %5, %18, 0x0\n\t"
        "s_load_dword %6, %19, 0x0\n\t"
        "s_load_dwordx2 %7, %20, 0x0\n\t"
        "s_load_dwordx2 %8, %21, 0x0\n\t"
        "s_load_dwordx2 %9, %22, 0x0\n\t"
        "s_load_dword %10, %23, 0x0\n\t"
        "s_load_dword %11, %24, 0x0\n\t"
        "s_load_dword %12, %25, 0x0\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(v_inv_t), "=&s"(v_top_k), "=&s"(v_race), "=&s"(v_top_p), "=&s"(v_min_p), "=&s"(v_hoff), "=&s"(v_hlen), "=&s"(v_boff),
          "=&s"(v_seed), "=&s"(v_step), "=&s"(v_rep), "=&s"(v_pres), "=&s"(v_freq)
        : "s"(p_inv_t), "s"(p_top_k), "s"(p_race), "s"(p_top_p), "s"(p_min_p), "s"(p_hoff), "s"(p_hlen), "s"(p_boff), "s"(p_seed),
          "s"(p_step), "s"(p_rep), "s"(p_pres), "s"(p_freq)
        : "memory");
    P.inv_t = __uint_as_float(v_inv_t);
    P.top_k = A.top_k ? v_top_k : 0u;
    P.race = A.race != nullptr && v_race != 0u;
    P.top_p = A.top_p ? __longlong_as_double(static_cast<long long>(v_top_p)) : 1.0;
    P.min_p = A.min_p ? __longlong_as_double(static_cast<long long>(v_min_p)) : 0.0;
    P.h0 = A.hist ? v_hoff : 0u;
    P.nh = A.hist ? (A.hist_len ? v_hlen : v_hlen - P.h0) : 0u;
    P.b0 = A.bias_ids ? static_cast<uint32_t>(v_boff) : 0u;
    P.nb = A.bias_ids ? static_cast<uint32_t>(v_boff >> 32) - P.b0 : 0u;
    P.seed = v_seed;
    P.step = v_step;
    P.rep = A.rep ? __uint_as_float(v_rep) : 1.f;
    P.pres = A.pres ? __uint_as_float(v_pres) : 0.f;
    P.freq = A.freq ? __uint_as_float(v_freq) : 0.f;
    return P;
}

__device__ __forceinline__ LeanRowParams load_row_params(const BatchArgs& A, const uint32_t row) {
    return load_row_params(A, row, (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr());
}

// what wave 0 works out from the searches' answers for everybody
struct LeanSel {
    double X, m0base, m1base;
    int r0lo, r0hi, r1lo, r1hi;
    uint32_t c0base, n_r0, c1base, n_r1;
    uint32_t topp_in_list, minp_in_list, ok, n_bytes;
    alignas(16) uint32_t bytes[8];  // the different cache bytes of the ranges' bins (n_bytes of them), each repeated four times
};

// a bin as the select's searches hand it round: mass ranked before it and up to and with it, tokens before it and in it
struct LeanBinRec {
    double mex, min_;
    uint32_t b, cex, c, pad;
};

// the lean path's static LDS, declared once by the kernel
struct LeanShared {
    double s_exp[128];  // kExpHi, kExpLo
    double red_d[WS_WAVES];
    double s_d[10];
    alignas(16) LeanSel sel;
    LeanBinRec rec[4 * WS_WAVES + 2];  // [search][wave], then the two bins named outright
    unsigned long long s_q[6];
    alignas(16) unsigned long long b_mass[kLeanBuckets], b_fpre[kLeanBuckets];  // (read four words at a time, all of these)
    alignas(16) uint32_t b_cnt[kLeanBuckets], b_cpre[kLeanBuckets];
    alignas(16) uint32_t b_mid[4 * kLeanMaxBins];
    uint32_t s_w[16];
    uint32_t red_u[WS_WAVES];
    float red_f[WS_WAVES];
    // what lean_row leaves when it returns false: which way the row goes, its maximum, the tokens its history and bias list touch, its normaliser
    float top, m_left;
    uint32_t touched_left;
    double z_left;
#ifdef WS_PHASE_TIMERS
    long long marks[32];
#endif
};

#ifdef WS_PHASE_TIMERS
__device__ __forceinline__ double sel_dbg(const LeanShared& S) { return S.sel.n_r0 + 1e5 * S.sel.n_r1 + 1e10 * (S.sel.r0hi - S.sel.r0lo + 1) + 1e12 * (S.sel.r1hi - S.sel.r1lo + 1); }
#endif
// One row. Returns false when the row is left to others (nothing has been written for it then): S.top is NaN, and it is the three-pass code's; or infinite, and its cut or its
// draw lies among tokens that the list does not take (the touched tokens' tables are where the exact path looks for them); or the row's maximum, and it is to be swept once
// more from there down (AGAIN; its arguments are at `args`).
template <bool MASKED, bool AGAIN, int NREG>
__device__ __forceinline__ bool lean_row(const BatchArgs& A, const LeanArgPtr args, const uint32_t row, LeanShared& S) {
    constexpr uint32_t kTok = 4u, kTokLog = 2u;  // tokens in a 128-bit vector, which is one register of the bin cache: the low eight bits of each bin
    // (a scan for a bin also finds the tokens of the bins 256 apart, some hundreds each, and drops them afterwards)
#ifdef WS_PHASE_TIMERS
    const long long wsl_t0 = clock64();  // debug builds: the marks go to LDS, and at the end to `entropy`, 16 doubles a row
    if (threadIdx.x < 32) S.marks[threadIdx.x] = 0;
#endif
    extern __shared__ __align__(16) unsigned char lds[];
    float* red_f = S.red_f;
    uint32_t* red_u = S.red_u;
    double* red_d = S.red_d;
    double* s_exp = S.s_exp;
    uint32_t* s_w = S.s_w;
    unsigned long long* s_q = S.s_q;
    double* s_d = S.s_d;
    uint32_t* b_cnt = S.b_cnt;
    uint32_t* b_cpre = S.b_cpre;
    unsigned long long* b_mass = S.b_mass;
    unsigned long long* b_fpre = S.b_fpre;

    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    const uint32_t V = A.vocab;
    const uint32_t nW = (V + 31u) >> 5;

    RowView rv;
    rv.V = V;
    rv.dtype = 0;
    rv.base = static_cast<const unsigned char*>(A.logits) + static_cast<size_t>(row) * A.row_stride * 4u;
    rv.vec = true;
    rv.allow = MASKED ? A.allow + static_cast<size_t>(row) * A.allow_stride : nullptr;
    rv.touched = nullptr;
    const uint32_t nv = (V + kTok - 1u) >> kTokLog, j_part = V % kTok ? nv - 1u : 0xffffffffu;  // (the vector the row ends inside, if it does)
    const unsigned char* __restrict__ xv = static_cast<const unsigned char*>(rv.base);
    // The row's loads run through a ring of three batches, two in flight while one is consumed (a compute unit holds about
    // that much in flight: a wave that asks for more waits at the request). The first two batches are asked for before
    // anything else - their address needs the kernel's arguments only - and travel while the row's parameters and then
    // the history ids are fetched, two dependent trips to memory; the first kEarly batches are binned before those ids
    // are looked at (what the ids touch there is put right afterwards), so that phase 0 costs its LDS work and no wait.
    constexpr int kRing = 3, kEarly = WS_LEAN_EARLY;
    constexpr int NB = NREG / kLeanBatch;
    uint4 q[kRing][kLeanBatch];
    uint32_t na[kRing][kLeanBatch];
    auto load = [&](int bt, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kLeanBatch; ++u) {
            const uint32_t j = (bt * kLeanBatch + u) * WS_BLOCK + t;
            q[slot][u] = row_vector<0>(xv, j, V);  // (unconditional, clamped to the row: a load behind a branch makes the compiler wait for every load before it)
            na[slot][u] = MASKED ? rv.allow[(min(j, nv - 1u) * kTok) >> 5] : 0xffffffffu;  // (complemented where it is used: nothing waits for the load here)
        }
    };
    load(0, 0);
    load(1, 1);

    uint64_t* hist = reinterpret_cast<uint64_t*>(lds);
    uint4* stage = reinterpret_cast<uint4*>(lds + 32768);
    uint32_t* touched = reinterpret_cast<uint32_t*>(lds + A.lds_ab);
    uint16_t* wprefix = reinterpret_cast<uint16_t*>(lds + A.lds_ab + nW * 4u);
    float* pv = reinterpret_cast<float*>(lds + A.lds_ab + nW * 4u + ((nW * 2u + 15u) & ~15u));
    uint32_t* cnt = reinterpret_cast<uint32_t*>(lds + A.lds_cnt);
    uint32_t* first = cnt + A.patch_cap;
    uint64_t* hist2 = A.lds_tie ? reinterpret_cast<uint64_t*>(lds + A.lds_tie) : nullptr;
    rv.wprefix = wprefix;
    rv.pv = pv;
    for (uint32_t b = t; b < kBins; b += WS_BLOCK) hist[b] = 0ull;
    if (hist2)
        for (uint32_t b = t; b < kBins; b += WS_BLOCK) hist2[b] = 0ull;
    // (phase 0's tables as well, while the first loads travel: their sizes are the launch's, not the row's)
    if (A.hist || A.bias_ids) {  // (a launch without either has no room for them)
        for (uint32_t w = t; w < nW; w += WS_BLOCK) touched[w] = 0u;
        for (uint32_t r = t; r < A.patch_cap; r += WS_BLOCK) {
            cnt[r] = 0u;
            first[r] = 0xffffffffu;
        }
    }

    const LeanRowParams P = load_row_params(A, row, AGAIN ? args : (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr());
    const float inv_t = P.inv_t;
    const uint32_t top_k = P.top_k;
    const bool race = P.race;
    const double top_p = P.top_p, min_p = P.min_p;
    const bool use_top_p = top_p < 1.0, use_min_p = min_p > 0.0;
    double neg_log_min_p = 0.0;  // wave 15 only (for the select, which has no time for a logarithm)
    if (wv == WS_WAVES - 1u && use_min_p) neg_log_min_p = -log(min_p);
    const uint32_t h0 = P.h0, nh = P.nh, b0 = P.b0, nb = P.nb;
    // Rows this code does not take: a top-k, no filter at all, the race draw, parameters the three-pass code reports; and more than 2047 bias entries, which a row may have -
    // only history and bias list together are bounded by the launch's tables - and which the eleven bits below a claim's do not count. (As a condition of its own that
    // one made the masked build of 38 registers spill 17, 3 to 8 % of its rows' time.)
    if ((top_k | (nb >> 11)) != 0u || !(use_top_p || use_min_p) || race || !(inv_t > 0.f) || nh + nb > A.patch_cap) WSL_FAIL(1);

    const int32_t* hist_ids = A.hist + h0;
    const int32_t* bias_ids = A.bias_ids + b0;
    const float* bias_vals = A.bias_vals + b0;
    constexpr int kHid = 4;
    uint32_t hid[kHid];
#pragma unroll
    for (int k = 0; k < kHid; ++k) hid[k] = t + k * WS_BLOCK < nh ? static_cast<uint32_t>(hist_ids[t + k * WS_BLOCK]) : 0xffffffffu;
    const uint32_t bid = t < nb ? static_cast<uint32_t>(bias_ids[t]) : 0xffffffffu;  // the first bias ids
    if (wv == WS_WAVES - 1u) {  // one wave draws the row's uniform for everybody
        // (the seed by way of a vector register: as scalar arithmetic the generator's rounds are moved out of this
        // branch, and sixteen waves work them out)
        uint32_t seed_lo = static_cast<uint32_t>(P.seed);
        asm volatile("" : "+v"(seed_lo));
        const double u_ = batch_uniform(A.rng, (P.seed & 0xffffffff00000000ull) | seed_lo, row, P.step, 0);
        if (lane == 0u) {
            s_d[6] = u_;
            s_d[8] = neg_log_min_p;
        }
    }
    WSL_MARK(0);

    // ------------------------------------------------------------------ the anchor: the head of the row + kLeanAbove exponent units
    const float c64 = inv_t * 64.f;
    float aq;
    {
        float s = -INFINITY, allowed = -INFINITY;
#pragma unroll
        for (int u = 0; u < kLeanBatch; ++u) {
            const uint32_t w[4] = {q[0][u].x, q[0][u].y, q[0][u].z, q[0][u].w};
            const int32_t out = MASKED ? static_cast<int32_t>(~na[0][u] >> ((min(u * WS_BLOCK + t, nv - 1u) * kTok) & 31u)) : 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s = fmaxf(s, __uint_as_float(w[e]));
                if (MASKED) allowed = fmaxf(allowed, __uint_as_float(w[e] | static_cast<uint32_t>((out << (31 - e)) >> 31)));
            }
        }
        // (its barriers also publish the zeroed histogram)
        if (MASKED) block_max2(s, allowed, red_f, reinterpret_cast<float*>(red_u));
        else s = block_max(s, red_f);
        // (of the allowed tokens, where there are any: one that is masked out may lie so far above the others that their masses would be lost)
        const float anchor = AGAIN ? S.top : (MASKED && allowed > -INFINITY ? allowed : s) + kLeanAbove / inv_t;
        aq = anchor_product(anchor, c64);
        if (!(anchor > -INFINITY && anchor < INFINITY)) WSL_FAIL(2);
    }

    // ------------------------------------------------------------------ the sweep
    uint32_t cache[NREG];
    float m = -INFINITY;
    float vm_early[kEarly * kLeanBatch];  // maxima of the early batches' vectors, until the bitmap says which hold a touched token
    const float tail_f = static_cast<float>(kLeanRoom - kLeanTail - static_cast<int>(t));  // the height of this thread's own tail bin
    const LeanWord at_anchor = (LeanWord)(((hist2 && (t & 1u)) ? hist2 : hist) + kLeanRoom);
    const uint32_t stage_cap = 2047u;
    const uint32_t n_full = (V >> kTokLog) / WS_BLOCK;  // rounds of whole vectors for every thread
    bool any_touched = false;               // uniform
    // the bitmap words of a batch are read a batch ahead, before the batch in between adds to the histogram: LDS
    // operations of a wave finish in order, and a read asked for behind the additions would wait for all of them
    uint32_t tws[2][kLeanBatch], wps[2][kLeanBatch];
    auto read_words = [&](int bt) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kLeanBatch; ++u) {
            const uint32_t word = (((bt * kLeanBatch + u) * WS_BLOCK + t) * kTok) >> 5;  // (past the row: a word past the bitmap, inside the block's LDS)
            tws[bt & 1][u] = any_touched ? touched[word] : 0u;
            wps[bt & 1][u] = any_touched ? wprefix[word] : 0u;
        }
    };
    // one batch: every token into the histogram, its bin's low byte into the cache; `early`: before phase 0. (A macro, not a
    // function: the cache stays in registers only while every index into it is a constant where the loops are unrolled.)
#define WSL_SWEEP_BATCH(bt, early)                                                                                                   \
    {                                                                                                                                \
        const int slot = (bt) % kRing;                                                                                               \
        if (!(early) && (bt) + 1 < NB) read_words((bt) + 1);                                                                         \
        _Pragma("unroll") for (int u = 0; u < kLeanBatch; ++u) {                                                                     \
            const uint32_t j = ((bt) * kLeanBatch + u) * WS_BLOCK + t;                                                               \
            const int c = (bt) * kLeanBatch + u;                                                                                     \
            uint32_t tw = (early) ? 0u : tws[(bt) & 1][u], nal = MASKED ? ~na[slot][u] : 0u;                                         \
            if (static_cast<uint32_t>(c) >= n_full) { /* uniform: only the row's last round has lanes past it */                      \
                if (j == j_part) q[slot][u] = part_vector<0>(q[slot][u], kTok - V % kTok);                                           \
                const bool past = j >= nv;            /* NaN: the tail bins, nobody's candidate (in place: no copy of the vector) */  \
                q[slot][u].x = past ? 0xffffffffu : q[slot][u].x;                                                                    \
                q[slot][u].y = past ? 0xffffffffu : q[slot][u].y;                                                                    \
                q[slot][u].z = past ? 0xffffffffu : q[slot][u].z;                                                                    \
                q[slot][u].w = past ? 0xffffffffu : q[slot][u].w;                                                                    \
                tw = past ? 0u : tw;                                                                                                 \
            }                                                                                                                        \
            const uint32_t w[4] = {q[slot][u].x, q[slot][u].y, q[slot][u].z, q[slot][u].w};                                          \
            const int32_t bw = MASKED ? static_cast<int32_t>(nal >> ((j * kTok) & 31u)) : 0;                                         \
            float vm = -INFINITY;                                                                                                    \
            int bins[4];                                                                                                                     \
            _Pragma("unroll") for (int e = 0; e < 4; ++e) {                                                                                  \
                uint32_t bits = w[e];                                                                                                        \
                if (MASKED) bits |= static_cast<uint32_t>((bw << (31 - e)) >> 31);                                                           \
                const float x = __uint_as_float(bits);                                                                                       \
                vm = fmaxf(vm, x);                                                                                                           \
                const float h = lean_height(aq, c64, x, tail_f);                                                                             \
                LeanWord word;                                                                                                               \
                bins[e] = lean_bin(h, at_anchor, word);                                                                                      \
                __hip_atomic_fetch_add(word, bin_word(-h), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);                                  \
            }                                                                                                                                \
            /* (kLeanRoom is a multiple of 256: the low bytes are those of the histogram's indices) */                                       \
            const uint32_t lo2 = __builtin_amdgcn_perm(bins[1], bins[0], 0x0c0c0400u);                                                       \
            uint32_t packed = __builtin_amdgcn_perm(bins[3], bins[2], 0x04000c0cu) | lo2;                                                    \
            if (MASKED) packed ^= masked_bytes(bw) & lean_other_byte(c);                                                                     \
            asm volatile("" : "+v"(packed)); /* (packed here, not where the tail first looks at it: four bins would stay live) */            \
            cache[c] = packed;                                                                                                               \
            if (early) {                                                                                                             \
                vm_early[c < kEarly * kLeanBatch ? c : 0] = vm;                                                                      \
            } else {                                                                                                                 \
                const uint32_t sh = (j * kTok) & 31u;                                                                                \
                const bool touched_vec = ((tw >> sh) & ((1u << kTok) - 1u)) != 0u;                                                   \
                m = fmaxf(m, touched_vec ? -INFINITY : vm); /* (a vector with a touched token is looked at when that token is collected) */ \
                if (touched_vec) {                                                                                                   \
                    const uint32_t r = wps[(bt) & 1][u] + __popc(tw & ((1u << sh) - 1u));                                            \
                    stage[min(r, stage_cap)] = q[slot][u];                                                                           \
                }                                                                                                                    \
            }                                                                                                                        \
        }                                                                                                                            \
    }
    // ------------------------------------------------------------------ phase 0 (ws_sample.h): bitmap of the touched ids,
    // popcount prefix per word (rank of a touched id), per-rank history count and bias entries
    uint32_t n_touched = 0;
    auto phase0 = [&]() __attribute__((always_inline)) {
    if (nh + nb > 0) {  // (the tables were cleared at the top; the anchor's barriers lie in between)
#pragma unroll
        for (int k = 0; k < kHid; ++k)
            if (static_cast<uint32_t>(k) * WS_BLOCK < nh && hid[k] < V) atomicOr(&touched[hid[k] >> 5], 1u << (hid[k] & 31u));
        for (uint32_t j = t + kHid * WS_BLOCK; j < nh; j += WS_BLOCK) {
            const uint32_t id = static_cast<uint32_t>(hist_ids[j]);
            if (id < V) atomicOr(&touched[id >> 5], 1u << (id & 31u));
        }
        if (bid < V) atomicOr(&touched[bid >> 5], 1u << (bid & 31u));
        for (uint32_t j = t + WS_BLOCK; j < nb; j += WS_BLOCK) {
            const uint32_t id = static_cast<uint32_t>(bias_ids[j]);
            if (id < V) atomicOr(&touched[id >> 5], 1u << (id & 31u));
        }
        __syncthreads();
        constexpr uint32_t kChunk = (NREG + 7) / 8;  // words per thread: NREG * 4096 / 32 / 1024
        const uint32_t w0 = t * kChunk;
        uint32_t wd[kChunk], local = 0;
#pragma unroll
        for (uint32_t k = 0; k < kChunk; ++k) wd[k] = touched[min(w0 + k, nW - 1u)];
#pragma unroll
        for (uint32_t k = 0; k < kChunk; ++k) {
            if (w0 + k >= nW) wd[k] = 0u;
            local += __popc(wd[k]);
        }
        uint32_t n_uniq;
        uint32_t run = block_excl_scan(local, red_u, &n_uniq);
#pragma unroll
        for (uint32_t k = 0; k < kChunk; ++k) {
            if (w0 + k < nW) wprefix[w0 + k] = static_cast<uint16_t>(run);
            run += __popc(wd[k]);
        }
        __syncthreads();
        rv.touched = touched;
        const bool ids_now = nb == 0;  // without a bias list the second table takes the token id of each rank right away
#pragma unroll
        for (int k = 0; k < kHid; ++k)
            if (static_cast<uint32_t>(k) * WS_BLOCK < nh && hid[k] < V) {
                const uint32_t r = rank_of(rv, hid[k]);
                atomicAdd(&cnt[r], 1u);
                if (ids_now) first[r] = hid[k];
            }
        for (uint32_t j = t + kHid * WS_BLOCK; j < nh; j += WS_BLOCK) {
            const uint32_t id = static_cast<uint32_t>(hist_ids[j]);
            if (id < V) {
                const uint32_t r = rank_of(rv, id);
                atomicAdd(&cnt[r], 1u);
                if (ids_now) first[r] = id;
            }
        }
        for (uint32_t j = t; j < nb; j += WS_BLOCK) {
            const uint32_t id = j == t ? bid : static_cast<uint32_t>(bias_ids[j]);
            if (id < V) {
                const uint32_t r = rank_of(rv, id);
                atomicMin(&first[r], j);
                atomicAdd(&cnt[r], 1u << 20);
            }
        }
        n_touched = n_uniq;
        any_touched = n_uniq != 0u;
    }
    WSL_MARK(1);
    // the early batches' vectors: those without a touched token count for the running maximum
#pragma unroll
    for (int c = 0; c < kEarly * kLeanBatch; ++c) {
        const uint32_t j = static_cast<uint32_t>(c) * WS_BLOCK + t;
        const uint32_t tw = any_touched ? touched[(j * kTok) >> 5] : 0u;
        m = fmaxf(m, ((tw >> ((j * kTok) & 31u)) & ((1u << kTok) - 1u)) ? -INFINITY : vm_early[c]);
    }
    read_words(kEarly);
    };
    const uint32_t early_end = min(static_cast<uint32_t>(kEarly * kLeanBatch) * WS_BLOCK * kTok, V);  // tokens below this were binned before phase 0: not staged
    load(2, 2);
    double exp_tab = 0.0;
    // (one unrolled loop for all batches, phase 0 inside it: the bin cache stays in registers only while every index into
    // it is a constant once the loop is unrolled)
#pragma unroll
    for (int bt = 0; bt < NB; ++bt) {
        if (bt == kEarly) {
            WSL_MARK(11);
            phase0();
        }
        if (bt == (NB > 4 ? NB - 4 : 0)) exp_tab = t < 64 ? kExpHi[t] : (t < 128 ? kExpLo[t - 64] : 0.0);  // the histogram scan's tables: asked for now, parked in LDS after the sweep
        if (bt < kEarly) {
            WSL_SWEEP_BATCH(bt, true)
        } else if (static_cast<uint32_t>(bt * kLeanBatch) * WS_BLOCK < nv) {  // uniform
            WSL_SWEEP_BATCH(bt, false)
        } else {  // past the row (no way out of the loop here: with one, the cache no longer stays in registers)
#pragma unroll
            for (int u = 0; u < kLeanBatch; ++u) cache[bt * kLeanBatch + u] = 0u;
        }
        if (bt + kRing < NB) load(bt + kRing, bt % kRing);  // the slot is free: the batch three ahead
    }
    if constexpr (NB <= kEarly) phase0();
    if (t < 128) s_exp[t] = exp_tab;
#undef WSL_SWEEP_BATCH
    __syncthreads();
    WSL_MARK(2);
    // Everything behind the sweep reads its arguments again, through a pointer the compiler cannot see through: none of
    // them stays in a register across the sweep (they spilled there, dozens of them, and every phase paid for it).
    // (the kernel's argument segment itself, where BatchArgs is the first and only argument: scalar loads, no copy)
    LeanArgPtr Ap = AGAIN ? args : (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    const float rep = P.rep, pres = P.pres, freq = P.freq;
    const int32_t* hist_ids2 = Ap->hist + h0;
    const int32_t* bias_ids2 = Ap->bias_ids + b0;
    const float* bias_vals2 = Ap->bias_vals + b0;

    // ------------------------------------------------------------------ the touched tokens (collect_fused of ws_sample.h):
    // every history / bias entry claims its token's rank; the owner adjusts the token's logit and moves the token from the
    // bin of its raw logit to the bin of the adjusted one
    float ma = -INFINITY, mu = -INFINITY;
    if (n_touched) {
        constexpr uint32_t kClaim = 0x80000000u;
        uint64_t* const anchors = hist + kLeanRoom;
        const float tail_own = static_cast<float>(kLeanRoom - kLeanTail - static_cast<int>(t));
        const uint32_t stage_cap = 2047u;
        // K ids a thread and pass (a pass with nothing in its later slots would still issue their instructions)
        auto take = [&](auto kc, const int32_t* ids, uint32_t n, uint32_t j0, const uint32_t* kept_id) __attribute__((always_inline)) {
            constexpr int K = decltype(kc)::value;
            if (j0 + wv * 64u < n) {  // (per wave: one with no id left issues nothing, and the others have the SIMDs to themselves)
                uint32_t id[K], al[K], tw[K], wp[K], rk[K], old[K];
                uint4 vec[K];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const uint32_t j = j0 + k * WS_BLOCK + t;
                    if (K == 1 && kept_id != nullptr) id[k] = *kept_id;  // (the one id that stayed in a register through the sweep)
                    else id[k] = j < n ? static_cast<uint32_t>(ids[j]) : 0xffffffffu;  // (read again: the sweep has the registers)
                    if (id[k] >= V) id[k] = 0xffffffffu;
                }
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const uint32_t i = id[k] < V ? id[k] : 0u;
                    al[k] = MASKED ? rv.allow[i >> 5] : 0xffffffffu;
                    tw[k] = touched[i >> 5];
                    wp[k] = wprefix[i >> 5];
                }
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const uint32_t i = id[k] < V ? id[k] : 0u;
                    const uint32_t vb = i & ~(kTok - 1u);
                    const uint32_t rf = id[k] < V ? wp[k] + __popc(tw[k] & ((1u << (vb & 31u)) - 1u)) : 0u;
                    rk[k] = wp[k] + __popc(tw[k] & ((1u << (i & 31u)) - 1u));
                    old[k] = id[k] < V ? atomicOr(&cnt[rk[k]], kClaim) : kClaim;
                    if (rf < stage_cap && i >= early_end) {
                        vec[k] = stage[rf];
                    } else {
                        vec[k] = row_vector<0>(xv, i >> kTokLog, V);
                        if (i >> kTokLog == j_part) vec[k] = part_vector<0>(vec[k], kTok - V % kTok);
                    }
                }
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    if (old[k] & kClaim) continue;
                    const uint32_t i = id[k];
                    const uint32_t w[4] = {vec[k].x, vec[k].y, vec[k].z, vec[k].w};
                    const uint32_t e_ = i & (kTok - 1u);
                    const uint32_t bits = pick4(e_, w[0], w[1], w[2], w[3]);
                    const float raw = ((al[k] >> (i & 31u)) & 1u) ? fmaxf(__uint_as_float(bits), -INFINITY) : -INFINITY;
                    {  // the vector's tokens that nothing touches count for the maximum here (those past the row are NaN)
                        const uint32_t free_bits = (al[k] & ~tw[k]) >> (i & (32u - kTok));
#pragma unroll
                        for (uint32_t e = 0; e < kTok; ++e) {
                            if ((free_bits >> e) & 1u) mu = fmaxf(mu, __uint_as_float(w[e]));
                        }
                    }
                    const uint32_t cw = old[k], c = cw & 0xfffffu, n_bias = (cw >> 20) & 0x7ffu;
                    float x = raw;
                    if (__ballot(n_bias != 0u)) {  // uniform
                        const uint32_t j = n_bias ? first[rk[k]] : 0u;
                        if (n_bias) x = __fadd_rn(x, bias_vals2[j]);
                        x = add_other_bias(n_bias > 1u, i, j, x, bias_ids2, bias_vals2, nb);
                    }
                    if (c) {
                        x = x > 0.f ? __fdiv_rn(x, rep) : __fmul_rn(x, rep);
                        x = __fsub_rn(x, __fadd_rn(__fmul_rn(freq, static_cast<float>(c)), pres));
                    }
                    pv[rk[k]] = x;
                    first[rk[k]] = i;  // the token id of the rank from here on
                    ma = fmaxf(ma, x);
                    const float from = lean_height(aq, c64, raw, tail_own), to = lean_height(aq, c64, x, tail_own);
                    atomicAdd(reinterpret_cast<unsigned long long*>(&anchors[lean_bin(from)]), 0ull - bin_word(-from));
                    atomicAdd(reinterpret_cast<unsigned long long*>(&anchors[lean_bin(to)]), bin_word(-to));
                }
            }
        };
        auto take_all = [&](const int32_t* ids, uint32_t n, const uint32_t* first_id) __attribute__((always_inline)) {
            if (n <= WS_BLOCK) {  // (the usual case: one id a thread, and that one is at hand)
                if (n) take(std::integral_constant<int, 1>{}, ids, n, 0u, first_id);
                return;
            }
            uint32_t j0 = 0;
            for (; j0 + 2u * WS_BLOCK < n; j0 += 4u * WS_BLOCK) take(std::integral_constant<int, 4>{}, ids, n, j0, nullptr);
            if (j0 + WS_BLOCK < n) take(std::integral_constant<int, 2>{}, ids, n, j0, nullptr);
            else if (j0 < n) take(std::integral_constant<int, 1>{}, ids, n, j0, nullptr);
        };
        take_all(hist_ids2, nh, &hid[0]);
        take_all(bias_ids2, nb, &bid);
    }
    WSL_MARK(3);
    {
        float m_all = fmaxf(fmaxf(m, mu), ma);
        m = block_max(m_all, red_f);  // its barriers also end the moves in the histogram
    }
    {  // the sweep stands if no token lies above the first bin and that one is not wastefully high (and not on a row without any token: m = -inf)
        const float above = __fmaf_rn(m, c64, -aq);
        if (!(above <= static_cast<float>(kLeanRoom) && above >= static_cast<float>(kLeanRoom - 1024))) {
            if (AGAIN || !(m > -INFINITY && above <= static_cast<float>(kLeanFar))) WSL_FAIL(3);
            if (t == 0u) S.top = m;
            return false;
        }
    }

    // ------------------------------------------------------------------ scan of the histogram: four consecutive bins a thread,
    // the prefixes stay in registers
    const double lift = (static_cast<double>(aq) + kLeanRoom) * (1.0 / 64.0) - static_cast<double>(m) * static_cast<double>(inv_t);  // >= 0
    if (wv == 0u) {  // one wave: the factor that takes masses from the first bin to the maximum
        const double tm = exp(lift);
        if (lane == 0u) s_d[7] = tm;
    }
    const uint32_t bb = 4u * t;  // this thread's bins: bb .. bb + 3
    uint32_t c4b[4], ce[4];      // tokens in the bin, tokens ranked before it
    double me[5];                // mass ranked before the bin; me[4]: before the next thread's first bin
    double Z;
    {
        uint64_t h[4];
        {
            const ulonglong2 h01 = *reinterpret_cast<const ulonglong2*>(&hist[bb]), h23 = *reinterpret_cast<const ulonglong2*>(&hist[bb + 2u]);
            h[0] = h01.x, h[1] = h01.y, h[2] = h23.x, h[3] = h23.y;
            if (hist2) {
                const ulonglong2 g01 = *reinterpret_cast<const ulonglong2*>(&hist2[bb]), g23 = *reinterpret_cast<const ulonglong2*>(&hist2[bb + 2u]);
                h[0] += g01.x, h[1] += g01.y, h[2] += g23.x, h[3] += g23.y;
            }
        }
        double ms[4];
        uint32_t lc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            c4b[k] = bb + k < static_cast<uint32_t>(kLeanTail) ? static_cast<uint32_t>(h[k] >> kCountShift) : 0u;  // (the tail's words are not looked at one by one)
            ms[k] = 0.0;
            lc += c4b[k];
        }
        const bool wave_has = __ballot(lc != 0u) != 0ull;
        if (wave_has) {  // uniform: a wave whose 256 bins hold no token needs no arithmetic
            const double eh = s_exp[bb >> 6];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t fl = static_cast<uint32_t>(h[k]), fh = static_cast<uint32_t>(h[k] >> 32) & ((1u << (kCountShift - 32)) - 1u);
                const double fix = (static_cast<double>(fh) * 4294967296.0 + static_cast<double>(fl)) * kFixInv;  // exact: below 2^44
                ms[k] = c4b[k] ? eh * s_exp[64 + ((bb + k) & 63u)] * (static_cast<double>(c4b[k]) - fix) : 0.0;
            }
        }
        const uint32_t ic = wave_has ? wave_incl_scan(lc) : 0u;
        __syncthreads();  // the factor is in place (and every read of the histogram is done)
        const double to_max = s_d[7];
        double lm = 0.0, im = 0.0, up = 0.0;
        if (wave_has) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                ms[k] *= to_max;
                lm += ms[k];
            }
            im = wave_incl_scan(lm);
            up = __shfl_up(im, 1);
        }
        if (lane == 63u) {
            red_u[wv] = ic;
            red_d[wv] = im;
        }
        __syncthreads();
        WSL_MARK(16);
        // the waves' totals, scanned by every wave again: lane w holds wave w's
        const uint32_t wc = lane < WS_WAVES ? red_u[lane] : 0u;
        const double wm = lane < WS_WAVES ? red_d[lane] : 0.0;
        const uint32_t wci = wave_incl_scan(wc);
        const double wmi = wave_incl_scan(wm);
        const uint32_t base_c = wv ? lane_value(wci, wv - 1u) : 0u;
        const double base_m = wv ? lane_value(wmi, wv - 1u) : 0.0;
        Z = lane_value(wmi, WS_WAVES - 1u);
        uint32_t rc = base_c + ic - lc;
        double rm = base_m + (lane ? up : 0.0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            ce[k] = rc;
            me[k] = rm;
            rc += c4b[k];
            rm += ms[k];
        }
        me[4] = base_m + im;  // (what the next thread starts from, bit for bit)
        if (t == WS_BLOCK - 1u) {
            me[4] = Z;
            S.m_left = m;  // (for lean_rest; written here, where they are at hand: on the way out they cost the longest build registers)
            S.z_left = Z;
            S.touched_left = n_touched;
        }
    }
    WSL_MARK(4);
    const double Zf = static_cast<double>(static_cast<float>(Z));  // Sampler::sum is a float (src/sampling/sampler.h:38)

    // ------------------------------------------------------------------ select (the rules of ws_sample.h): the bins the cut
    // and the draw can fall in. Every thread looks at the four bins it has just scanned; a search - the first bin with a
    // token whose mass prefix reaches a value - is one ballot per wave, one record per wave in LDS and one barrier.
    using BinRec = LeanBinRec;
    BinRec* rec = S.rec;  // [search][wave]
    // this thread's first bin with a token whose inclusive prefix satisfies the test; 4 when none does. Only one wave has
    // such a bin that counts - the wave in whose 256 bins the prefix passes the value: the waves before it reach no such
    // bin, the waves behind it are not the first - so the others answer without looking.
    const double wave_lo = lane_value(me[0], 0u), wave_hi = lane_value(me[4], 63u);  // prefix before the wave's bins and behind them
    auto first_own = [&](double Xq, bool strict) {
        uint32_t k = 4u;
        const bool mine = strict ? (wave_hi > Xq && !(wave_lo > Xq)) : (wave_hi >= Xq && !(wave_lo >= Xq));  // uniform
        if (mine) {
#pragma unroll
            for (int j = 3; j >= 0; --j)
                if (c4b[j] != 0u && (strict ? me[j + 1] > Xq : me[j + 1] >= Xq)) k = static_cast<uint32_t>(j);
        }
        return k;
    };
    auto publish = [&](uint32_t search, uint32_t k) {  // the wave's first such bin
        const uint64_t any = __ballot(k < 4u);
        if (any == 0ull) {
            if (lane == 0u) rec[search * WS_WAVES + wv].b = 0xffffffffu;
        } else if (lane == static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1)) {
            BinRec r;
            r.b = bb + k;
            r.mex = pick4(k, me[0], me[1], me[2], me[3]);
            r.min_ = pick4(k, me[1], me[2], me[3], me[4]);
            r.cex = pick4(k, ce[0], ce[1], ce[2], ce[3]);
            r.c = pick4(k, c4b[0], c4b[1], c4b[2], c4b[3]);
            r.pad = 0u;
            rec[search * WS_WAVES + wv] = r;
        }
    };
    auto found = [&](uint32_t search) {  // the first wave's record that holds a bin (b = 0xffffffff: none)
        BinRec r;
        r.b = 0xffffffffu;
        r.mex = r.min_ = 0.0;
        r.cex = r.c = r.pad = 0u;
        const uint32_t mine = lane < WS_WAVES ? rec[search * WS_WAVES + lane].b : 0xffffffffu;
        const uint64_t any = __ballot(mine != 0xffffffffu);
        if (any) r = rec[search * WS_WAVES + static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1)];
        return r;
    };
    // the record of a bin named outright, by the thread that owns it (searches 4..7)
    auto publish_bin = [&](uint32_t search, int b) {
        if (b >= 0 && static_cast<uint32_t>(b) >> 2 == t) {
            const uint32_t k = static_cast<uint32_t>(b) & 3u;
            BinRec r;
            r.b = static_cast<uint32_t>(b);
            r.mex = pick4(k, me[0], me[1], me[2], me[3]);
            r.min_ = pick4(k, me[1], me[2], me[3], me[4]);
            r.cex = pick4(k, ce[0], ce[1], ce[2], ce[3]);
            r.c = pick4(k, c4b[0], c4b[1], c4b[2], c4b[3]);
            r.pad = 0u;
            rec[4u * WS_WAVES + (search - 4u)] = r;
        }
    };
    // The searches are every wave's work; what follows from their answers is worked out by wave 0 alone and handed
    // round through LDS (sixteen waves doing the same arithmetic side by side take four times as long as one).
    LeanSel& sel = S.sel;
    // first search: the top-p cut against the float normaliser and against the exact one; the min-p bins by name
    int lo3 = kBins, hi3 = -1;
    if (use_min_p) {
        const double astar = (s_d[8] + lift) * 64.0;
        const double lo = floor(astar - 4e-3), hi = floor(astar + 4e-3);
        lo3 = lo < 0 ? 0 : (lo > kLeanTail ? kLeanTail : static_cast<int>(lo));
        hi3 = hi < 0 ? 0 : (hi > kLeanTail ? kLeanTail : static_cast<int>(hi));
    }
    if (use_top_p) {
        const double Xf = top_p * Zf, Xz = top_p * Z;
        publish(0u, Xf > 0.0 ? first_own(Xf, false) : 4u);
        publish(1u, Xz > 0.0 ? first_own(Xz, false) : 4u);
    }
    if (use_min_p) {
        publish_bin(4u, min(lo3, kLeanTail - 1));
        publish_bin(5u, min(hi3, kLeanTail - 1));
    }
    WSL_MARK(17);
    __syncthreads();
    WSL_MARK(15);
    if (wv == 0u) {
        int r1lo = 0, r1hi = -1;
        bool minp_in_list = false, topp_in_list = false;
        double X = 0, zlo = Z, zhi = Z;  // zlo, zhi: bounds of the kept mass
        uint32_t r1c0 = 0, r1c1 = 0;     // tokens ranked before range 1, and up to and with its last bin
        int b2 = -1;
        BinRec cut;
        cut.b = 0xffffffffu;
        cut.mex = cut.min_ = 0.0;
        cut.cex = cut.c = cut.pad = 0u;
        if (use_top_p) {
            X = top_p * Zf;
            cut = found(0u);
            if (cut.b != 0xffffffffu && cut.cex >= 16384u) {
                X = top_p * Z;
                cut = found(1u);
            }
            b2 = cut.b != 0xffffffffu ? static_cast<int>(cut.b) : kLeanTail;
        }
        const BinRec flo = use_min_p ? rec[4u * WS_WAVES] : cut, fhi = use_min_p ? rec[4u * WS_WAVES + 1u] : cut;
        if (use_top_p && (!use_min_p || b2 < lo3)) {
            r1lo = r1hi = b2;
            topp_in_list = true;
            zlo = cut.mex, zhi = cut.min_;
            r1c0 = cut.cex, r1c1 = cut.cex + cut.c;
        } else if (use_min_p && (!use_top_p || hi3 < b2)) {
            r1lo = lo3;
            r1hi = hi3;
            minp_in_list = true;
            zlo = flo.mex, zhi = fhi.min_;
            r1c0 = flo.cex, r1c1 = fhi.cex + fhi.c;
        } else if (use_top_p && use_min_p) {
            r1lo = min(b2, lo3);
            r1hi = max(b2, hi3);
            minp_in_list = topp_in_list = true;
            zlo = b2 < lo3 ? cut.mex : flo.mex;
            zhi = b2 > hi3 ? cut.min_ : fhi.min_;
            r1c0 = b2 < lo3 ? cut.cex : flo.cex;
            r1c1 = b2 > hi3 ? cut.cex + cut.c : fhi.cex + fhi.c;
        }
        const double m1lo = zlo;                           // mass ranked before range 1
        if (topp_in_list && !minp_in_list && cut.b != 0xffffffffu && cut.c != 0u) kept_bounds(X, cut.c, zlo, zhi);
        if (r1lo == 0 && zlo < 1.0) zlo = fmin(1.0, zhi);  // the top token is always kept
        if (lane == 0u) {
            sel.X = X;
            sel.m1base = m1lo;
            sel.r1lo = r1lo, sel.r1hi = r1hi;
            sel.c1base = r1c0, sel.n_r1 = r1c1;  // (until the second round: tokens before range 1, and up to and with it)
            sel.topp_in_list = topp_in_list, sel.minp_in_list = minp_in_list;
            sel.ok = r1hi < kLeanTail;               // the tail has no mass resolution
            const double u = s_d[6];
            s_d[4] = u * zlo * (1.0 - 1e-9);     // second search: the bins the draw can land in
            s_d[5] = u * zhi * (1.0 + 1e-9);
            s_w[0] = 0u;
            s_w[5] = 0u;
        }
    }
    __syncthreads();
    if (!sel.ok) WSL_FAIL(4);
    publish(2u, first_own(s_d[4], true));
    publish(3u, first_own(s_d[5], true));
    WSL_MARK(18);
    __syncthreads();
    WSL_MARK(19);
    if (wv == 0u) {
        int r0lo = 0, r0hi = -1, r1lo = sel.r1lo, r1hi = sel.r1hi;
        const uint32_t r1c0 = sel.c1base, r1c1 = sel.n_r1;
        const double m1lo = sel.m1base;
        uint32_t c0base = 0, n_r0 = 0, c1base = 0, n_r1 = 0;
        double m0base = 0.0, m1base = 0.0;
        const BinRec dlo = found(2u), dhi = found(3u);
        const int b4lo = dlo.b != 0xffffffffu ? static_cast<int>(dlo.b) : 0;
        int b4hi = dhi.b != 0xffffffffu ? static_cast<int>(dhi.b) : ((r1hi >= r1lo) ? r1hi : kLeanTail - 1);
        if (b4hi < b4lo) b4hi = b4lo;
        // (a bound that was not found by a search has no record: such rows are rare and go the other way)
        bool ok = !(dlo.b == 0xffffffffu || dhi.b == 0xffffffffu || static_cast<int>(dhi.b) < b4lo);
        if (r1hi >= r1lo && b4hi >= r1lo - 1) {  // adjacent or overlapping: one range
            r0lo = min(b4lo, r1lo);
            r0hi = max(b4hi, r1hi);
            c0base = b4lo <= r1lo ? dlo.cex : r1c0;
            m0base = b4lo <= r1lo ? dlo.mex : m1lo;
            n_r0 = (b4hi >= r1hi ? dhi.cex + dhi.c : r1c1) - c0base;
            r1lo = 0;
            r1hi = -1;
        } else {
            r0lo = b4lo;
            r0hi = b4hi;
            c0base = dlo.cex;
            m0base = dlo.mex;
            n_r0 = dhi.cex + dhi.c - c0base;
            if (r1hi >= r1lo) {
                c1base = r1c0;
                n_r1 = r1c1 - r1c0;
                m1base = m1lo;
            }
        }
        const bool has_r1 = r1hi >= r1lo;
        const uint32_t nb0 = static_cast<uint32_t>(r0hi - r0lo + 1), nb1 = has_r1 ? static_cast<uint32_t>(r1hi - r1lo + 1) : 0u;
        ok = ok && r0hi < kLeanTail && nb0 <= kLeanWide && nb1 <= kLeanWide && n_r0 + n_r1 != 0u && n_r0 + n_r1 <= kLeanMaxList;
        {  // the bytes to scan the cache for: lane k looks at the k-th bin of the ranges, the first of a kind is listed
            uint32_t my_bin = lane < nb0 ? static_cast<uint32_t>(r0lo) + lane : static_cast<uint32_t>(r1lo) + (lane - nb0);
            uint32_t n_bins = nb0 + nb1;
            if (ok && n_bins > 8u) {  // (more bins than the scan takes bytes)
                // (uniform, rare) A peaked row: a handful of tokens, dozens of bins apart, where the draw may land. Only
                // the bins that hold a token count: the lanes look them up in the histogram, 64 bins a round, and those
                // with a token move up to the first lanes in order.
                uint32_t found_bin = 0xffffffffu, n_found = 0;
                for (uint32_t base = 0; base < nb0 + nb1; base += 64u) {
                    const uint32_t k = base + lane;
                    const uint32_t b = k < nb0 ? static_cast<uint32_t>(r0lo) + k : static_cast<uint32_t>(r1lo) + (k - nb0);
                    uint64_t word = 0ull;
                    if (k < nb0 + nb1) word = hist[b] + (hist2 ? hist2[b] : 0ull);
                    const uint64_t has = __ballot((word >> kCountShift) != 0ull);
                    // lane n_found + j takes the j-th bin of this round that holds a token
                    const uint32_t want_j = lane - n_found;
                    uint64_t rest = has;
                    uint32_t src = 0xffffffffu;
                    if (lane >= n_found && want_j < static_cast<uint32_t>(__popcll(has))) {
                        for (uint32_t j = 0; j < want_j; ++j) rest &= rest - 1ull;
                        src = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(rest)) - 1);
                    }
                    const uint32_t b_src = __shfl(b, static_cast<int>(src & 63u));
                    if (src != 0xffffffffu) found_bin = b_src;
                    n_found += static_cast<uint32_t>(__popcll(has));
                }
                my_bin = found_bin;
                n_bins = n_found;
                ok = ok && n_found <= kLeanMaxBins;
            }
            const uint32_t my_byte = my_bin & 0xffu;
            bool is_first = lane < n_bins && lane < kLeanMaxBins;
#pragma unroll
            for (uint32_t j = 0; j + 1u < kLeanMaxBins; ++j) {
                const uint32_t other = lane_value(my_byte, j);
                if (j < lane && j < n_bins && other == my_byte) is_first = false;
            }
            const uint64_t firsts = __ballot(is_first);
            const uint32_t place = static_cast<uint32_t>(__popcll(firsts & ((1ull << lane) - 1ull)));
            if (is_first && place < 8u) sel.bytes[place] = my_byte * 0x01010101u;
            const uint32_t n_bytes = static_cast<uint32_t>(__popcll(firsts));
            if (lane == 0u) sel.n_bytes = n_bytes;
            ok = ok && n_bytes <= 8u;
        }
        if (lane == 0u) {
            sel.r0lo = r0lo, sel.r0hi = r0hi, sel.r1lo = r1lo, sel.r1hi = r1hi;
            sel.c0base = c0base, sel.n_r0 = n_r0, sel.c1base = c1base, sel.n_r1 = n_r1;
            sel.m0base = m0base, sel.m1base = m1base;
            sel.ok = ok;
        }
    }
    __syncthreads();
    if (!sel.ok) {  // (what follows from it is worked out by lean_rest, for the same reason)
        if (t == 0u) S.top = INFINITY;
        return false;
    }
    const int r0lo = sel.r0lo, r0hi = sel.r0hi, r1lo = sel.r1lo, r1hi = sel.r1hi;
    const bool has_r1 = r1hi >= r1lo;
    const uint32_t nb0 = static_cast<uint32_t>(r0hi - r0lo + 1), nb1 = has_r1 ? static_cast<uint32_t>(r1hi - r1lo + 1) : 0u;
    const uint32_t c0base = sel.c0base, n_r0 = sel.n_r0, c1base = sel.c1base, n_r1 = sel.n_r1;
    const uint32_t n_list = n_r0 + n_r1;
    const bool topp_in_list = sel.topp_in_list != 0u, minp_in_list = sel.minp_in_list != 0u;
    const double X = sel.X, m0base = sel.m0base, m1base = sel.m1base;
    WSL_MARK(5);

    // ------------------------------------------------------------------ the tokens of those bins
    // (the sort's tables, cleared here for the barrier behind the scan: smallest and largest logit key in each of the (up
    // to sixteen) bins of the ranges, eight copies a bin - a lane adds to copy lane % 8 - and the buckets' counts)
    if (t < kLeanBuckets) {
        b_cnt[t] = 0xffffffffu;
        b_cpre[t] = 0u;
        if (t < 4u * kLeanMaxBins) S.b_mid[t] = 0xffffffffu;
    }
    if (t < 256u) reinterpret_cast<uint32_t*>(b_mass)[t] = 0u;
    uint2* list = reinterpret_cast<uint2*>(lds + 32768);
    constexpr uint32_t kListCap = 4096u;
    const uint32_t u0 = static_cast<uint32_t>(r0lo), w0 = nb0 - 1u;
    const uint32_t u1r = has_r1 ? static_cast<uint32_t>(r1lo) : 0xffff0000u, w1 = has_r1 ? nb1 - 1u : 0u;
    auto bin_at = [&](float x) { return static_cast<uint32_t>(lean_bin(lean_height(aq, c64, x, static_cast<float>(kLeanRoom - 4095))) + kLeanRoom); };
    auto in_ranges = [&](float x) {
        const uint32_t b = bin_at(x);
        return b - u0 <= w0 || b - u1r <= w1;
    };
    {
        LeanHits<NREG> H;
        constexpr int kGroups = LeanHits<NREG>::kGroups;
        const void* xg = rv.base;
        const uint32_t nt = sel.n_bytes;
        const uint4 by0 = *reinterpret_cast<const uint4*>(&sel.bytes[0]);
        {
            const uint32_t c4[4] = {by0.x, by0.y, by0.z, by0.w};
            const uint32_t n = min(4u, nt);
            if (n == 1u) lean_scan<1, false>(cache, c4, xg, H, list, &s_w[0], kListCap, V);
            else if (n == 2u) lean_scan<2, false>(cache, c4, xg, H, list, &s_w[0], kListCap, V);
            else if (n == 3u) lean_scan<3, false>(cache, c4, xg, H, list, &s_w[0], kListCap, V);
            else lean_scan<4, false>(cache, c4, xg, H, list, &s_w[0], kListCap, V);
        }
        if (nt > 4u) {  // uniform, rare: a second round for the other bytes, every find through the list
            const uint4 by1 = *reinterpret_cast<const uint4*>(&sel.bytes[4]);
            const uint32_t c4[4] = {by1.x, nt > 5u ? by1.y : by1.x, nt > 6u ? by1.z : by1.x, nt > 7u ? by1.w : by1.x};
            lean_scan<4, true>(cache, c4, xg, H, list, &s_w[0], kListCap, V);
        }
        WSL_MARK(20);
        // touched tokens whose adjusted logit lies in the ranges
        auto list_touched = [&]() __attribute__((always_inline)) {
            for (uint32_t r = t; r < n_touched; r += WS_BLOCK) {
                const float x = pv[r];
                if (in_ranges(x)) {
                    const uint32_t slot = atomicAdd(&s_w[0], 1u);
                    if (slot < kListCap) list[slot] = make_uint2(first[r] | kListAdjusted, __float_as_uint(x));
                }
            }
        };
        list_touched();
        WSL_MARK(21);
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < 2 * kGroups; ++k) mine += H.idx[k] != 0xffffffffu ? 1u : 0u;
        const uint32_t inc = wave_incl_scan(mine);
        uint32_t base = 0;
        if (lane == 63u && inc) base = atomicAdd(&s_w[0], inc);
        uint32_t slot = __shfl(base, 63) + inc - mine;
#pragma unroll
        for (int k = 0; k < 2 * kGroups; ++k) {
            if (H.idx[k] == 0xffffffffu) continue;
            if (slot < kListCap) list[slot] = make_uint2(H.idx[k], H.bits[k]);
            ++slot;
        }
        if constexpr (NREG >= kLeanLooks) {
            // A long row whose finds are more than the list holds (a byte finds a thousand tokens of 262144): once more, and each find is looked at before it is
            // listed, one after the other - 20 us, a quarter of what the three-pass code takes.
            __syncthreads();
            if (s_w[0] > kListCap) {  // uniform
                __syncthreads();
                if (t == 0u) s_w[0] = 0u;
                __syncthreads();
                auto wanted = [&](uint32_t bits) { return in_ranges(fmaxf(__uint_as_float(bits), -INFINITY)); };
#pragma unroll 1
                for (uint32_t b0_ = 0; b0_ < nt; b0_ += 4u) {
                    const uint4 by = *reinterpret_cast<const uint4*>(&sel.bytes[b0_]);
                    const uint32_t c4[4] = {by.x, nt > b0_ + 1u ? by.y : by.x, nt > b0_ + 2u ? by.z : by.x, nt > b0_ + 3u ? by.w : by.x};
                    lean_scan<4, true>(cache, c4, xg, H, list, &s_w[0], kListCap, V, wanted);
                }
                list_touched();
            }
        }
    }
    WSL_MARK(22);
    __syncthreads();
    WSL_MARK(6);
    const uint32_t n_hit = s_w[0];
#ifdef WS_PHASE_TIMERS
    if (t == 0) {
        S.marks[12] = nb0 + nb1;
        S.marks[13] = n_hit;
        S.marks[14] = n_list;
    }
#endif
    if (n_hit > kListCap) WSL_FAIL(6);
    // The sort's buckets: 1024 of them in the last 8 KiB of the list's region when the finds (and so the sorted keys,
    // which go there) leave them free, cleared here for the barrier behind the filter; the 256 of the static tables else.
    const bool wide_sort = n_hit <= kListCap - 1024u;
    uint32_t* bcnt = wide_sort ? reinterpret_cast<uint32_t*>(lds + 32768 + (kListCap - 1024u) * 8u) : reinterpret_cast<uint32_t*>(b_mass);
    uint32_t* bstart = wide_sort ? bcnt + 1024 : reinterpret_cast<uint32_t*>(b_fpre);
    const uint32_t n_buckets = wide_sort ? 1024u : 256u;
    if (wide_sort) bcnt[t] = 0u;

    // ------------------------------------------------------------------ the finds that are candidates: a token of another
    // bin with the same low bits, a masked-out token and a touched token found by its raw logit are dropped
    uint2* cand = reinterpret_cast<uint2*>(lds);  // (token | slot << 28, logit bits), kLeanMaxList entries at most
    const bool r1_first = has_r1 && r1lo < r0lo;  // range 1 holds the larger logits
    // a candidate's slot: the number of its bin among the ranges' bins in descending order of the logits
    // (a range of more than eight bins puts 2, 4, 8 .. neighbouring bins into one slot)
    const uint32_t sh0 = nb0 > 8u ? 29u - static_cast<uint32_t>(__clz(static_cast<int>(nb0 - 1u))) : 0u;
    const uint32_t sh1 = nb1 > 8u ? 29u - static_cast<uint32_t>(__clz(static_cast<int>(nb1 - 1u))) : 0u;
    const uint32_t ns0 = ((nb0 - 1u) >> sh0) + 1u, ns1 = has_r1 ? ((nb1 - 1u) >> sh1) + 1u : 0u;  // slots of the ranges
    auto slot_of = [&](float x) {
        const uint32_t b = bin_at(x);
        const bool in1 = has_r1 && b - static_cast<uint32_t>(r1lo) < nb1;
        const uint32_t s_ = in1 ? (r1_first ? 0u : ns0) + ((b - static_cast<uint32_t>(r1lo)) >> sh1) : (r1_first ? ns1 : 0u) + ((b - static_cast<uint32_t>(r0lo)) >> sh0);
        return min(s_, kLeanMaxBins - 1u);
    };
    {
        constexpr int kR = 4;
        uint2 en[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            const uint32_t k = r * WS_BLOCK + t;
            en[r] = k < n_hit ? list[k] : make_uint2(0xffffffffu, 0u);
        }
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            if (static_cast<uint32_t>(r) * WS_BLOCK + wv * 64u >= n_hit) continue;  // per wave
            const bool live = en[r].x != 0xffffffffu;
            const uint32_t id = live ? en[r].x & kListIdMask : 0u;
            float x = __uint_as_float(en[r].y);
            bool ok = live;
            if (!(en[r].x & kListAdjusted)) {
                if (en[r].x & kListNeedsLoad)
                    x = __uint_as_float(static_cast<const uint32_t*>(rv.base)[id]);
                x = fmaxf(x, -INFINITY);
                ok = ok && (!MASKED || is_allowed(rv, id)) && !is_touched(rv, id) && in_ranges(x);
            }
            const uint64_t mk = __ballot(ok);
            uint32_t base = 0;
            if (lane == 0u && mk) base = atomicAdd(&s_w[5], static_cast<uint32_t>(__popcll(mk)));
            const uint32_t slot = __shfl(base, 0) + static_cast<uint32_t>(__popcll(mk & ((1ull << lane) - 1ull)));
            if (ok && slot < kLeanMaxList) {
                const uint32_t s_ = slot_of(x), k32 = static_cast<uint32_t>(key64(x, 0u) >> 32);
                cand[slot] = make_uint2(id | (s_ << 28), __float_as_uint(x));
                atomicMin(&b_cnt[s_ * 8u + (lane & 7u)], k32);
                atomicMax(&b_cpre[s_ * 8u + (lane & 7u)], k32);
                S.b_mid[s_ * 4u + (lane & 3u)] = k32;  // (four of the bin's candidates, any: whichever stores land last)
            }
        }
    }
    if (t == 0) {
        s_q[0] = ~0ull;  // smallest mass at or above the min-p floor
        s_q[1] = 0ull;   // largest mass below it
        s_q[2] = ~0ull;  // the cut: (rank in the row << 32) | slot
        s_q[3] = ~0ull;  // the draw
        s_w[1] = 0u;     // candidates at or above the floor
        s_w[3] = 0u;     // the last kept candidate was found
    }
    __syncthreads();
    WSL_MARK(7);
    if (s_w[5] != n_list) WSL_FAIL(7);  // the histogram and the gather disagree
    // ---- the candidates in order (logit descending, id ascending): their 64-bit keys sorted by buckets. A bucket is
    // a bin of the ranges (eight at most) and, inside the bin, a 32nd of the span of the bin's logits - or, when all
    // its candidates tie, a 32nd of the vocabulary's ids: either way some dozens
    // of keys to compare with, and no limit on ties. A key's place is the start of its bucket plus the number of larger
    // keys among the bucket's members, which it reads once all keys lie bucket by bucket.
    constexpr int kRounds = kLeanMaxList / WS_BLOCK;  // the candidates at places kRounds t .. kRounds t + kRounds - 1 of the order
    uint64_t* keys = reinterpret_cast<uint64_t*>(lds);            // bucket by bucket (over the candidates' pairs, which are in registers by then)
    uint64_t* sorted = reinterpret_cast<uint64_t*>(lds + 32768);  // in order (over the finds' list)
    {
        uint32_t* kmin = b_cnt;
        uint32_t* kmax = b_cpre;
        uint64_t own[kRounds];
        uint32_t sl[kRounds], bk[kRounds], pos[kRounds];
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const uint32_t k = r * WS_BLOCK + t;
            const uint2 en = k < n_list ? cand[k] : make_uint2(0u, 0u);
            own[r] = key64(__uint_as_float(en.y), en.x & 0x0fffffffu);
            sl[r] = en.x >> 28;
        }
        // A bin's share of the buckets is cut in three: the logits above one of the bin's own candidates' (`mid`), by
        // logit; the candidates with exactly that logit, by id; the logits below, by logit. Where hundreds tie, `mid`
        // is theirs (two of four sampled candidates agree on it), and they spread over half the bin's buckets; where
        // no two logits are the same the middle part holds one candidate and the other half of the buckets serves.
        const uint32_t nt_ = ns0 + ns1;
        const uint32_t nsub = n_buckets >> (nt_ <= 1u ? 0u : (nt_ <= 2u ? 1u : (nt_ <= 4u ? 2u : (nt_ <= 8u ? 3u : 4u))));  // buckets a bin
        const uint32_t nl = nsub / 2u - 1u, nid = nsub / 2u;
        const float ids_scale = static_cast<float>(nid) / static_cast<float>(V);
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const uint32_t k = r * WS_BLOCK + t;
            if (static_cast<uint32_t>(r) * WS_BLOCK + wv * 64u < n_list && k < n_list) {
                const uint4 a0 = *reinterpret_cast<const uint4*>(&kmin[sl[r] * 8u]), a1 = *reinterpret_cast<const uint4*>(&kmin[sl[r] * 8u + 4u]);
                const uint4 b0 = *reinterpret_cast<const uint4*>(&kmax[sl[r] * 8u]), b1 = *reinterpret_cast<const uint4*>(&kmax[sl[r] * 8u + 4u]);
                // (`mid`: the logit two of the four sampled candidates share, or else the smallest of the four)
                const uint4 sm = *reinterpret_cast<const uint4*>(&S.b_mid[sl[r] * 4u]);
                uint32_t mid = min(min(sm.x, sm.y), min(sm.z, sm.w));
                if (sm.z != 0xffffffffu && sm.z == sm.w) mid = sm.z;
                if (sm.y != 0xffffffffu && (sm.y == sm.z || sm.y == sm.w)) mid = sm.y;
                if (sm.x != 0xffffffffu && (sm.x == sm.y || sm.x == sm.z || sm.x == sm.w)) mid = sm.x;
                const uint32_t lo = min(min(min(a0.x, a0.y), min(a0.z, a0.w)), min(min(a1.x, a1.y), min(a1.z, a1.w)));
                const uint32_t hi = max(max(max(b0.x, b0.y), max(b0.z, b0.w)), max(max(b1.x, b1.y), max(b1.z, b1.w)));
                const uint32_t k32 = static_cast<uint32_t>(own[r] >> 32);
                // (Levels by the logits themselves, not by their keys: a bin that holds the logit 0 spans a billion keys,
                // nearly all of its tokens among the topmost few million. None of the expressions rises along the order,
                // whatever the rounding: difference, product and truncation keep it.)
                const float x_hi = unkey32(hi), x_lo = unkey32(lo);
                const float per = static_cast<float>(nl) * __builtin_amdgcn_rcpf(fmaxf(__fsub_rn(x_hi, x_lo), 1e-30f));
                const uint32_t lk = min(nl - 1u, static_cast<uint32_t>(__fmul_rn(__fsub_rn(x_hi, unkey32(k32)), per)));
                const uint32_t lm = min(nl - 1u, static_cast<uint32_t>(__fmul_rn(__fsub_rn(x_hi, unkey32(mid)), per)));
                const uint32_t by_id = min(nid - 1u, static_cast<uint32_t>(static_cast<float>(0xffffffffu - static_cast<uint32_t>(own[r])) * ids_scale));
                const uint32_t sub = k32 > mid ? lk : (k32 == mid ? lm + 1u + by_id : lk + 1u + nid);
                bk[r] = sl[r] * nsub + sub;
                pos[r] = atomicAdd(&bcnt[bk[r]], 1u);
            }
        }
        __syncthreads();
        if (wv == 0u) {  // one wave: four or sixteen consecutive counts a lane
            if (wide_sort) {
                uint4 c[4];
                uint32_t sum = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    c[i] = *reinterpret_cast<const uint4*>(&bcnt[lane * 16u + 4u * i]);
                    sum += c[i].x + c[i].y + c[i].z + c[i].w;
                }
                uint32_t run = wave_incl_scan(sum) - sum;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    *reinterpret_cast<uint4*>(&bstart[lane * 16u + 4u * i]) = make_uint4(run, run + c[i].x, run + c[i].x + c[i].y, run + c[i].x + c[i].y + c[i].z);
                    run += c[i].x + c[i].y + c[i].z + c[i].w;
                }
            } else {
                const uint4 c = *reinterpret_cast<const uint4*>(&bcnt[lane * 4u]);
                const uint32_t sum = c.x + c.y + c.z + c.w;
                const uint32_t run = wave_incl_scan(sum) - sum;
                *reinterpret_cast<uint4*>(&bstart[lane * 4u]) = make_uint4(run, run + c.x, run + c.x + c.y, run + c.x + c.y + c.z);
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
            if (static_cast<uint32_t>(r) * WS_BLOCK + wv * 64u < n_list && r * WS_BLOCK + t < n_list) {
                bk[r] = bstart[bk[r]] | (bcnt[bk[r]] << 16);  // (start and count of the bucket: below 65536 both)
                keys[(bk[r] & 0xffffu) + pos[r]] = own[r];
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
            if (static_cast<uint32_t>(r) * WS_BLOCK + wv * 64u < n_list && r * WS_BLOCK + t < n_list) {
                const uint32_t b0 = bk[r] & 0xffffu, c = bk[r] >> 16;
                uint32_t above = 0;
                for (uint32_t i = 0; i < c; i += 4u) {  // four reads on their way together
                    uint64_t o[4];
#pragma unroll
                    for (uint32_t q_ = 0; q_ < 4u; ++q_) o[q_] = keys[b0 + min(i + q_, c - 1u)];
#pragma unroll
                    for (uint32_t q_ = 0; q_ < 4u; ++q_) above += (i + q_ < c && o[q_] > own[r]) ? 1u : 0u;
                }
                sorted[b0 + above] = own[r];
            }
        __syncthreads();
    }
    WSL_MARK(8);
    // every candidate: its rank in the row and the mass up to and with it
    const uint32_t nA = r1_first ? n_r1 : n_r0;  // candidates of the range with the larger logits: they come first
    const double mA = r1_first ? m1base : m0base, mB = r1_first ? m0base : m1base;
    const uint32_t cA = r1_first ? c1base : c0base, cB = r1_first ? c0base : c1base;
    // Thread t takes the places kr t .. kr t + kr - 1 of the order, kr as small as the number of candidates allows
    // (one thread's candidates are worked through one after the other). Only the waves that hold places work from
    // here on (wave 0 always does); the others pass the barriers and issue nothing else.
    const uint32_t kr = (n_list + WS_BLOCK - 1u) / WS_BLOCK;  // 1 .. kRounds
    const bool act = wv * 64u * kr < n_list;
    uint32_t cid[kRounds], cpos[kRounds];
    uint64_t ckey[kRounds];
    double cem[kRounds], cin[kRounds], cex[kRounds], pre[kRounds];
    double mine_ = 0.0, inc = 0.0, total = 0.0;
    if (act) {
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const uint32_t pos = kr * t + static_cast<uint32_t>(r);
            const bool on = static_cast<uint32_t>(r) < kr && pos < n_list;
            ckey[r] = on ? sorted[pos] : 0ull;
            cid[r] = 0xffffffffu - static_cast<uint32_t>(ckey[r]);
            cem[r] = 0.0;
            if (static_cast<uint32_t>(r) < kr && on) cem[r] = exp_neg(static_cast<double>(__fsub_rn(m, unkey32(static_cast<uint32_t>(ckey[r] >> 32)))) * static_cast<double>(inv_t), s_exp);
            mine_ += cem[r];
        }
        inc = wave_incl_scan(mine_);
    }
    if (lane == 63u) red_d[wv] = inc;
    __syncthreads();
    if (act) {
        const double wm = lane < WS_WAVES ? red_d[lane] : 0.0;
        const double wmi = wave_incl_scan(wm);
        total = lane_value(wmi, WS_WAVES - 1u);
        pre[0] = (wv ? lane_value(wmi, wv - 1u) : 0.0) + (inc - mine_);
#pragma unroll
        for (int r = 1; r < kRounds; ++r) pre[r] = pre[r - 1] + cem[r - 1];
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
            if (static_cast<uint32_t>(r) < kr && kr * t + static_cast<uint32_t>(r) == nA) s_d[2] = pre[r];  // mass of the first range's candidates
    }
    __syncthreads();
    WSL_MARK(9);
    // ---- the cuts (src/sampling/sampler.cpp:35-74): the first candidate at which the running mass reaches X
    const uint32_t n1 = V;
    if (act) {
        const double massA = nA < n_list ? s_d[2] : total;
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const uint32_t pos = kr * t + static_cast<uint32_t>(r);
            cpos[r] = 0xffffffffu;
            cin[r] = cex[r] = 0.0;
            if (static_cast<uint32_t>(r) >= kr) continue;  // uniform
            if (pos < n_list) {
                const bool inA = pos < nA;
                cex[r] = (inA ? mA : mB) + (pre[r] - (inA ? 0.0 : massA));
                cin[r] = cex[r] + cem[r];
                cpos[r] = (inA ? cA + pos : cB + (pos - nA));
            }
            if (use_min_p && minp_in_list) {  // uniform
                const bool pass = pos < n_list && cem[r] >= min_p;
                const uint64_t np = __ballot(pass);
                if (lane == 0u && np) atomicAdd(&s_w[1], static_cast<uint32_t>(__popcll(np)));
                if (pass) atomicMin(&s_q[0], static_cast<unsigned long long>(__double_as_longlong(cem[r])));
                if (pos < n_list && !pass) atomicMax(&s_q[1], static_cast<unsigned long long>(__double_as_longlong(cem[r])));
            }
            if (use_top_p && topp_in_list && cpos[r] != 0xffffffffu && cin[r] >= X && !(cex[r] >= X) && cin[r] > cex[r])
                atomicMin(&s_q[2], (static_cast<unsigned long long>(cpos[r]) << 32) | (static_cast<uint32_t>(r) * WS_BLOCK + t));
        }
    }
    __syncthreads();
    double mg_top_p = 1.0, mg_min_p = 1.0;
    uint32_t n2 = n1, n3 = n1;
    bool cut_found = false;
    if (act) {
        if (use_top_p && topp_in_list) {
            const unsigned long long cq = s_q[2];
            if (cq != ~0ull && static_cast<uint32_t>(cq >> 32) < n1) {
                cut_found = true;
                n2 = static_cast<uint32_t>(cq >> 32) + 1u;
            } else {  // rounding: the cut falls just past the gathered bins
                n2 = min(n1, has_r1 ? c1base + n_r1 : c0base + n_r0);
                mg_top_p = 0.0;
            }
        }
        n3 = n2;
        if (use_min_p && minp_in_list) {
            const uint32_t passed = s_w[1];
            double near = 1.0;
            if (passed > 0u) near = fmin(near, fabs(__longlong_as_double(static_cast<long long>(s_q[0])) - min_p) / min_p);
            if (passed < n_list) near = fmin(near, fabs(__longlong_as_double(static_cast<long long>(s_q[1])) - min_p) / min_p);
            uint32_t n3p;
            if (has_r1) n3p = passed >= n_r0 ? c1base + (passed - n_r0) : c0base + passed;
            else n3p = c0base + passed;
            n3 = min(n2, n3p);
            if (n3 < 1u) n3 = 1u;
            mg_min_p = near;
        }
        // the cut's margin, and the last kept candidate: mass of the kept set, its key, its own mass
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            if (static_cast<uint32_t>(r) >= kr || cpos[r] == 0xffffffffu) continue;
            if (cut_found && cpos[r] == n2 - 1u) s_d[3] = fmin(cin[r] - X, cpos[r] > 0u ? X - cex[r] : X) / X;
            if (cpos[r] == n3 - 1u) {
                s_d[0] = cin[r];
                s_d[1] = cem[r];
                s_q[4] = ckey[r];
                s_w[3] = 1u;
            }
        }
    }
    __syncthreads();
    const bool have_last = s_w[3] != 0u;
    double Zk = Z, target = 0.0;
    if (act) {
        if (cut_found) mg_top_p = s_d[3];
        if (have_last) Zk = s_d[0];
        else if (has_r1 && n3 == c1base) Zk = m1base;  // the cut falls on the upper edge of range 1: everything in earlier bins
        else if (n3 == c0base && n_r0) Zk = m0base;
        else Zk = Z;
        // ---- the draw (src/sampling/sampler.cpp:118-131): the first candidate at which the running mass passes u * Zk
        target = s_d[6] * Zk;
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
            if (static_cast<uint32_t>(r) < kr && cpos[r] != 0xffffffffu && cpos[r] < n3 && cin[r] > target && !(cex[r] > target) && cin[r] > cex[r])
                atomicMin(&s_q[3], (static_cast<unsigned long long>(cpos[r]) << 32) | (static_cast<uint32_t>(r) * WS_BLOCK + t));
    }
    __syncthreads();
    const unsigned long long dq = s_q[3];
    if (dq == ~0ull && !have_last) WSL_FAIL(8);  // no candidate for the draw and none to fall back on
#ifndef WS_PHASE_TIMERS  // (that build has a barrier at the end)
    if (!act) return true;
#endif
    const uint32_t d_slot = static_cast<uint32_t>(dq), d_pos = static_cast<uint32_t>(dq >> 32);
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        if (static_cast<uint32_t>(r) < kr && dq != ~0ull && static_cast<uint32_t>(r) * WS_BLOCK + t == d_slot) {
            const double mg = fmin(cin[r] - target, d_pos > 0u ? target - cex[r] : 1e300) / Zk;
            uint32_t flags = 0;
            const double tol = Ap->tol;
            if (mg_top_p < tol) flags |= kNearTopP;
            if (mg_min_p < tol) flags |= kNearMinP;
            if (mg < tol) flags |= kNearDraw;
            Ap->token[row] = static_cast<int32_t>(cid[r]);
            Ap->flags[row] = flags | kRouteLean | (AGAIN ? kRouteRedone : 0u);
            if (Ap->prob) Ap->prob[row] = static_cast<float>(cem[r] / Zk);
            if (Ap->margin) Ap->margin[3 * row + 2] = mg;
        }
    }
    if (t == 0) {
        if (dq == ~0ull) {  // the walk falls through to the last kept candidate (src/sampling/sampler.cpp:131)
            const double tol = Ap->tol;
            uint32_t flags = kNearDraw;
            if (mg_top_p < tol) flags |= kNearTopP;
            if (mg_min_p < tol) flags |= kNearMinP;
            Ap->token[row] = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(s_q[4]));
            Ap->flags[row] = flags | kRouteLean | (AGAIN ? kRouteRedone : 0u);
            if (Ap->prob) Ap->prob[row] = static_cast<float>(s_d[1] / Zk);
            if (Ap->margin) Ap->margin[3 * row + 2] = 0.0;
        }
        if (Ap->n_kept) Ap->n_kept[row] = n3;
        if (Ap->stats) {
            Ap->stats[2 * row] = m;
            Ap->stats[2 * row + 1] = static_cast<float>(Z);
        }
        if (Ap->margin) {
            Ap->margin[3 * row] = mg_top_p;
            Ap->margin[3 * row + 1] = mg_min_p;
        }
    }
    WSL_MARK(10);
#ifdef WS_PHASE_TIMERS
    __syncthreads();
    if (t < 32 && Ap->entropy) Ap->entropy[row * 32 + t] = static_cast<double>(S.marks[t]);
#endif
    return true;
}

// the three-pass code of ws_sample.h for one row, a function of its own: its registers and code stay out of the lean path.
// It takes the kernel's argument segment, and reads there where the three-pass layout of the LDS lies (sample_row's BACK).
// What it is handed comes in vector registers; said to be one value for the whole wave, so that everything that follows from it is scalar again. Not a tail
// call: only then does the compiler leave out saving the callers' registers, which nobody reads any more - thirty-five scalar registers went to memory one by one,
// each a round trip of a vector register that had to be free for it, and back at the end: 30 us of every handed-back row. (Before that, the arguments once
// copied, and now, us: one row of 50257 without a filter 75 / 44, the same beside 255 others with one 94 / 54, ten rows of 256 of 151937 with sigma / T = 8
// 137 / 95; ws_sample.h's own kernel takes 40, 48 and 88.)
__device__ __forceinline__ LeanArgPtr wave_args(LeanArgPtr Ap) {
    const uint64_t at = reinterpret_cast<uint64_t>(Ap);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at)), hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at >> 32));
    return reinterpret_cast<LeanArgPtr>((static_cast<uint64_t>(hi) << 32) | lo);
}
template <bool KEPT>  // (KEPT: the build that can write the kept-set dump)
__device__ __noinline__ __attribute__((not_tail_called)) void three_pass_row(LeanArgPtr Ap, const uint32_t row_) {
    const uint32_t row = __builtin_amdgcn_readfirstlane(row_);
    const BatchArgs& A = *(const BatchArgs*)wave_args(Ap);
    sample_row<false, false, KEPT, true>(A, row);
    __syncthreads();  // (the row's flags are written by whichever thread finished it)
    if (threadIdx.x == 0) A.flags[row] |= kRouteHandedBack;
}

// A row whose cut or draw falls among more tokens than a list holds: answered by the exact path as the three-pass code would have it done, from the sweep's maximum and normaliser
// and with the touched tokens' tables that the sweep has left. (Logits in steps of 0.5, us, by way of the
// three-pass code and straight: 64 rows of 262144 at top-p 0.9 1157 / 1030, at 0.6 1072 / 947, a lone one 806 / 682; without the sweep in vain, as they were before this kernel took rows of that
// length, 954 and 692 at top-p 0.6.)
__device__ __noinline__ __attribute__((not_tail_called)) void exact_left_row(LeanArgPtr Ap_, const uint32_t row_, __attribute__((address_space(3))) LeanShared* S) {
    const LeanArgPtr Ap = wave_args(Ap_);
    const uint32_t row = __builtin_amdgcn_readfirstlane(row_);
    const BatchArgs& A = *(const BatchArgs*)Ap;
    const LeanRowParams P = load_row_params(A, row, Ap);
    ExactIn in;
    in.base = static_cast<const unsigned char*>(A.logits) + static_cast<size_t>(row) * A.row_stride * 4u;
    in.allow = A.allow ? A.allow + static_cast<size_t>(row) * A.allow_stride : nullptr;
    in.V = A.vocab;
    in.dtype = 0;
    in.touched_at = __builtin_amdgcn_readfirstlane(S->touched_left) ? A.lds_ab : 0xffffffffu;
    in.m = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(S->m_left)));
    in.inv_t = P.inv_t;
    in.top_k = in.n1_asked = 0u;
    in.top_p = P.top_p;
    in.min_p = P.min_p;
    in.u = batch_uniform(A.rng, P.seed, row, P.step, 0);
    in.rbase = 0ull;
    in.mode = (P.top_p < 1.0 ? 4u : 0u) | (P.min_p > 0.0 ? 8u : 0u);
    const float m = in.m, z = static_cast<float>(S->z_left);
    const ExactOut out = exact_row(in);
    if (threadIdx.x == 0) {
        A.token[row] = out.token;
        A.flags[row] = kRouteHandedBack | kRouteExact | (out.mg_top_p < A.tol ? kNearTopP : 0u) | (out.mg_min_p < A.tol ? kNearMinP : 0u) | (out.mg_draw < A.tol ? kNearDraw : 0u);
        if (A.prob) A.prob[row] = static_cast<float>(out.ptok);
        if (A.n_kept) A.n_kept[row] = out.n3;
        if (A.stats) {
            A.stats[2 * row] = m;
            A.stats[2 * row + 1] = z;
        }
        if (A.margin) {
            A.margin[3 * row] = out.mg_top_p;
            A.margin[3 * row + 1] = out.mg_min_p;
            A.margin[3 * row + 2] = out.mg_draw;
        }
    }
}

// What lean_row has left of a row. (A function of its own, as above: as a loop around that code in the kernel it cost the kernel some hundred spilled registers.)
template <bool MASKED, int NREG>
__device__ __noinline__ __attribute__((not_tail_called)) void lean_rest(LeanArgPtr Ap_, const uint32_t row_, __attribute__((address_space(3))) LeanShared* S) {
    LeanArgPtr Ap = wave_args(Ap_);
    const uint32_t row = __builtin_amdgcn_readfirstlane(row_);
    float top = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(S->top)));
    if (top < INFINITY) {
        if (lean_row<MASKED, true, NREG>(*(const BatchArgs*)Ap, Ap, row, *(LeanShared*)S)) return;
        __syncthreads();
        top = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(S->top)));
    }
    bool ties = top == INFINITY;  // uniform
    if (ties) {
        // Tied or flat rows. The three-pass code would count the row once more, to find that its list does not hold the tokens either: its bins lie elsewhere, but what
        // one bin has too many of it has as well, and half as many again of several bins are taken to be too many for both.
        auto found = [&](uint32_t search) {  // the first wave's record that holds a bin
            LeanBinRec r;
            r.b = 0xffffffffu;
            r.c = 0u;
            r.cex = 0u;
            for (uint32_t w = 0; w < WS_WAVES && r.b == 0xffffffffu; ++w) {
                r.b = S->rec[search * WS_WAVES + w].b;
                r.cex = S->rec[search * WS_WAVES + w].cex;
                r.c = S->rec[search * WS_WAVES + w].c;
            }
            return r;
        };
        const LeanBinRec dlo = found(2u), dhi = found(3u);
        uint32_t most = max(dlo.c, dhi.c);
        if (S->sel.topp_in_list) {
            LeanBinRec cut = found(0u);
            if (cut.b != 0xffffffffu && cut.cex >= 16384u) cut = found(1u);
            if (cut.b != 0xffffffffu) most = max(most, cut.c);
        }
        ties = dlo.b != 0xffffffffu && dhi.b != 0xffffffffu && dhi.b >= dlo.b && S->sel.r0hi < kLeanTail && (most > kLeanMaxList || S->sel.n_r0 + S->sel.n_r1 > kLeanMaxList + kLeanMaxList / 2u);
        ties = __builtin_amdgcn_readfirstlane(ties ? 1 : 0) != 0;
    }
    if (ties) exact_left_row(Ap, row, S);
    else three_pass_row<false>(Ap, row);
}

// MASKED: the batch has an allow mask (a kernel of its own: one build carrying both paths spilled far more registers)
template <bool MASKED, int NREG>
__global__ void __launch_bounds__(WS_BLOCK) lean_batch_kernel(BatchArgs A) {
    __shared__ LeanShared shared;
    const uint32_t row = blockIdx.x;
    if (lean_row<MASKED, false, NREG>(A, nullptr, row, shared)) return;
    __syncthreads();  // whatever the lean path left in LDS is dead
    LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    lean_rest<MASKED, (NREG <= 40 ? 40 : 64)>(Ap, row, (__attribute__((address_space(3))) LeanShared*)&shared);  // (one for all shorter rows: few are swept twice)
}

}  // namespace ws
