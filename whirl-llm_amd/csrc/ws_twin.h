// The short-list sampler (ws_short.h) for batches of more rows than compute units: 512 threads a row and tables small enough that a compute
// unit holds two rows.
//
// What bounds it: memory while rows are swept, and nothing while they are not. 1024 threads with a unit to themselves took 177K clocks
// for a row of 262144 tokens, a tenth of them allowed, with a history of 8192 and a top-k of 1000, 80K of them without a sweep: the tables, the
// threshold, the sort, the rules. Here a unit's other row sweeps in the meantime, as far as the two are not at the same place (they start together);
// a row of a small vocabulary is all such stretches, and two of them are at work instead of one. Microseconds, ws_short.h and this: 1024 rows as above 389 / 323
// (280 since ws_common.h's search of bias lists), without history 266 / 239; top-k 50, 1000-id histories: 512 of 151936 83.8 / 73.3, 300 of 151936 77.2 / 63.9, 1000 of 50257 108 / 72.9, 1000 of 8000
// 55.9 / 38.1; min-p alone, 1000 of 151936 149 / 139. (1024 of 262144 with a top-k of 50: 195, 5.5 TB/s.)
//
// While both rows sweep, the vector instructions of a unit are all in use (with the loads aimed at eight chunks in L2 a sweep took 84 us of the 91), so
// what a listed token costs counts: 1850 of a row are one in five vectors out of six. A wave takes its places in the list thirty-two at a time, writes
// logit and id as they are, and keeps its count in a scalar register (an atomic addition and its answer a token, the key made on the spot: 278 -> 270 us for
// the rows above); the entries of a history that a mask rules out are looked at once (270 -> 253 with the registers below, 247 without a
// spilled one): the sample's masked-out tokens become NaN in place, so that the mask's words are done with before the row is asked for. 512 rows of 151936, min-p
// alone 108.8 -> 98.2, 300 of 262144 with a top-k of 1000 106.2 -> 101.2, 1000 bf16 rows of 12288 with a top-k of 200 52.3 -> 49.0, 300 of 151936 with a top-k of 300 and 4096 ids 86.5 -> 81.8.
//
// Against ws_short.h the touched tokens come before the sweep, not behind it: their tables are dead when it begins and can lie where the list
// will be. A history entry's count, a token's bias marks and its claim are 16 bits, not 48: a token is claimed by clearing its word, and where a bias entry
// names it only those claim it, so that nobody has to look the entry up. Rows for which a check fails are marked in `flags`, and a
// kernel launched behind this one gives them to the three-pass code, which needs a unit's whole LDS.
// Tried and dropped: the workgroups of half the rows started later (no faster at any delay up to 80K clocks); all batches asked for before the threshold, or
// the ids before the sample (both within 1 %); the mask's words kept in registers for the second use (spills: 339 us against 330).
#pragma once
#include "ws_short.h"

namespace ws {

constexpr uint32_t kTwinHead = 8u;  // vectors a thread of the sample that the threshold is fitted to
constexpr uint32_t kTwinEmpty = 0xffffffffu;  // in the place of an id
constexpr uint32_t kTwinPlaces = 32u;  // places of the list a wave takes at a time, where the list has kTwinSpare places more than the tokens it may hold
static_assert((kTwinPlaces - 1u) * WS_WAVES <= kTwinSpare && kTwinSpare <= 64u * WS_WAVES, "room for the places that are taken and not filled; a thread each to close them");

// LDS: the list at 0 (32 KiB; first the sample's bin counts), the bitmap of the touched tokens at lds_ab, and at lds_cnt its 16-bit popcount
// prefixes and a 16-bit word per rank: history count | kBias | kBiases. These two are dead when the sweep begins, and where a second
// row would not fit beside them they lie in the upper part of the list's place.
// Returns false when the row has to go to the three-pass code (uniform over the workgroup; nothing has been written for it).
template <int DT, bool MASKED>
__device__ __forceinline__ bool twin_row(const BatchArgs& A, const uint32_t row, ShortShared& S) {
#ifdef WS_SHORT_TIMERS
    const long long wss_t0 = clock64();
    if (threadIdx.x == 0) S.marks[13] = 0.f;
#endif
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr uint32_t TPV = DT == 0 ? 4u : 8u;  // tokens in a 128-bit vector
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    const uint32_t V = A.vocab, nW = (V + 31u) >> 5;
    const unsigned char* base = static_cast<const unsigned char*>(A.logits) + static_cast<size_t>(row) * A.row_stride * (DT == 0 ? 4u : 2u);
    const uint32_t* allow = MASKED ? A.allow + static_cast<size_t>(row) * A.allow_stride : nullptr;

    uint64_t* list = reinterpret_cast<uint64_t*>(lds);
    uint32_t* head_cnt = reinterpret_cast<uint32_t*>(lds);
    uint32_t* touched = reinterpret_cast<uint32_t*>(lds + A.lds_ab);
    uint32_t* invalid = touched;  // (what it holds from the sweep on)
    uint16_t* wprefix = reinterpret_cast<uint16_t*>(lds + A.lds_cnt);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(lds + A.lds_cnt + ((nW * 2u + 3u) & ~3u));  // two ranks a word
    const uint32_t spare = min(kTwinSpare, (A.lds_ab >> 3) - kShortCap);  // places behind the list's
    const uint32_t early_slots = A.lds_cnt < A.lds_ab ? min(kShortCap, A.lds_cnt >> 3) : kShortCap;  // of the list, while the tables are needed

    // The row: chunks of a vector a thread, whole ones and at most one that is not, and a few tokens behind the last vector
    const uint32_t nv = V / TPV, n_odd = V % TPV, n_full = nv / WS_BLOCK;
    auto vector_at = [&](uint32_t j) __attribute__((always_inline)) {
        const LooseVec v = *reinterpret_cast<const LooseVec*>(base + min(j, nv - 1u) * 16u);
        return make_uint4(v.x, v.y, v.z, v.w);
    };
    auto word_at = [&](uint32_t j) __attribute__((always_inline)) { return (min(j, nv - 1u) * TPV) >> 5; };

    // The sample: 8 of the row's chunks of a vector a thread, evenly spread over it (a vocabulary's first ids are its frequent tokens).
    const uint32_t spread = max(1u, n_full / kTwinHead);
    uint4 hq[kTwinHead];
    uint32_t hna[kTwinHead];
#pragma unroll
    for (uint32_t k = 0; k < kTwinHead; ++k) {
        const uint32_t j = k * spread * WS_BLOCK + t;
        hq[k] = vector_at(j);
        hna[k] = MASKED ? allow[word_at(j)] : 0xffffffffu;
    }
    // the list's place takes the bin counts first; all tables are cleared while the parameters travel
    reinterpret_cast<uint4*>(head_cnt)[t] = make_uint4(0u, 0u, 0u, 0u);
    static_assert(kTwinBins == 4u * WS_BLOCK, "");
    if (A.hist || A.bias_ids) {
        for (uint32_t w = t; w < nW; w += WS_BLOCK) touched[w] = 0u;
        for (uint32_t r = t; r < (A.patch_cap + 1u) >> 1; r += WS_BLOCK) cnt[r] = 0u;
    }
    const LeanRowParams P = load_row_params(A, row);
    WSS_MARK(0);  // parameters in
    const float inv_t = P.inv_t;
    const uint32_t top_k = P.top_k, nh = P.nh, nb = P.nb, n_all = nh + nb;
    const double top_p = P.top_p, min_p = P.min_p;
    const bool by_k = top_k >= 1u && top_k <= kShortMaxK && top_k <= V;  // the top_k largest decide
    const bool by_p = top_k == 0u && min_p > 0.0 && min_p <= 1.0;      // no top-k: what the min-p floor lets through decides
    constexpr uint32_t kBias = 0x4000u, kBiases = 0x8000u;  // a bias entry names the token, a second one does
    if (!(by_k || by_p) || !(inv_t > 0.f) || n_all > A.patch_cap || nh >= kBias) return false;
    const int32_t* hist_ids = A.hist + P.h0;
    const int32_t* bias_ids = A.bias_ids + P.b0;
    const float* bias_vals = A.bias_vals + P.b0;

    // The history and bias ids, one sequence, stay in registers (9 rounds: 4608 of them) until their tokens have been taken. They are asked for behind
    // the sample, which does not have to know the parameters first.
    constexpr uint32_t kIds = 9u, kMore = 4u;
    uint32_t ids[kIds];
    auto entry = [&](uint32_t j) __attribute__((always_inline)) {  // (unconditional, as all these loads: one behind a branch makes the compiler wait for every load before it)
        const int32_t* at = j < nh ? hist_ids + j : (j < n_all ? bias_ids + (j - nh) : reinterpret_cast<const int32_t*>(A.seed));
        const uint32_t id = static_cast<uint32_t>(*at);
        return j < n_all ? id : 0xffffffffu;
    };
#pragma unroll
    for (uint32_t k = 0; k < kIds; ++k) {
        ids[k] = 0xffffffffu;
        if (k * WS_BLOCK < n_all) ids[k] = entry(k * WS_BLOCK + t);  // uniform
    }
    constexpr uint32_t kWords = 16u;  // words a thread of the allow mask (262144 tokens) in registers
    uint32_t aw[kWords];
    if (MASKED && n_all) {
#pragma unroll
        for (uint32_t k = 0; k < kWords; ++k) aw[k] = allow[min(k * WS_BLOCK + t, nW - 1u)];
    }

    // a listed entry: its id, and the number of a bias entry plus one
    constexpr uint32_t kFew = 4u, kFewShift = 20u, kFewId = (1u << kFewShift) - 1u, kFewBias = (1u << (32u - kFewShift)) - 1u;
    static_assert(kWords * WS_BLOCK * 32u <= kFewId, "an id of a row that is listed, and none that is 0xffffffff");
    const uint32_t few_room = MASKED ? min(kFew * WS_BLOCK, (early_slots * 8u - kTwinBins * 4u) / 4u) : 0u;
    uint32_t n_few = 0xffffffffu;
    const bool long_lists = MASKED && n_all > kFew * WS_BLOCK;  // uniform: more entries than the listed ones' rounds take as they are
    if (long_lists) {  // the tokens the mask allows: most rows' are few
        uint32_t allowed = 0;
#pragma unroll
        for (uint32_t k = 0; k < kWords; ++k) allowed += k * WS_BLOCK + t < nW ? static_cast<uint32_t>(__popc(aw[k])) : 0u;
        allowed = wave_sum(allowed);
        if (lane == 0u) S.red_u[wv] = allowed;
        if (t == 0u) S.s_w[4] = 0u;
    }

    // the other whole chunks in order
    uint32_t c_next = spread == 1u ? kTwinHead : 1u, c_skip = spread == 1u ? 0xffffffffu : spread;
    auto next_chunk = [&]() __attribute__((always_inline)) {
        const uint32_t c = c_next++;
        if (c_next == c_skip) {
            ++c_next;
            c_skip = c_skip + spread < kTwinHead * spread ? c_skip + spread : 0xffffffffu;
        }
        return c;
    };

    // ---- the bitmap of the touched tokens (of a masked row those that its mask allows: the others count nowhere), their ranks, history
    // counts and bias entries
    __syncthreads();  // (the tables are cleared)
    // a touched token's rank, or none (an id outside of the vocabulary, a token that is masked out)
    auto rank = [&](uint32_t id) __attribute__((always_inline)) {
        if (id >= V) return 0xffffffffu;
        const uint32_t w = touched[id >> 5], b = id & 31u;
        if (MASKED && !((w >> b) & 1u)) return 0xffffffffu;
        return static_cast<uint32_t>(wprefix[id >> 5]) + __popc(w & ((1u << b) - 1u));
    };
    if (n_all) {
        auto mark = [&](uint32_t id) {
            if (id < V) atomicOr(&touched[id >> 5], 1u << (id & 31u));
        };
        // entries beyond those in registers, some at a time
        auto others = [&](auto&& what) {
            for (uint32_t j0 = kIds * WS_BLOCK; j0 < n_all; j0 += kMore * WS_BLOCK) {
                uint32_t id[kMore];
#pragma unroll
                for (uint32_t k = 0; k < kMore; ++k) id[k] = entry(j0 + k * WS_BLOCK + t);
#pragma unroll
                for (uint32_t k = 0; k < kMore; ++k) what(id[k], j0 + k * WS_BLOCK + t);
            }
        };
        // Of a masked row only the entries that its mask allows are gone on with - the mask where the bitmap will be, the entries listed behind the
        // sample's counts, then in registers -, if they are few enough for it. (Nine in ten of 8692 masked out: 17 entries a thread, each looked up in
        // three passes, were 25 us of a row's 125.) Lists of up to four entries a thread are as fast without: 257 rows of 10496 with 606 ids took 18.7 us and 20.0 by
        // the list, 700 of 13952 with 32 bias entries 31 and 33.
        bool by_list = false;
        if (long_lists) {
            uint32_t n_allowed = 0;
#pragma unroll
            for (uint32_t w = 0; w < WS_WAVES; ++w) n_allowed += S.red_u[w];
            // (a row may have more bias entries than the number has room for: only history and bias list together are bounded by the launch's tables)
            by_list = nW <= kWords * WS_BLOCK && nb <= kFewBias && static_cast<float>(n_allowed) * static_cast<float>(n_all) * 1.1f + 64.f * static_cast<float>(V) < static_cast<float>(V) * static_cast<float>(few_room);  // uniform
        }
        if (MASKED && by_list) {
#pragma unroll
            for (uint32_t k = 0; k < kWords; ++k)
                if (k * WS_BLOCK + t < nW) touched[k * WS_BLOCK + t] = aw[k];
            __syncthreads();
            uint32_t* listed = head_cnt + kTwinBins;
            auto list_allowed = [&](auto n, auto&& id_of, uint32_t j0) __attribute__((always_inline)) {
                constexpr uint32_t N = decltype(n)::value;
                uint32_t word[N], all = 0;
                uint64_t on[N];
#pragma unroll
                for (uint32_t k = 0; k < N; ++k) word[k] = touched[min(id_of(k), V - 1u) >> 5] >> (id_of(k) & 31u);
#pragma unroll
                for (uint32_t k = 0; k < N; ++k) {
                    on[k] = __ballot(id_of(k) < V && (word[k] & 1u));
                    all += static_cast<uint32_t>(__popcll(on[k]));
                }
                uint32_t from = 0;
                if (lane == 0u && all) from = atomicAdd(&S.s_w[4], all);
                from = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(from)));
#pragma unroll
                for (uint32_t k = 0; k < N; ++k) {
                    const uint32_t at = from + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(on[k] >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(on[k]), 0u));
                    const uint32_t j = j0 + k * WS_BLOCK + t;
                    if (id_of(k) < V && (word[k] & 1u) && at < few_room) listed[at] = id_of(k) | (j < nh ? 0u : (j - nh + 1u) << kFewShift);
                    from += static_cast<uint32_t>(__popcll(on[k]));
                }
            };
            uint32_t next[kMore];
#pragma unroll
            for (uint32_t k = 0; k < kMore; ++k) next[k] = entry((kIds + k) * WS_BLOCK + t);
            constexpr uint32_t kThird = kIds / 3u;
#pragma unroll
            for (uint32_t h = 0; h < 3u; ++h)
                if (h * kThird * WS_BLOCK < n_all) list_allowed(std::integral_constant<uint32_t, kThird>{}, [&](uint32_t k) { return ids[h * kThird + k]; }, h * kThird * WS_BLOCK);  // uniform
            for (uint32_t j0 = kIds * WS_BLOCK; j0 < n_all; j0 += kMore * WS_BLOCK) {
                uint32_t id[kMore];
#pragma unroll
                for (uint32_t k = 0; k < kMore; ++k) {
                    id[k] = next[k];
                    next[k] = entry(j0 + (kMore + k) * WS_BLOCK + t);
                }
                list_allowed(std::integral_constant<uint32_t, kMore>{}, [&](uint32_t k) { return id[k]; }, j0);
            }
            __syncthreads();
            n_few = S.s_w[4];
            if (n_few <= few_room) {  // uniform
#pragma unroll
                for (uint32_t k = 0; k < kFew; ++k) ids[k] = k * WS_BLOCK + t < n_few ? listed[k * WS_BLOCK + t] : 0xffffffffu;
            }
            for (uint32_t w = t; w < nW; w += WS_BLOCK) touched[w] = 0u;
            __syncthreads();
        }
        if (MASKED && n_few <= few_room) {  // uniform
#pragma unroll
            for (uint32_t k = 0; k < kFew; ++k)
                if (k * WS_BLOCK < n_few) mark(ids[k] & kFewId);
            __syncthreads();
        } else {
#pragma unroll
            for (uint32_t k = 0; k < kIds; ++k)
                if (k * WS_BLOCK < n_all) mark(ids[k]);  // uniform
            others([&](uint32_t id, uint32_t) { mark(id); });
            __syncthreads();
            if (MASKED) {
#pragma unroll
                for (uint32_t k = 0; k < kWords; ++k)
                    if (k * WS_BLOCK + t < nW) touched[k * WS_BLOCK + t] &= aw[k];
                for (uint32_t w = kWords * WS_BLOCK + t; w < nW; w += WS_BLOCK) touched[w] &= allow[w];
                __syncthreads();
            }
        }
        {  // popcount prefixes: an odd number of consecutive words a thread (no two lanes of a read in one bank)
            const uint32_t per = ((nW + WS_BLOCK - 1u) / WS_BLOCK) | 1u, w0 = min(t * per, nW), w1 = min(w0 + per, nW);
            uint32_t local = 0, total;
            for (uint32_t w = w0; w < w1; ++w) local += __popc(touched[w]);
            uint32_t run = block_excl_scan(local, S.red_u, &total);
            for (uint32_t w = w0; w < w1; ++w) {
                wprefix[w] = static_cast<uint16_t>(run);
                run += __popc(touched[w]);
            }
        }
        __syncthreads();
        auto count = [&](uint32_t id, uint32_t j) {
            const uint32_t r = rank(id), sh = (r & 1u) * 16u;
            if (r == 0xffffffffu) return;
            if (j < nh) atomicAdd(&cnt[r >> 1], 1u << sh);
            else if ((atomicOr(&cnt[r >> 1], kBias << sh) >> sh) & kBias) atomicOr(&cnt[r >> 1], kBiases << sh);
        };
        if (n_few <= few_room) {  // uniform
#pragma unroll
            for (uint32_t k = 0; k < kFew; ++k)
                if (k * WS_BLOCK < n_few) count(ids[k] & kFewId, ids[k] <= kFewId ? 0u : nh);  // uniform
        } else {
#pragma unroll
            for (uint32_t k = 0; k < kIds; ++k)
                if (k * WS_BLOCK < n_all) count(ids[k], k * WS_BLOCK + t);  // uniform
            others(count);
        }
    }
    WSS_MARK(1);  // bitmap done
    // one vector: its tokens as floats, masked-out / touched / NaN ones as -inf
    auto unpack = [&](uint4 q, uint32_t na, uint32_t j, float (&x)[TPV]) {
        const uint32_t i0 = j * TPV;
        uint32_t invalid = 0u;  // bit e: token e does not count here
        if (MASKED) invalid = ~(na >> (i0 & 31u));
        if (n_all) invalid |= touched[i0 >> 5] >> (i0 & 31u);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (uint32_t e = 0; e < TPV; ++e) {
            uint32_t bits = DT == 0 ? w[e] : ((e & 1u) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
            bits |= static_cast<uint32_t>(static_cast<int32_t>(invalid << (31u - e)) >> 31);  // -> NaN
            x[e] = fmaxf(__uint_as_float(bits), -INFINITY);
        }
    };

    // The sample without the tokens that do not count: they become NaN where they are, and the mask's words need no registers from here on.
    auto values = [&](const uint4& q, float (&x)[TPV]) __attribute__((always_inline)) {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (uint32_t e = 0; e < TPV; ++e)
            x[e] = fmaxf(__uint_as_float(DT == 0 ? w[e] : ((e & 1u) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16))), -INFINITY);
    };
    if (MASKED || n_all) {
#pragma unroll
        for (uint32_t k = 0; k < kTwinHead; ++k) {
            if (k * spread * WS_BLOCK >= nv) break;  // uniform
            const uint32_t i0 = min(k * spread * WS_BLOCK + t, nv - 1u) * TPV;
            uint32_t invalid = 0u;  // bit e: token e does not count here
            if (MASKED) invalid = ~(hna[k] >> (i0 & 31u));
            if (n_all) invalid |= touched[i0 >> 5] >> (i0 & 31u);
            auto gone = [&](uint32_t e) { return static_cast<uint32_t>(static_cast<int32_t>(invalid << (31u - e)) >> 31); };
            uint32_t* w = &hq[k].x;
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) w[e] |= DT == 0 ? gone(e) : (gone(2u * e) & 0xffffu) | (gone(2u * e + 1u) << 16);
        }
    }

    // The first two batches behind the sample travel while the threshold is worked out. (A whole chunk's address is the
    // same register for every thread and a lane's offset: nothing to add or to clamp a vector.)
    constexpr uint32_t KB = 4;  // vectors a thread and batch, two batches in flight
    uint4 qa[KB], qb[KB], q_part;
    uint32_t ca[KB], cb[KB];
    const uint32_t my_offset = (n_full ? t : min(t, nv - 1u)) * 16u;
    auto load = [&](uint4 (&q)[KB], uint32_t (&c)[KB]) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t k = 0; k < KB; ++k) {
            c[k] = next_chunk();
            const LooseVec v = *reinterpret_cast<const LooseVec*>(base + static_cast<size_t>(min(c[k], max(n_full, 1u) - 1u)) * (WS_BLOCK * 16u) + my_offset);
            q[k] = make_uint4(v.x, v.y, v.z, v.w);
        }
    };
    load(qa, ca);

    // ---- the threshold: the sample's logits counted in 2048 bins of 1/32 e-fold below the sample's maximum
    float ref = -INFINITY;
    {
        float x[TPV];
#pragma unroll
        for (uint32_t k = 0; k < kTwinHead; ++k) {
            const uint32_t j = k * spread * WS_BLOCK + t;
            if (j < nv) {
                values(hq[k], x);
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e) ref = fmaxf(ref, x[e]);
            }
        }
        ref = block_max(ref, S.red_f);
    }
    if (!(ref > -INFINITY)) return false;  // (a sample without any token)
    const float c32 = inv_t * 32.f;
    float thr = -INFINITY;  // tokens above it are listed
    const bool whole = nv <= kTwinHead * WS_BLOCK;  // the sample is the row
    const uint32_t n_sample = whole ? V : kTwinHead * WS_BLOCK * TPV;
    // Tokens to list: of the row's top_k the sample holds about top_k * n_sample / V, give or take the root of that; the rank in the
    // sample that the threshold is read off lies six such roots above, half of top_k and 150 tokens of the row at least. (A sample that
    // is the row: the count is exact but for the tokens of a bin, and twice top_k will do.)
    uint32_t want = 2u * top_k + 6u;
    if (!whole) {
        const float roots = 6.f * __builtin_sqrtf(static_cast<float>(top_k) * static_cast<float>(V) / static_cast<float>(n_sample));
        want = top_k + max(max(top_k >> 1, 150u), static_cast<uint32_t>(roots)) + 16u;
    }
    bool list_all = by_k && whole && want >= V;
    if (by_p) thr = __fadd_rn(ref, __fdiv_rn(static_cast<float>(log(min_p)) - 0.02f, inv_t));  // (0.02 e-folds below the floor: roundings)
    if (by_k && !list_all) {
        // rank in the sample that about `want` tokens of the row lie above
        const uint64_t r_star64 = (static_cast<uint64_t>(n_sample) * want + V - 1u) / V;
        const uint32_t r_star = static_cast<uint32_t>(r_star64 < 4u ? 4u : r_star64);
        uint32_t still = r_star;
        float top = ref;
        if (t == 0) S.s_w[0] = 0xffffffffu;  // (the bin, once found; the barrier behind the counting publishes this)
        // whether the bin is among those counted
        auto found = [&]() __attribute__((always_inline)) {
            __syncthreads();
            constexpr uint32_t PER = kTwinBins / WS_BLOCK;
            uint32_t c[PER], mine = 0;
#pragma unroll
            for (uint32_t k = 0; k < PER; k += 4u) {
                const uint4 c4 = *reinterpret_cast<const uint4*>(&head_cnt[PER * t + k]);
                c[k] = c4.x;
                c[k + 1u] = c4.y;
                c[k + 2u] = c4.z;
                c[k + 3u] = c4.w;
                mine += c4.x + c4.y + c4.z + c4.w;
            }
            uint32_t total;
            const uint32_t before = block_excl_scan(mine, S.red_u, &total);
            if (before < still && before + mine >= still) {  // the bin in which the sample's r_star-th largest lies
                uint32_t run = before, b = PER * t;
#pragma unroll
                for (uint32_t k = 0; k < PER; ++k) {
                    if (run < still && run + c[k] >= still) b = PER * t + k;
                    run += c[k];
                }
                S.s_w[0] = b;
            }
            __syncthreads();
            return total;
        };
        // The bins near the top are all that matters: first only the tokens within 8 e-folds of the sample's maximum are counted - an LDS
        // atomic each, and a sixth of the tokens -, the others only when those turn out to be fewer than r_star.
        // (what is 64 e-folds down - and masked-out tokens, nine in ten of some rows - is not counted: a wave's additions to one
        // word would queue up sixty-four deep)
        constexpr float kNear = 256.f, kFar = 2047.f;
        uint32_t total = 0;
        for (int round = 0; round < 2; ++round) {  // uniform
            float x[TPV];
#pragma unroll
            for (uint32_t k = 0; k < kTwinHead; ++k) {
                const uint32_t j = k * spread * WS_BLOCK + t;
                if (j < nv) {
                    values(hq[k], x);
#pragma unroll
                    for (uint32_t e = 0; e < TPV; ++e) {
                        const float d = fminf(__fmul_rn(__fsub_rn(top, x[e]), c32), kFar);
                        if (round == 0 ? d < kNear : (d >= kNear && d < kFar)) atomicAdd(&head_cnt[static_cast<uint32_t>(d)], 1u);
                    }
                }
            }
            total = found();
            if (S.s_w[0] != 0xffffffffu) break;
        }
        // A row whose largest tokens lie further above the others (a cold one): from the largest of those once more. (The sample is read again:
        // there are no registers for another copy of the loop above.)
        for (int more = 0; more < 4 && S.s_w[0] == 0xffffffffu; ++more) {  // uniform
            still -= total;
            float below = -INFINITY, x[TPV];
#pragma unroll 1
            for (uint32_t k = 0; k < kTwinHead; ++k) {
                const uint32_t j = k * spread * WS_BLOCK + t;
                if (j >= nv) break;
                unpack(vector_at(j), MASKED ? allow[word_at(j)] : 0xffffffffu, j, x);
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e) below = __fmul_rn(__fsub_rn(top, x[e]), c32) >= kFar ? fmaxf(below, x[e]) : below;
            }
            reinterpret_cast<uint4*>(head_cnt)[t] = make_uint4(0u, 0u, 0u, 0u);
            top = block_max(below, S.red_f);
            if (!(top > -INFINITY)) break;
#pragma unroll 1
            for (uint32_t k = 0; k < kTwinHead; ++k) {
                const uint32_t j = k * spread * WS_BLOCK + t;
                if (j >= nv) break;
                unpack(vector_at(j), MASKED ? allow[word_at(j)] : 0xffffffffu, j, x);
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e) {
                    const float d = __fmul_rn(__fsub_rn(top, x[e]), c32);
                    if (d >= 0.f && d < kFar) atomicAdd(&head_cnt[static_cast<uint32_t>(d)], 1u);
                }
            }
            total = found();
        }
        const uint32_t b_star = S.s_w[0];
        if (b_star == 0xffffffffu) list_all = true;  // (fewer than r_star tokens in the sample: everything is listed)
        else thr = __fsub_rn(top, __fdiv_rn(static_cast<float>(b_star + 1u), c32));
    }
    if (list_all) thr = -INFINITY;
    if (t == 0) {
        S.s_w[1] = 0u;  // tokens listed
        S.s_w[2] = 0u;  // the touched tokens did not fit
        S.s_w[3] = 0u;  // how many they are
    }
    __syncthreads();  // (the counts and the bin have been read: the list takes the counts' place)
    WSS_MARK(2);  // threshold known
    load(qb, cb);
    const double k2_d = static_cast<double>(inv_t) * 1.44269504088896340736;
    const float k2 = static_cast<float>(k2_d), k2lo = static_cast<float>(k2_d - static_cast<double>(k2));
    float m = -INFINITY, s0 = 0.f, s1 = 0.f;  // the largest token listed; two sums, of the tokens of even and of odd places (a thread has V / 512)
    auto term = [&](float x) {
        const float a = fmaxf(__fsub_rn(x, ref), -1e30f);
        return __builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2));  // (v_exp_f32: arguments below -126 give 0, which is what they are worth)
    };
    auto push = [&](float x, uint32_t id, bool yes, bool early = false) {  // (one LDS atomic a listed token: they are few)
        if (yes) {
            m = fmaxf(m, x);
            const uint32_t slot = atomicAdd(&S.s_w[1], 1u);
            if (slot < (early ? early_slots : kShortCap + spare)) list[slot] = (static_cast<uint64_t>(__float_as_uint(x)) << 32) | id;
            else if (early) S.s_w[2] = 1u;
            if (early) atomicAdd(&S.s_w[3], 1u);
        }
    };

    // (The list takes tokens as they are, logit and id; the sort's keys are made of them behind the sweep, all lanes at work.)
    // ---- the touched tokens: their adjusted logits (bias entries in list order, then repetition, then frequency / presence, as
    // ws_sample.h applies them), into the sum and - above the threshold - the list. A token is taken by the entry that finds its word there
    // and clears it: a bias entry where one names it, else one of its history.
    if (n_all) {
        // (j_of: an entry's number; of a listed one that of a bias entry behind nh, or 0)
        auto take_touched = [&](auto n, auto&& id_of, auto&& j_of, uint32_t j0, uint32_t n_of) __attribute__((always_inline)) {
            constexpr uint32_t N = decltype(n)::value;
            uint32_t word[N];
            float raw[N];
#pragma unroll
            for (uint32_t k = 0; k < N; ++k) {
                word[k] = 0u;
                if (j0 + k * WS_BLOCK >= n_of) continue;  // uniform
                const uint32_t r = rank(id_of(k)), sh = (r & 1u) * 16u;
                if (r == 0xffffffffu) continue;
                if (j_of(k) < nh && ((cnt[r >> 1] >> sh) & kBias)) continue;
                word[k] = (atomicAnd(&cnt[r >> 1], ~(0xffffu << sh)) >> sh) & 0xffffu;
            }
#pragma unroll
            for (uint32_t k = 0; k < N; ++k) {
                raw[k] = -INFINITY;
                if (word[k]) raw[k] = DT == 0 ? reinterpret_cast<const float*>(base)[id_of(k)] : bf16_to_f32(reinterpret_cast<const uint16_t*>(base)[id_of(k)]);
            }
#pragma unroll
            for (uint32_t k = 0; k < N; ++k) {
                if (j0 + k * WS_BLOCK >= n_of) continue;  // uniform
                float x = fmaxf(raw[k], -INFINITY);
                const bool several = (word[k] & kBiases) != 0u;
                if ((word[k] & kBias) && !several) x = __fadd_rn(x, bias_vals[j_of(k) - nh]);
                // (from the first of them; all lanes, which share the search: the few with an allowed token alone took 5 us)
                if (__ballot(several)) x = add_other_bias(several, id_of(k), 0xffffffffu, x, bias_ids, bias_vals, nb);
                if (word[k]) {
                    const uint32_t c = word[k] & (kBias - 1u);
                    if (c) {
                        x = x > 0.f ? __fdiv_rn(x, P.rep) : __fmul_rn(x, P.rep);
                        x = __fsub_rn(x, __fadd_rn(__fmul_rn(P.freq, static_cast<float>(c)), P.pres));
                    }
                    x = fmaxf(x, -INFINITY);
                    s0 += term(x);
                }
                push(x, id_of(k), word[k] && x > thr, true);
            }
        };
        if (MASKED && n_few <= few_room) {  // uniform
            take_touched(std::integral_constant<uint32_t, kFew>{}, [&](uint32_t k) { return ids[k] & kFewId; },
                         [&](uint32_t k) { return ids[k] <= kFewId ? 0u : nh + (ids[k] >> kFewShift) - 1u; }, 0u, n_few);
        } else {
            constexpr uint32_t kThird = kIds / 3u;
#pragma unroll
            for (uint32_t h = 0; h < 3u; ++h)
                if (h * kThird * WS_BLOCK < n_all)
                    take_touched(std::integral_constant<uint32_t, kThird>{}, [&](uint32_t k) { return ids[h * kThird + k]; },
                                 [&](uint32_t k) { return (h * kThird + k) * WS_BLOCK + t; }, h * kThird * WS_BLOCK, n_all);
            for (uint32_t j0 = kIds * WS_BLOCK; j0 < n_all; j0 += kMore * WS_BLOCK) {
                uint32_t id[kMore];
#pragma unroll
                for (uint32_t k = 0; k < kMore; ++k) id[k] = entry(j0 + k * WS_BLOCK + t);
                take_touched(std::integral_constant<uint32_t, kMore>{}, [&](uint32_t k) { return id[k]; }, [&](uint32_t k) { return j0 + k * WS_BLOCK + t; }, j0, n_all);
            }
        }
        __syncthreads();  // (the tables are done with: the list may take their place)
    }
    // from here on the bitmap says which tokens do not count
    if (MASKED) {  // (the mask is read again: its words have no registers to stay in)
        for (uint32_t w = t; w < nW; w += WS_BLOCK) invalid[w] = ~allow[w] | (n_all ? invalid[w] : 0u);
        __syncthreads();
    }
    q_part = vector_at(n_full * WS_BLOCK + t);
    // ---- the sweep: sum of exp, tokens above the threshold to the list
    const bool mapped = MASKED || n_all != 0u;  // uniform
    // A wave lists its tokens at places that it takes thirty-two of at a time, so that most vectors need no word of the other waves; the few
    // places left over at the end are filled from the list's end. What is taken and not filled - one place less than that a wave, at most - has to
    // fit beside a full list: fewer at a time where there is no such room (rows of 370000 tokens and more, two a unit). 300 rows of 100000, us, with a list of
    // 4096 tokens: top-k 97.9, min-p 99.3 (a place a token 110 and 112; what is not filled counted against the list 236, handed back, and 134, read twice).
    const uint32_t places = min(kTwinPlaces, spare / WS_WAVES + 1u);  // uniform
    uint32_t my_next = 0, my_end = 0;  // uniform
    float my_thr = thr;
    auto wave_value = [](uint32_t v) __attribute__((always_inline)) { return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v))); };
    const float thr_a = __fsub_rn(thr, ref);  // (rounding is monotonous: x > thr makes x - ref, rounded, no smaller than this)
    auto take = [&](const uint4& q, uint32_t word, uint32_t shift, uint32_t i0) __attribute__((always_inline)) {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        float x[TPV], highest = -1e30f;
        word >>= shift;
#pragma unroll
        for (uint32_t e = 0; e < TPV; ++e) {
            uint32_t bits = DT == 0 ? w[e] : ((e & 1u) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
            if (mapped) bits |= static_cast<uint32_t>(static_cast<int32_t>(word << (31u - e)) >> 31);  // -> NaN
            x[e] = __uint_as_float(bits);
            const float a = fmaxf(__fsub_rn(x[e], ref), -1e30f);  // (NaN as well: 0 in the sum; and never above `thr` below)
            highest = fmaxf(highest, a);
            (e & 1u ? s1 : s0) += __builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2));
        }
        if (__ballot(highest >= thr_a)) {  // uniform: a vector that may have a token for the list
            uint64_t on[TPV];
            uint32_t n = 0;
            float top = x[0];
#pragma unroll
            for (uint32_t e = 0; e < TPV; ++e) {
                on[e] = __ballot(x[e] > my_thr);
                n += static_cast<uint32_t>(__popcll(on[e]));
                if (e) top = fmaxf(top, x[e]);
            }
            m = fmaxf(m, top);  // (whatever of it is not listed lies below what is)
            auto list_at = [&](auto&& at) __attribute__((always_inline)) {
                uint32_t i = 0;  // uniform
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e) {
                    if (x[e] > my_thr) {
                        const uint32_t k = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(on[e] >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(on[e]), 0u));
                        uint32_t* to = reinterpret_cast<uint32_t*>(list) + 2u * at(k, i);
                        to[0] = i0 + e;
                        to[1] = __float_as_uint(x[e]);
                    }
                    i += static_cast<uint32_t>(__popcll(on[e]));
                }
            };
            if (n <= my_end - my_next) {  // uniform
                list_at([&](uint32_t k, uint32_t i) { return k + (my_next + i); });
                my_next = wave_value(my_next + n);
            } else {  // the rest of the wave's places, then new ones
                const uint32_t left = my_end - my_next, more = max(n - left, places);
                uint32_t from = 0;
                if (lane == 0u) from = atomicAdd(&S.s_w[1], more);
                from = wave_value(from);
                if (from + more > kShortCap + spare) {
                    my_thr = INFINITY;  // (more tokens than the list may hold: nothing more to it)
                } else {
                    list_at([&](uint32_t k, uint32_t i) { return k + i < left ? k + i + my_next : k + i + (from - left); });
                    my_next = wave_value(from + (n - left));
                    my_end = wave_value(from + more);
                }
            }
        }
    };
    auto take_at = [&](uint4 q, uint32_t j) __attribute__((always_inline)) {  // (every lane of a wave: those past the row bring NaN)
        if (j >= nv) q = make_uint4(0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu);
        take(q, mapped ? invalid[(min(j, nv - 1u) * TPV) >> 5] : 0u, (j * TPV) & 31u, j * TPV);
    };
#pragma unroll
    for (uint32_t k = 0; k < kTwinHead; ++k) {
        uint32_t j0 = k * spread * WS_BLOCK;
        asm volatile("" : "+s"(j0));  // (so that no vector's place in the bitmap waits in a register since the vector was asked for)
        if (j0 < nv) take_at(hq[k], j0 + t);  // uniform
    }
    const uint32_t my_word = (t * TPV) >> 5, my_shift = (t * TPV) & 31u;
    auto eat = [&](const uint4 (&q)[KB], const uint32_t (&c)[KB]) __attribute__((always_inline)) {
        uint32_t word[KB];
#pragma unroll
        for (uint32_t k = 0; k < KB; ++k) word[k] = mapped ? invalid[min(c[k], n_full - 1u) * (WS_BLOCK * TPV / 32u) + my_word] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < KB; ++k)
            if (c[k] < n_full) take(q[k], word[k], my_shift, (c[k] * WS_BLOCK + t) * TPV);  // uniform
    };
    for (uint32_t i = kTwinHead; i < n_full; i += 2u * KB) {
        eat(qa, ca);
        load(qa, ca);
        eat(qb, cb);
        load(qb, cb);
    }
    if (!whole && n_full * WS_BLOCK < nv) take_at(q_part, n_full * WS_BLOCK + t);  // uniform
    if (n_odd) {  // uniform: the tokens behind the last whole vector
        float x = -INFINITY;
        const uint32_t id = nv * TPV + t;
        if (t < n_odd && !(mapped && ((invalid[id >> 5] >> (id & 31u)) & 1u)))
            x = fmaxf(DT == 0 ? reinterpret_cast<const float*>(base)[id] : bf16_to_f32(reinterpret_cast<const uint16_t*>(base)[id]), -INFINITY);
        if (t < n_odd) s0 += term(x);
        push(x, id, t < n_odd && x > thr);
    }
    WSS_MARK(4);  // sweep done
#ifdef WS_SHORT_TIMERS
    if (lane == 0u) atomicMax(reinterpret_cast<int*>(&S.marks[13]), __float_as_int(static_cast<float>(clock64() - wss_t0)));  // the slowest wave's
#endif
    double z;  // the sum against `ref`
    uint64_t my_token;  // what lies at the thread's own place of the list
    uint32_t n_list, no_room;
    {          // the block's maximum and sum with one barrier between them
        const float wm_ = wave_max(m);
        const double ws_ = wave_sum(static_cast<double>(s0) + static_cast<double>(s1));
        if (lane < my_end - my_next) reinterpret_cast<uint32_t*>(list)[2u * (my_next + lane)] = kTwinEmpty;
        if (lane == 0u) {  // (words that nobody has looked at since the threshold's barriers)
            S.red_f[wv] = wm_;
            S.red_d[wv] = ws_;
            S.bstart[wv] = my_next;
            S.bcnt[wv] = my_end - my_next;
        }
        __syncthreads();
        my_token = list[t];
        n_list = S.s_w[1];
        no_room = S.s_w[2];
        m = S.red_f[0];
        z = S.red_d[0];
#pragma unroll
        for (uint32_t w = 1; w < WS_WAVES; ++w) {
            m = fmaxf(m, S.red_f[w]);
            z += S.red_d[w];
        }
    }
    WSS_MARK(5);
    auto as_key = [](uint64_t token) __attribute__((always_inline)) { return key64(__uint_as_float(static_cast<uint32_t>(token >> 32)), static_cast<uint32_t>(token)); };
    // Few places, most of them empty as a rule (a confident row's, with a min-p alone): a place a thread, and what is filled moves up, as a key. (us, a place a token / the
    // way below / this: 300 rows of 10292, Zipfian, min-p 0.03, 13.5 / 14.4 / 14.0; 512 bf16 rows of 12452 with 34 ids 16.6 / 18.9 / 17.8; 400 of 16320 14.5 / 16.2 / 15.7. Places taken one at
    // a time at first, or moved by the wave that has filled them: slower where lists are longer, 400 of 35044 39.3 / 41.4.)
    const bool few_places = n_list <= WS_BLOCK;  // uniform
    if (few_places) {
        const bool filled = t < n_list && static_cast<uint32_t>(my_token) != kTwinEmpty;
        const uint64_t on = __ballot(filled);
        if (lane == 0u) S.red_u[wv] = static_cast<uint32_t>(__popcll(on));
        __syncthreads();
        uint32_t at = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(on >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(on), 0u));
        n_list = 0;
#pragma unroll
        for (uint32_t w = 0; w < WS_WAVES; ++w) {
            const uint32_t n = S.red_u[w];
            at += w < wv ? n : 0u;
            n_list += n;
        }
        if (filled) list[at] = as_key(my_token);
        __syncthreads();
    } else {  // the places no wave has filled: the last n_left of the list take their contents to the others
        uint32_t n_left = 0;
#pragma unroll
        for (uint32_t w = 0; w < WS_WAVES; ++w) n_left += S.bcnt[w];
        if (n_list <= kShortCap + spare && n_left) {  // uniform
            n_list -= n_left;
            // (a wave has 64 of them; one wave for all of them took 1 us longer)
            const uint32_t first = n_list + wv * 64u, from = first + lane;
            if (wv * 64u < n_left) {  // uniform
                bool filled = wv * 64u + lane < n_left;
                uint32_t r = wv * 64u;  // how many of the waves before have contents
#pragma unroll
                for (uint32_t w = 0; w < WS_WAVES; ++w) {
                    const uint32_t at = S.bstart[w], end = at + S.bcnt[w];
                    filled = filled && !(from >= at && from < end);
                    r -= max(min(end, first), n_list) - min(max(at, n_list), max(min(end, first), n_list));
                }
                const uint64_t on = __ballot(filled);
                r += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(on >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(on), 0u));
                uint32_t to = from;
#pragma unroll
                for (uint32_t w = 0; w < WS_WAVES; ++w) {  // the r-th place that lies below the list's end
                    const uint32_t at = S.bstart[w], n = at < n_list ? min(S.bcnt[w], n_list - at) : 0u;
                    if (r < n) to = at + r;
                    r = r < n ? 0xffffffffu : r - n;
                }
                if (filled) list[to] = list[from];
            }
            __syncthreads();
        }
    }
    if (by_p && n_list > kShortCap) {
        // A min-p row whose sample's maximum lies well below its own: the floor is known now, and the row is read once more, for the list alone.
        // (All of it, not what lies above the list's lowest: a row's sum has been taken. Of 65 rows of 50257 3 came this way.)
        double floor_ = min_p;
        asm volatile("" : "+v"(floor_));  // (so that nothing of its logarithm waits in registers from the threshold on)
        thr = fmaxf(thr, __fadd_rn(m, __fdiv_rn(static_cast<float>(log(floor_)) - 0.02f, inv_t)));
        __syncthreads();
        if (t == 0) S.s_w[1] = S.s_w[3];
        __syncthreads();
        auto list_from = [&](uint32_t id, uint32_t bits, bool there) {
            const float x = fmaxf(__uint_as_float(bits), -INFINITY);
            push(x, id, there && x > thr && !(mapped && ((invalid[id >> 5] >> (id & 31u)) & 1u)));
        };
        for (uint32_t j0 = t; j0 < nv; j0 += 4u * WS_BLOCK) {
            uint4 q[4];
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) q[k] = vector_at(j0 + k * WS_BLOCK);
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) {
                const uint32_t w[4] = {q[k].x, q[k].y, q[k].z, q[k].w}, j = j0 + k * WS_BLOCK;
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e)
                    list_from(j * TPV + e, DT == 0 ? w[e] : ((e & 1u) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16)), j < nv);
            }
        }
        if (t < n_odd)
            list_from(nv * TPV + t, DT == 0 ? reinterpret_cast<const uint32_t*>(base)[nv * TPV + t] : static_cast<uint32_t>(reinterpret_cast<const uint16_t*>(base)[nv * TPV + t]) << 16, true);
        __syncthreads();
        n_list = S.s_w[1];
    }
    const uint32_t n_cand = by_k ? top_k : n_list;  // candidates the rules look at
    if (no_room != 0u || n_list > kShortCap || !(m > -INFINITY) || !(__fsub_rn(m, ref) * inv_t < 80.f) || n_list < n_cand || n_cand == 0u) return false;
    if (!few_places) {  // uniform
        for (uint32_t k = t; k < n_list; k += WS_BLOCK) list[k] = as_key(list[k]);
        if (n_list <= WS_BLOCK / 4u) __syncthreads();  // (the sort of a short list begins with other threads' keys; a longer list's with a thread's own)
    }
    float inv_t_ = inv_t;
    asm volatile("" : "+v"(inv_t_));  // (so that its 64-bit value does not wait in registers from the sweep on)
    // Tokens above `ref` can be most of the sum, and the larger the exponent, the less of a fraction 32 bits leave it (1.2e-6 of
    // the normaliser where the maximum lies 60 units above the sample's; 2e-7 up to the four units below which nothing is done):
    // they are all on the list, and their terms are taken out and put back in 64 bits.
    if (__fsub_rn(m, ref) * inv_t > 4.f) {  // uniform
        double more = 0.0;
        for (uint32_t k = t; k < n_list; k += WS_BLOCK) {
            const float x = unkey32(static_cast<uint32_t>(list[k] >> 32));
            if (x > ref) more += exp((static_cast<double>(x) - static_cast<double>(ref)) * static_cast<double>(inv_t_)) - static_cast<double>(term(x));
        }
        z += block_sum(more, S.red_d);
    }
    auto rules_of = [&]() __attribute__((always_inline)) {
        ShortRow R;
        R.top_p = top_p;
        R.min_p = min_p;
        R.u = batch_uniform(A.rng, P.seed, row, P.step, 0);
        R.z = z * exp((static_cast<double>(ref) - static_cast<double>(m)) * static_cast<double>(inv_t_));
        R.inv_t = inv_t_;
        R.m = m;
        R.n_cand = n_cand;
        R.by_k = by_k;
        return R;
    };
    // A wide top-k, two candidates a thread and more: its cuts and draw without an order (us, with the sort and without, top-k 1000: 1024 masked rows of 262144 248 / 243, 300
    // of 262144 91.9 / 88.6, 512 of 151936 74.6 / 71.2, 1000 of 32000 67.9 / 63.7; level at a top-k of 100 to 500, and rows with a min-p alone, whose keys crowd at the floor, slower: 86.7 / 95.4).
    // Rows with a bucket too full for it are sorted after all: of fp32 logits that were bf16 once 512 rows of 151936, nearly all of which have one, take 84.9 / 85.8, 300 of 262144,
    // half of which have, 102.6 / 103.2, 1024 masked ones, few of which have, 260 / 247.
    ShortSpan span;
    const LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    if (DT == 0 && by_k && n_cand > WS_BLOCK && n_list <= kShortCap - 1024u && !Ap->kept_ids && !Ap->entropy && !Ap->query_prob) {  // uniform
        const ShortRow R = rules_of();
        if (t == 0u) S.s_d[7] = R.z;
        __syncthreads();  // (the words that say which places were left over have been read as well)
        if (short_pick(list, n_list, row, R, S, span)) return true;
        __syncthreads();
    }
    short_sort(list, n_list, m, S, span);
    WSS_MARK(6);  // sorted
    // the k-th largest has to lie above the threshold (below it, the sweep has left out tokens that rank before it); a min-p row's
    // threshold lies below its floor by construction
    const float x_k = unkey32(static_cast<uint32_t>(list[n_cand - 1u] >> 32));
    if ((by_k && !(x_k > thr)) || !(x_k > -INFINITY)) return false;
    short_rules(list, row, rules_of(), S);
#ifdef WS_SHORT_TIMERS
    WSS_MARK(8);
    __syncthreads();
    if (t < 16 && A.kept_logits) A.kept_logits[static_cast<size_t>(row) * A.kept_cap + 100u + t] = t == 15 ? static_cast<float>(n_list) : S.marks[t];
#endif
    return true;
}

// (two workgroups a compute unit are four waves a SIMD: 128 registers)
template <int DT, bool MASKED>
__global__ void __launch_bounds__(WS_BLOCK) __attribute__((amdgpu_waves_per_eu(4, 4))) twin_batch_kernel(BatchArgs A) {
    __shared__ ShortShared shared;
    if (!twin_row<DT, MASKED>(A, blockIdx.x, shared) && threadIdx.x == 0) A.flags[blockIdx.x] = kTwinRest;
}

}  // namespace ws
