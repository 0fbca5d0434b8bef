// The sampler for few rows: every row is shared by up to sixteen workgroups, each of which keeps its share of the row in
// registers. It takes the rows the short-list kernel (ws_short.h) takes - a top-k of at most kShortMaxK, or no top-k but a
// min-p - and ends with the same sort and rules.
//
// With few rows nothing streams: 600 KB over sixteen compute units are 3 us of loads, and what counts is the chain of
// dependent steps. Against the short-list kernel's shared rows, whose workgroups met over a histogram of the head each,
// this one is built to make that chain short:
//   * the eight waves of a workgroup work on their own until they publish: a wave's threshold is the d-th largest of its
//     64 lanes' maxima (ballots, no barrier, no histogram), its list and its sum of exp go straight from registers to the
//     row's workspace. A row of P parts is 8 P wave shares;
//   * the vectors of a row are dealt to the waves in chunks of eight lanes, so that tokens that are large together - the
//     low ids of a vocabulary - end up in different waves' lists;
//   * history counts are 16-bit words indexed by the token's place in the share (no ranks, no prefix sums): two barriers;
//     a touched token's logit is asked for as soon as its id is known;
//   * the part that arrives last - a ticket, nobody waits - reads the waves' headers and lists. With top_k at most the
//     number of waves, the top_k-th largest of the waves' maxima bounds the row's top_k-th largest logit from below, so
//     that about as many keys as top_k are left to sort.
//   * a row's parts are on one chiplet where its compute units take all parts of its rows at once (few_place).
// What bounds it is that chain: parameters, ids, their tokens' logits, the stores of the keys, headers and keys are six trips to
// memory, between them some 1100 instructions of the average wave (582 vector, 538 scalar; the last part's do more); with 64 rows and more the instructions a token, which two waves a SIMD
// issue one after the other. 512 threads rather than 1024: the cost of a wave's own
// work (threshold, sums, publishing) is paid half as often, and a share still fits the registers. Measured against the
// short-list kernel's shared rows (151936 fp32, microseconds a launch): one row, top-k 40: 20.6 -> 11.9; 64 rows of mixed
// filters with 4096-id histories: 50 (126 when a row's min-p list ran over) -> 32.5; 32 rows of 50257, which went through
// the three-pass kernel: 55.6 -> 15.4. Since then 11.8 -> 9.9, 31.6 -> 28.4 and 15.6 -> 14.3: a bit a token for those that lists name and a look a vector
// for those to list (64 rows 8 %, 40 rows 12 %), the waves' maxima and thresholds by a third of the instructions, the last part's exponentials by a quarter,
// its places in the list by one addition a wave (one row 9 %), and a row's parts on one chiplet (1 to 2 %; 6 % of a row whose parameters come over the bus).
#pragma once
#include "ws_short.h"

namespace ws {

constexpr uint32_t kFewWaves = kFewMaxParts * WS_WAVES;
// Workspace of a row: kFewKeys keys, slot by slot with one key a wave in each, then what every wave says of its share -
// {maximum, threshold} as order keys; the sum of exp against the maximum; how many keys it has listed, kFewBad when it could not
// list them -, then {parts arrived, largest logit so far as an order key}. Zero-filled between launches.
constexpr uint32_t kFewHead = kFewKeys * 8u, kFewCount = kFewHead + kFewWaves * 16u, kFewCtrl = kFewCount + kFewWaves * 4u;
static_assert(kFewCtrl + 256u <= 64512u && 64512u < kFewRowBytes, "a row's workspace (debug builds put their clocks at 64512)");
constexpr uint32_t kFewBad = 0xffffffffu;
constexpr uint32_t kFewExt = 2048u;  // touched tokens of a share
constexpr uint32_t kFewDup = 0x4000u, kFewTaken = 0x8000u;  // in a token's 16-bit word, above its history count: a second bias entry, somebody takes it
constexpr uint32_t kFewDups = 64u;  // bias entries of tokens that another entry has taken

#ifdef WS_SHORT_TIMERS  // (debug builds: clocks since the kernel began, at the unused end of the row's workspace)
#define WSF_MARK(k) \
    if (threadIdx.x == 0) reinterpret_cast<long long*>(work + 64512)[k] = clock64() - F.t0
#else
#define WSF_MARK(k)
#endif
struct FewShared {
#ifdef WS_SHORT_TIMERS
    long long t0;
#endif
    ShortShared sh;
    uint16_t dup_at[kFewDups], dup_j[kFewDups];  // (places of a share and entries of a bias list: below 2^16)
    float dup_v[kFewDups];
    float red_f[WS_WAVES];  // (few_collect: the row's maximum, and the lowest logit looked at)
    uint32_t w[16];
    double u, z[kFewWaves / 64u];  // (z: the row's normaliser, in as many summands)
    __device__ __forceinline__ double sum() const {
        double all = z[0];
#pragma unroll
        for (uint32_t i = 1; i < kFewWaves / 64u; ++i) all += z[i];
        return all;
    }
};

// the largest prefix (bits 31 .. 14) of an order key that at least d lanes of the wave reach; top: the largest key. Five instructions a bit (two bits a step
// are fifteen, and no shorter a chain); the first eight bits are those of the top, or one octave below, as a rule.
__device__ __forceinline__ uint32_t few_lane_threshold(uint32_t k32, uint32_t top, uint32_t d) {
    auto reached = [&](uint32_t c) { return static_cast<uint32_t>(__popcll(__ballot(k32 >= c))) >= d; };
    const uint32_t near = (top & 0xff000000u);
    uint32_t at = 0u;
    if (reached(near)) {  // uniform
        at = near;
    } else {
#pragma unroll
        for (int b = 31; b >= 24; --b) at = reached(at | (1u << b)) ? at | (1u << b) : at;
    }
#pragma unroll
    for (int b = 23; b >= 14; --b) at = reached(at | (1u << b)) ? at | (1u << b) : at;
    return at;
}
__device__ __forceinline__ uint32_t lanes_before(uint64_t m) {  // set bits of m below this lane
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
}

// Which row a workgroup has, and which part of it; false: none. Workgroups go to the chiplets in turn, so parts whose numbers lie
// kChiplets apart share one, and its L2: what they leave for each other need not go through memory.
__device__ __forceinline__ bool few_place(uint32_t together, uint32_t rows, uint32_t& row, uint32_t& part) {
    row = blockIdx.y;
    part = blockIdx.x;
    if (together) {
        row = row * kChiplets + part % kChiplets;
        part /= kChiplets;
    }
    return row < rows;
}
// What a workgroup of a shared row is given: which share of the row is its own, and how the row is dealt out. Chunk c of the
// row (2^cl vectors) is wave c mod G's; vector k of a lane lies in its wave's chunk number k * (chunks a load) + lane / (lanes a
// chunk).
struct FewShare {
    uint32_t parts, part, G, g, cl, V, nv, n_vec, slots;  // G: waves a row, g: this one, nv: vectors of the row, n_vec: of a lane, slots: keys a wave can list
    template <int DT>
    __device__ __forceinline__ static FewShare of(uint32_t V, uint32_t parts, uint32_t part, uint32_t cl, uint32_t n_vec, uint32_t slots) {
        constexpr uint32_t TPV = DT == 0 ? 4u : 8u;
        FewShare L;
        L.parts = parts;
        L.part = part;
        L.G = parts * WS_WAVES;
        L.g = part * WS_WAVES + static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
        L.cl = cl;
        L.V = V;
        L.nv = (V + TPV - 1u) / TPV;
        L.slots = slots;
        L.n_vec = n_vec;
        return L;
    }
    __device__ __forceinline__ uint32_t vec_of(uint32_t k) const {
        const uint32_t lane = threadIdx.x & 63u;
        return ((((k << (6u - cl)) + (lane >> cl)) * G + g) << cl) + (lane & ((1u << cl) - 1u));
    }
};
// What is wanted of the row: its top_k largest logits, or everything within min_p of its largest
struct FewWant {
    bool by_k, by_p;
    uint32_t top_k;
    float inv_t;
    double min_p;
};
__device__ __forceinline__ void few_exp_scale(float inv_t, float& k2, float& k2lo) {  // exp(a inv_t) = 2^(a k2 + a k2lo)
    k2 = inv_t * 1.44269504088896340736f;
    k2lo = static_cast<float>(static_cast<double>(inv_t) * 1.44269504088896340736 - static_cast<double>(k2));
}

// A logit as it stands in a row, a signalling NaN made a quiet one; the largest of three such (NaN: not among them). Written out: of bits that
// could be a signalling NaN the compiler would quiet every operand of every maximum.
__device__ __forceinline__ float few_logit(uint32_t bits) {
    float v;
    asm("v_max_f32 %0, %1, %1" : "=v"(v) : "v"(bits));
    return v;
}
__device__ __forceinline__ float few_max3(float a, float b, float c) {
    float v;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(v) : "v"(a), "v"(b), "v"(c));
    return v;
}
template <uint32_t TPV>
__device__ __forceinline__ float few_max_of(const float (&x)[TPV]) {
    float v = few_max3(x[0], x[1], x[2]);
#pragma unroll
    for (uint32_t e = 3; e + 1u < TPV; e += 2u) v = few_max3(v, x[e], x[e + 1u]);
    return few_max3(v, x[TPV - 1u], x[TPV - 1u]);
}

// Threshold, list and sum of every wave of this workgroup, published in the row's workspace. x: the share in registers (NaN or -inf:
// no token), vm: the largest of each vector, lm: this thread's largest logit, ext: n_ext more tokens {id, logit}; ok false: the share cannot be listed. SUM
// false: nobody asks for the normaliser. Returns whether this workgroup is the last of the row's: it has everything to go on.
template <int DT, int NV, bool SUM>
__device__ __forceinline__ bool few_publish(const FewShare& L, const FewWant& W, const float (&x)[NV][DT == 0 ? 4 : 8], const float (&vm)[NV], float lm, const uint4* ext, uint32_t n_ext,
                                            bool ok, unsigned char* work, FewShared& F) {
    constexpr uint32_t TPV = DT == 0 ? 4u : 8u;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    const uint32_t slots = L.slots;
    const float wm = wave_max(lm);
    unsigned long long* gkeys = reinterpret_cast<unsigned long long*>(work);
    unsigned long long* ghead = reinterpret_cast<unsigned long long*>(work + kFewHead);
    uint32_t* gcount = reinterpret_cast<uint32_t*>(work + kFewCount);
    uint32_t* ctrl = reinterpret_cast<uint32_t*>(work + kFewCtrl);

    WSF_MARK(1);
    // ---- the threshold
    float thr = -INFINITY;  // this wave lists its tokens from here up
    if (W.by_k) {
        // A wave has top_k / G of the row's top_k largest on average; two more and five times the scatter of that number
        // are listed, d of them in different lanes.
        const float lambda = static_cast<float>(W.top_k) * __builtin_amdgcn_rcpf(static_cast<float>(L.G));
        const uint32_t want = static_cast<uint32_t>(lambda + 5.f * __builtin_amdgcn_sqrtf(lambda) + 2.f) + 1u;
        const uint32_t d = min(60u, want <= 20u ? want : 20u + (want - 20u) / 2u);
        const uint32_t at = few_lane_threshold(key32(lm), key32(wm), d);
        thr = at > 0x007fffffu ? unkey32(at) : -INFINITY;  // (below that prefix: -inf and the NaN patterns under it)
    } else if (W.by_p) {
        // what the floor lets through lies within -ln(min_p) / W.inv_t of the row's maximum: of the largest logit any part
        // has reported so far, or this part's (0.02 units of the exponent below: roundings)
        if (lane == 0u) F.red_f[wv] = wm;
        __syncthreads();
        float top = F.red_f[0];
#pragma unroll
        for (uint32_t w = 1; w < WS_WAVES; ++w) top = fmaxf(top, F.red_f[w]);
        if (t == 0) {
            __hip_atomic_fetch_max(&ctrl[1], key32(top), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            F.w[8] = __hip_atomic_load(&ctrl[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        top = fmaxf(top, unkey32(F.w[8]));
        if (top > -INFINITY) thr = __fadd_rn(top, __fdiv_rn(static_cast<float>(log(W.min_p)) - 0.02f, W.inv_t));
    }

    WSF_MARK(2);
    // ---- the sum of exp against the wave's maximum, and the list
    float k2, k2lo;
    few_exp_scale(W.inv_t, k2, k2lo);
    const float ref = wm > -INFINITY ? wm : 0.f;
    float s = 0.f;
    auto add = [&](float v) {
        const float a = fmaxf(__fsub_rn(v, ref), -1e30f);
        s += __builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2));
    };
    uint32_t n_list = 0;  // uniform
    const float thr_list = fmaxf(thr, -3.402823466e38f);  // (-inf is no token)
    auto push = [&](float v, uint32_t id) {
        const bool yes = v >= thr_list;
        const uint64_t m = __ballot(yes);
        if (m) {  // uniform
            const uint32_t slot = n_list + lanes_before(m);
            if (yes && slot < slots) __hip_atomic_store(&gkeys[slot * L.G + L.g], key64(v, id), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            n_list += static_cast<uint32_t>(__popcll(m));
        }
    };
    if (ok && wm < INFINITY) {
        // (a look a vector, and at its tokens only where one of them is listed)
#pragma unroll
        for (uint32_t k = 0; k < NV; ++k)
            if (k < L.n_vec && __ballot(vm[k] >= thr_list)) {  // uniform
                const uint32_t id0 = L.vec_of(k) * TPV;
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e) push(x[k][e], id0 + e);
            }
        for (uint32_t i0 = 0; i0 < n_ext; i0 += WS_BLOCK) {  // uniform
            uint2 en = make_uint2(0u, 0xff800000u);
            if (i0 + t < n_ext) en = *reinterpret_cast<const uint2*>(&ext[i0 + t]);
            push(__uint_as_float(en.y), en.x);
            if (SUM) add(__uint_as_float(en.y));
        }
        if (SUM)
#pragma unroll
            for (uint32_t k = 0; k < NV; ++k)
                if (k < L.n_vec) {  // uniform
                    asm volatile("");  // (a branch: else the vectors a share does not have are summed and dropped)
#pragma unroll
                    for (uint32_t e = 0; e < TPV; ++e) add(x[k][e]);
                }
    }
    {
        const double z = wm > -INFINITY && wm < INFINITY ? wave_sum(static_cast<double>(s)) : 0.0;
        if (lane == 0u) {
            __hip_atomic_store(&ghead[L.g], (static_cast<unsigned long long>(key32(wm)) << 32) | key32(thr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&ghead[kFewWaves + L.g], static_cast<unsigned long long>(__double_as_longlong(z)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&gcount[L.g], !ok || !(wm < INFINITY) || n_list > slots ? kFewBad : n_list, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // What the parts exchange is written and read by device-scope atomic accesses, which go past this unit's caches, and a wave
    // waits until its stores have been acknowledged: whoever draws the last ticket finds every word and key of the row, and what it
    // clears stays clear. (Without the wait a key could come after the last part had cleared its place, and the next launch would
    // have taken it for its own. The wait costs 0.3 us, and reading once instead of again and again gives most of it back: one
    // row 11.75 -> 11.88 us, 64 rows of mixed filters 32.5 -> 32.3.)
    WSF_MARK(3);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // every wave's stores have arrived
    WSF_MARK(4);
    if (t == 0) F.w[2] = __hip_atomic_fetch_add(&ctrl[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    WSF_MARK(5);
    return F.w[2] == L.parts - 1u;
}

// The last part: everybody's keys from the larger of the waves' thresholds up - or from a higher bound of the row's top_k-th
// largest logit - to `list` (LDS, kShortCap keys), in no order; F.red_f[0] and F.sum(): the row's maximum and normaliser. Every place of
// the workspace is zero again afterwards. Returns the number of keys (which may be more than the list holds); 0 when a share could not be listed.
// fourth(): work of the caller's for the fourth wave, while others read the headers.
template <bool SUM, class FOURTH>
__device__ __forceinline__ uint32_t few_collect(const FewShare& L, const FewWant& W, unsigned char* work, FewShared& F, uint64_t* list, FOURTH&& fourth) {
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    unsigned long long* gkeys = reinterpret_cast<unsigned long long*>(work);
    unsigned long long* ghead = reinterpret_cast<unsigned long long*>(work + kFewHead);
    uint32_t* gcount = reinterpret_cast<uint32_t*>(work + kFewCount);
    uint32_t* ctrl = reinterpret_cast<uint32_t*>(work + kFewCtrl);
    const uint32_t G = L.G, slots = L.slots;
    // Headers and everybody's keys asked for (those of the first slots right away). Five waves read the headers side by side, each
    // for what it works out: the threshold, the normaliser (two of them: the exponentials are the longest chain here, and one a
    // lane is 0.1 us shorter than two), how many slots hold keys; and one the uniform.
    constexpr uint32_t kBlind = 4096u / WS_BLOCK, kHL = kFewWaves / 64u;
    static_assert(kHL == 2u, "a wave of this part for every 64 of the row");
    const uint32_t w0 = min(lane, G - 1u), w1 = min(64u + lane, G - 1u);
    const bool on0 = lane < G, on1 = 64u + lane < G;
    uint64_t h0 = 0ull, h1 = 0ull, zs = 0ull;
    uint32_t n0 = 0u, n1 = 0u;
    if (wv < 5u) {
        h0 = __hip_atomic_load(&ghead[w0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        h1 = __hip_atomic_load(&ghead[w1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (SUM && (wv == 1u || wv == 4u)) zs = __hip_atomic_load(&ghead[kFewWaves + (wv == 4u ? w1 : w0)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (wv == 2u) {
            n0 = __hip_atomic_load(&gcount[w0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            n1 = __hip_atomic_load(&gcount[w1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    uint64_t got[kBlind];
#pragma unroll
    for (uint32_t i = 0; i < kBlind; ++i) got[i] = __hip_atomic_load(&gkeys[i * WS_BLOCK + t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t == 0) F.w[5] = 0u;  // keys taken
    if (wv == 3u) {
        fourth();
    } else if (wv < 5u) {
        const float m0 = on0 ? unkey32(static_cast<uint32_t>(h0 >> 32)) : -INFINITY, m1 = on1 ? unkey32(static_cast<uint32_t>(h1 >> 32)) : -INFINITY;
        const float mx = wave_max(fmaxf(m0, m1));
        if (wv == 0u) {
            // the keys that are looked at: from the largest of the waves' thresholds up (every wave has listed what it has
            // there), or - higher - from the top_k-th largest of the waves' maxima
            float floor_v = wave_max(fmaxf(unkey32(static_cast<uint32_t>(h0)), unkey32(static_cast<uint32_t>(h1))));
            if (W.by_k && W.top_k <= G) {
                float lo = floor_v, hi = mx;
                auto reach = [&](float v) { return static_cast<uint32_t>(__popcll(__ballot(m0 >= v)) + __popcll(__ballot(m1 >= v))); };
                if (lo > -INFINITY && reach(lo) >= W.top_k)
#pragma unroll
                    for (int i = 0; i < 9; ++i) {
                        const float mid = 0.5f * lo + 0.5f * hi;
                        const bool enough = reach(mid) >= W.top_k;
                        lo = enough ? mid : lo;
                        hi = enough ? hi : mid;
                    }
                floor_v = lo;
            }
            if (W.by_p) floor_v = __fadd_rn(mx, __fdiv_rn(static_cast<float>(log(W.min_p)) - 0.02f, W.inv_t));
            if (lane == 0u) {
                F.red_f[0] = mx;
                F.red_f[1] = floor_v;
            }
        } else if (wv == 2u) {
            const bool bad = __ballot((on0 && n0 == kFewBad) || (on1 && n1 == kFewBad)) != 0ull || !(mx > -INFINITY);
            const uint32_t most = wave_max_u32(max(on0 ? n0 : 0u, on1 ? n1 : 0u));
            if (lane == 0u) {
                F.w[3] = bad ? slots : most;  // (a wave that could not list its share may have left keys in every slot)
                F.w[4] = bad ? 1u : 0u;
            }
        } else {
            double z = 0.0;
            if (SUM) {  // (the factors in 64 bits, as the rules work out the candidates' masses)
                const float own = wv == 4u ? m1 : m0;
                if (own > -INFINITY) z = __longlong_as_double(static_cast<long long>(zs)) * exp_down(static_cast<double>(__fsub_rn(mx, own)) * static_cast<double>(W.inv_t));
                z = wave_sum(z);
            }
            if (lane == 0u) F.z[wv == 4u ? 1u : 0u] = z;
        }
    }
    __syncthreads();
    WSF_MARK(6);
    const uint32_t floor_key = max(key32(F.red_f[1]), 1u);  // (no key: zeros)
    const uint32_t n_read = F.w[3] * G;
    const bool bad = F.w[4] != 0u;
    // (a wave's places in the list by one addition for all the slots it has read)
    auto keep = [&](const uint64_t (&key)[kBlind], uint32_t i0) __attribute__((always_inline)) {
        uint32_t mine = 0;
#pragma unroll
        for (uint32_t i = 0; i < kBlind; ++i) mine += i0 + i * WS_BLOCK < n_read && static_cast<uint32_t>(key[i] >> 32) >= floor_key ? 1u : 0u;
        const uint32_t inc = wave_incl_scan(mine), all = lane_value(inc, 63u);
        if (all) {  // uniform
            uint32_t slot = 0;
            if (lane == 0u) slot = lds_add(&F.w[5], all);
            slot = lane_value(slot, 0u) + inc - mine;
#pragma unroll
            for (uint32_t i = 0; i < kBlind; ++i)
                if (i0 + i * WS_BLOCK < n_read && static_cast<uint32_t>(key[i] >> 32) >= floor_key) {
                    if (slot < kShortCap) list[slot] = key[i];
                    ++slot;
                }
        }
    };
    keep(got, 0u);
    for (uint32_t i0 = kBlind * WS_BLOCK; i0 < n_read; i0 += kBlind * WS_BLOCK) {  // uniform
        uint64_t more[kBlind];
#pragma unroll
        for (uint32_t i = 0; i < kBlind; ++i) {
            const uint32_t at = i0 + i * WS_BLOCK + t;
            more[i] = at < n_read ? __hip_atomic_load(&gkeys[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        }
        keep(more, i0);
#pragma unroll
        for (uint32_t i = 0; i < kBlind; ++i)
            if (more[i] != 0ull) __hip_atomic_store(&gkeys[i0 + i * WS_BLOCK + t], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // the workspace as the next launch needs it, all zeros (cleared behind the sort instead, rows with long lists took 2 % longer and lone rows 1 % less)
#pragma unroll
    for (uint32_t i = 0; i < kBlind; ++i)
        if (i * WS_BLOCK < n_read && got[i] != 0ull) __hip_atomic_store(&gkeys[i * WS_BLOCK + t], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t < G) {
        __hip_atomic_store(&ghead[t], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ghead[kFewWaves + t], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&gcount[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (t < 2u) __hip_atomic_store(&ctrl[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    WSF_MARK(7);
    return bad ? 0u : F.w[5];
}

// The keys of the list (n_keys <= kShortCap) in descending order; returns where they lie.
__device__ __forceinline__ uint64_t* few_sort(uint64_t* list, uint32_t n_keys, FewShared& F) {
    const uint32_t t = threadIdx.x;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    if (n_keys <= 64u) {
        // WS_BLOCK / 64 threads a key, each counting the larger keys among its share of the 64 places: one barrier
        constexpr uint32_t kPer = WS_BLOCK / 64u, kEach = 64u / kPer;
        static_assert(kPer == 8u, "the sum below is over eight lanes");
        uint64_t* sorted = list + 4096;
        const uint32_t ki = t / kPer, q0 = (t % kPer) * kEach;
        const uint64_t own = ki < n_keys ? list[ki] : 0ull;
        uint32_t above = 0;
        if (wv * (64u / kPer) < n_keys) {  // (per wave)
#pragma unroll
            for (uint32_t i = 0; i < kEach; i += 2u) {
                const ulonglong2 o = *reinterpret_cast<const ulonglong2*>(&list[q0 + i]);
                above += (q0 + i < n_keys && o.x > own ? 1u : 0u) + (q0 + i + 1u < n_keys && o.y > own ? 1u : 0u);
            }
            above += dpp_or_zero<0x111, 0xf>(above);
            above += dpp_or_zero<0x112, 0xf>(above);
            above += dpp_or_zero<0x114, 0xf>(above);  // lanes 7 and 15 of a row of sixteen have the sums of their eight
            if (ki < n_keys && t % kPer == kPer - 1u) sorted[above] = own;
        }
        __syncthreads();
        list = sorted;
    } else {
        short_sort(list, n_keys, F.red_f[0], F.sh);
    }
    return list;
}

// LDS: [0, 32 KiB) the list, [32 KiB, 64 KiB) its sorted copy while it is short; the history counts from 32 KiB on (they are
// dead by then).
// OWN: the row's parameters are those of `own` (kernel arguments behind the batch's).
template <int DT, bool MASKED, int NV, bool OWN>
__device__ __forceinline__ bool few_row(const BatchArgs& A, const OwnRow* own, const uint32_t row, const uint32_t part, FewShared& F, bool& finisher) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr uint32_t TPV = DT == 0 ? 4u : 8u;  // tokens in a 128-bit vector
    static_assert(NV * TPV * WS_BLOCK <= kFewWide, "tokens a share");
    ShortShared& S = F.sh;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    const uint32_t V = A.vocab;
    const unsigned char* base = static_cast<const unsigned char*>(A.logits) + static_cast<size_t>(row) * A.row_stride * (DT == 0 ? 4u : 2u);
    const uint32_t* allow = MASKED ? A.allow + static_cast<size_t>(row) * A.allow_stride : nullptr;
    finisher = false;
#ifdef WS_SHORT_TIMERS
    if (threadIdx.x == 0) F.t0 = clock64();
    const long long wss_t0 = clock64();
#endif

    const FewShare L = FewShare::of<DT>(V, A.few_parts, part, A.few_chunk_log2, A.few_vecs, A.few_slots);
    const uint32_t G = L.G, cl = L.cl, nv = L.nv, n_vec = L.n_vec;
    const uint32_t j_part = V % TPV ? nv - 1u : 0xffffffffu;
    uint4 q[NV];
    uint32_t na[NV];
#pragma unroll
    for (uint32_t k = 0; k < NV; ++k) {
        const uint32_t j = L.vec_of(k);
        q[k] = row_vector<DT>(base, j, V);
        na[k] = MASKED ? allow[min(j * TPV, V - 1u) >> 5] : 0xffffffffu;
    }
    uint32_t* cnt = reinterpret_cast<uint32_t*>(lds + 32768);  // two 16-bit counts a word; bit 15 of a count: somebody takes the token
    // and a bit for each of a thread's tokens that a list names: [word][thread]. (The counts alone took a thread two LDS words and ten
    // instructions a vector to find out that none of its four is named.)
    constexpr uint32_t kBits = few_bit_words(NV * TPV);
    uint32_t* named = cnt + NV * TPV * WS_BLOCK / 2u;
    const bool lists = A.hist || A.bias_ids;
    if (lists) {
#pragma unroll
        for (uint32_t k = 0; k < NV * TPV / 8u + (NV * TPV % 8u ? 1u : 0u); ++k) reinterpret_cast<uint4*>(cnt)[k * WS_BLOCK + t] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (uint32_t w = 0; w < kBits; ++w) named[w * WS_BLOCK + t] = 0u;
    }

    // ---- the row's parameters
    const LeanRowParams P = OWN ? own->P : load_row_params(A, row);
    WSS_MARK(0);  // parameters in
    const float inv_t = P.inv_t;
    const uint32_t top_k = P.top_k, nh = P.nh, nb = P.nb, n_all = nh + nb;
    const double min_p = P.min_p;
    const bool by_k = top_k >= 1u && top_k <= kShortMaxK && top_k <= V;  // the top_k largest decide
    const bool by_p = top_k == 0u && min_p > 0.0 && min_p <= 1.0;      // no top-k: what the min-p floor lets through decides
    const bool not_mine = !(by_k || by_p) || !(inv_t > 0.f) || n_all > A.patch_cap;

    // ---- history and bias entries: those of this share are counted, and the first entry of each token puts it, with its
    // logit, on a list (touched tokens: `ext`). A token that both lists name stands there twice; the bias entry's stays.
    uint4* ext = reinterpret_cast<uint4*>(lds);  // {token | kExtBias, logit, bias, place in the bias list}
    constexpr uint32_t kExtBias = 0x80000000u;
    const bool any_ext = lists && !not_mine && n_all;  // uniform
    if (t < 2u) F.w[t] = 0u;                           // bias entries of tokens another entry has taken; length of `ext`
    // this share's place of a token; 0xffffffff: not of this share
    auto place_of = [&](uint32_t id) {
        const uint32_t v = id / TPV, c = v >> cl;
        const uint32_t cq = static_cast<uint32_t>((static_cast<uint64_t>(c) * A.few_magic) >> 32), cg = c - cq * G;  // c / G, c mod G
        const uint32_t at = (((cg % WS_WAVES) * (NV * 64u) + (cq << cl) + (v & ((1u << cl) - 1u))) * TPV) + id % TPV;
        return id < V && cg / WS_WAVES == part ? at : 0xffffffffu;
    };
    auto name = [&](uint32_t li) {  // its bit: a wave's places are [vector][lane][token]
        const uint32_t w = li / (NV * 64u * TPV), r = li % (NV * 64u * TPV), b = r / (64u * TPV) * TPV + li % TPV;
        atomicOr(&named[(b >> 5) * WS_BLOCK + w * 64u + r / TPV % 64u], 1u << (b & 31u));
    };
    if (any_ext) {
        typedef const __attribute__((address_space(1))) int32_t* Ids;
        Ids hist_ids = (Ids)(A.hist + P.h0);
        if (OWN && own->n_ids)  // uniform
            hist_ids = (Ids)((uintptr_t)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr() + sizeof(BatchArgs) + offsetof(OwnRow, ids));
        const int32_t* bias_ids = A.bias_ids + P.b0;
        const float* bias_vals = A.bias_vals + P.b0;
        constexpr uint32_t kR = 4u;  // entries a thread at a time, their loads together
        auto four = [&](auto is_bias, uint32_t n, uint32_t j0, bool first) __attribute__((always_inline)) {
            constexpr bool BIAS = decltype(is_bias)::value;
            uint32_t id[kR], li[kR], raw[kR], al[kR];
            float bv[kR];
#pragma unroll
            for (uint32_t r = 0; r < kR; ++r) {
                const uint32_t j = j0 + r * WS_BLOCK + t;
                id[r] = 0xffffffffu;
                if (j0 + r * WS_BLOCK < n && j < n) id[r] = static_cast<uint32_t>(BIAS ? bias_ids[j] : hist_ids[j]);
            }
            if (first) __syncthreads();  // the counts are clear
#pragma unroll
            for (uint32_t r = 0; r < kR; ++r) {
                if (j0 + r * WS_BLOCK >= n) continue;  // uniform
                li[r] = place_of(id[r]);
                if (li[r] != 0xffffffffu) {
                    raw[r] = DT == 0 ? reinterpret_cast<const uint32_t*>(base)[id[r]] : static_cast<uint32_t>(reinterpret_cast<const uint16_t*>(base)[id[r]]) << 16;
                    al[r] = MASKED ? allow[id[r] >> 5] >> (id[r] & 31u) : 1u;
                    bv[r] = BIAS ? bias_vals[j0 + r * WS_BLOCK + t] : 0.f;
                }
            }
#pragma unroll
            for (uint32_t r = 0; r < kR; ++r) {
                if (j0 + r * WS_BLOCK >= n) continue;  // uniform
                bool takes = false;
                if (li[r] != 0xffffffffu) {
                    const uint32_t sh = (li[r] & 1u) * 16u;
                    if (!BIAS) {
                        takes = ((atomicAdd(&cnt[li[r] >> 1], 1u << sh) >> sh) & (kFewDup - 1u)) == 0u;
                    } else if ((atomicOr(&cnt[li[r] >> 1], kFewTaken << sh) >> sh) & kFewTaken) {  // another entry has this token: left where that one finds it
                        atomicOr(&cnt[li[r] >> 1], kFewDup << sh);
                        const uint32_t at = atomicAdd(&F.w[0], 1u);
                        if (at < kFewDups) {
                            F.dup_at[at] = static_cast<uint16_t>(li[r]);
                            F.dup_j[at] = static_cast<uint16_t>(j0 + r * WS_BLOCK + t);
                            F.dup_v[at] = bv[r];
                        }
                    } else {
                        takes = true;
                    }
                }
                if (takes) name(li[r]);
                const uint64_t mk = __ballot(takes);
                if (mk) {  // uniform
                    uint32_t at0 = 0;
                    if (lane == 0u) at0 = atomicAdd(&F.w[1], static_cast<uint32_t>(__popcll(mk)));
                    const uint32_t at = lane_value(at0, 0u) + lanes_before(mk);
                    if (takes && at < kFewExt)
                        ext[at] = make_uint4(id[r] | (BIAS ? kExtBias : 0u), al[r] & 1u ? raw[r] : 0xff800000u, __float_as_uint(bv[r]), j0 + r * WS_BLOCK + t);
                }
            }
        };
        bool first = true;
        for (uint32_t j0 = 0; j0 < nh; j0 += kR * WS_BLOCK, first = false) four(std::false_type{}, nh, j0, first);
        for (uint32_t j0 = 0; j0 < nb; j0 += kR * WS_BLOCK, first = false) four(std::true_type{}, nb, j0, first);
    }
    __syncthreads();
    WSS_MARK(1);  // history and bias entries counted

    // ---- the share: tokens that do not count - masked out, past the row, named by a list - become NaN
    uint32_t out[kBits];
#pragma unroll
    for (uint32_t w = 0; w < kBits; ++w) out[w] = any_ext ? named[w * WS_BLOCK + t] : 0u;
    if (MASKED)
#pragma unroll
        for (uint32_t k = 0; k < NV; ++k) out[k * TPV / 32u] |= (~(na[k] >> ((L.vec_of(k) * TPV) & 31u)) & ((1u << TPV) - 1u)) << (k * TPV % 32u);
    float x[NV][TPV], vm[NV];
    float lm = -INFINITY;
#pragma unroll
    for (uint32_t k = 0; k < NV; ++k) {
        if (k >= n_vec) {  // uniform
#pragma unroll
            for (uint32_t e = 0; e < TPV; ++e) x[k][e] = -INFINITY;
            vm[k] = -INFINITY;
            continue;
        }
        if (k + 1u == n_vec) {  // uniform: the round the row ends in
            const uint32_t j = L.vec_of(k);
            if (j == j_part) q[k] = part_vector<DT>(q[k], TPV - V % TPV);
            if (j >= nv) q[k] = make_uint4(0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu);
        }
        const uint32_t w[4] = {q[k].x, q[k].y, q[k].z, q[k].w};
#pragma unroll
        for (uint32_t e = 0; e < TPV; ++e) {
            const uint32_t bits = DT == 0 ? w[e] : ((e & 1u) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
            x[k][e] = few_logit(bits | static_cast<uint32_t>(static_cast<int32_t>(out[k * TPV / 32u] << (31u - (k * TPV + e) % 32u)) >> 31));
        }
        vm[k] = few_max_of<TPV>(x[k]);
        lm = fmaxf(lm, vm[k]);
    }
    WSS_MARK(2);  // share in registers

    // ---- the touched tokens: bias, repetition, frequency / presence (as ws_sample.h applies them); from here on the list
    // holds {token, adjusted logit}, and every thread keeps to its own entries
    const uint32_t n_ext = any_ext ? min(F.w[1], kFewExt) : 0u, n_ext_all = any_ext ? F.w[1] : 0u;
    for (uint32_t i = t; i < n_ext; i += WS_BLOCK) {
        const uint4 en = ext[i];
        const bool bias = (en.x & kExtBias) != 0u;
        const uint32_t id = en.x & ~kExtBias, li = place_of(id), sh = (li & 1u) * 16u, c = cnt[li >> 1] >> sh;
        float v = fmaxf(__uint_as_float(en.y), -INFINITY);
        if (bias) {
            const uint32_t n_dup = F.w[0];
            if (!(c & kFewDup)) {
                v = __fadd_rn(v, __uint_as_float(en.z));
            } else if (n_dup <= kFewDups) {  // the token's entries in the order of the list: this one and those left behind
                for (uint32_t from = 0; from <= nb;) {
                    uint32_t next = en.w >= from ? en.w : 0xfffffffeu;
                    float val = __uint_as_float(en.z);
                    for (uint32_t k = 0; k < n_dup; ++k)
                        if (F.dup_at[k] == li && F.dup_j[k] >= from && F.dup_j[k] < next) {
                            next = F.dup_j[k];
                            val = F.dup_v[k];
                        }
                    if (next == 0xfffffffeu) break;
                    v = __fadd_rn(v, val);
                    from = next + 1u;
                }
            } else {
                for (uint32_t j = 0; j < nb; ++j)
                    if (static_cast<uint32_t>(A.bias_ids[P.b0 + j]) == id) v = __fadd_rn(v, A.bias_vals[P.b0 + j]);
            }
        } else if (c & kFewTaken) {
            v = -INFINITY;  // (the bias entry has this token)
        }
        if ((c & (kFewDup - 1u)) && v > -INFINITY) {
            v = v > 0.f ? __fdiv_rn(v, P.rep) : __fmul_rn(v, P.rep);
            v = __fsub_rn(v, __fadd_rn(__fmul_rn(P.freq, static_cast<float>(c & (kFewDup - 1u))), P.pres));
        }
        v = fmaxf(v, -INFINITY);
        *reinterpret_cast<uint2*>(&ext[i]) = make_uint2(id, __float_as_uint(v));
        lm = fmaxf(lm, v);
    }
    WSS_MARK(11);  // touched tokens in
    unsigned char* work = A.work + static_cast<size_t>(row) * kFewRowBytes;
    FewWant W;
    W.by_k = by_k;
    W.by_p = by_p;
    W.top_k = top_k;
    W.inv_t = inv_t;
    W.min_p = min_p;
    if (!few_publish<DT, NV, true>(L, W, x, vm, lm, ext, n_ext, !not_mine && n_ext_all <= kFewExt, work, F)) return true;  // not the last: done
    finisher = true;
    WSS_MARK(6);  // ticket
    uint64_t* list = reinterpret_cast<uint64_t*>(lds);
    const uint32_t n_keys = few_collect<true>(L, W, work, F, list, [&]() {
            // (the seed by way of a vector register: as scalar arithmetic the generator's rounds are moved out of this branch)
            uint32_t seed_lo = static_cast<uint32_t>(P.seed);
            asm volatile("" : "+v"(seed_lo));
            const double u_ = batch_uniform(A.rng, (P.seed & 0xffffffff00000000ull) | seed_lo, row, P.step, 0);
            if (lane == 0u) F.u = u_;
    });
    const float m = F.red_f[0];
    const uint32_t n_cand = by_k ? top_k : n_keys;
    if (n_keys < n_cand || n_cand == 0u || n_keys > kShortCap) return false;

    WSS_MARK(8);  // keys
    list = few_sort(list, n_keys, F);
    WSS_MARK(9);  // sorted
    ShortRow R;
    R.top_p = P.top_p;
    R.min_p = min_p;
    R.u = F.u;
    R.z = F.sum();
    R.inv_t = inv_t;
    R.m = m;
    R.n_cand = n_cand;
    R.by_k = by_k;
    short_rules(list, row, R, S);
#ifdef WS_SHORT_TIMERS
    WSS_MARK(10);
    __syncthreads();
    if (t < 16 && A.kept_logits) A.kept_logits[static_cast<size_t>(row) * A.kept_cap + 100u + t] = t == 15 ? static_cast<float>(n_keys) : (t == 14 ? 0.f : S.marks[t]);
#endif
    return true;
}

// LEAVE: a row for which a check fails is marked in `flags` and left to another launch.
template <int DT, bool MASKED, int NV, bool OWN, bool LEAVE>
__device__ __forceinline__ void few_batch(const BatchArgs& A, const OwnRow* own) {
    __shared__ FewShared shared;
    uint32_t row, part;
    if (!few_place(A.few_together, A.rows, row, part)) return;
    bool finisher;
    if (!few_row<DT, MASKED, NV, OWN>(A, own, row, part, shared, finisher) && finisher) {
        __syncthreads();
        LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(Ap));
        if constexpr (LEAVE) {
            if (threadIdx.x == 0) Ap->flags[row] = kRowLeft;
        } else {
            if (Ap->kept_ids) three_pass_row<true>(Ap, row);
            else three_pass_row<false>(Ap, row);
        }
    }
    if (A.done && finisher) {  // a host looks at this word instead of waiting for the stream: everything written for the row first
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(&A.done[row], A.done_value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
template <int DT, bool MASKED, int NV>
__global__ void __launch_bounds__(WS_BLOCK) few_batch_kernel(BatchArgs A) {
    few_batch<DT, MASKED, NV, false, false>(A, nullptr);
}
// A lone row whose parameters and ids lie in host memory: as arguments they come with the launch, where the kernel above makes two trips over the bus, one behind
// the other, before it knows its touched tokens (a decode step of 151936 tokens and 256 ids through the host API: 19.4 -> 16.6 us; of 700 ids 17.2, of 2000, which stay where they are, 19.3).
template <int DT, int NV>
__global__ void __launch_bounds__(WS_BLOCK) few_own_kernel(BatchArgs A, OwnRow own) {
    few_batch<DT, false, NV, true, false>(A, &own);
}
// Without the three-pass code, which takes the kernel from 99 registers to 248 and gives it scratch memory: 1.1 us of a launch on an idle GPU (a decode step of 151936
// tokens and 256 ids through the host API 16.5 / 15.35 us; of equal logits, which it leaves, 1646 / 1648 a step where the caller remembers that, 1662 where it does not).
template <int DT, int NV>
__global__ void __launch_bounds__(WS_BLOCK) few_try_kernel(BatchArgs A, OwnRow own) {
    few_batch<DT, false, NV, true, true>(A, &own);
}

}  // namespace ws
