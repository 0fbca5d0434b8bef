// The short-list sampler: rows that carry a top-k of at most kShortMaxK, or no top-k but a min-p (the caller says so:
// ws_batch.top_k_max, ws_batch.min_p_min).
//
// What src/sampling/sampler.cpp:15-78 keeps of such a row is decided among its top_k largest logits alone, so the row
// needs no histogram of every token. One sweep at the speed of the loads:
//   * from the head of the row (of the slice, for a shared row) a threshold is read off a 4096-bin count of the head's
//     logits, such that about top_k + max(top_k / 2, 150) tokens of the row lie above it;
//   * the sweep keeps the maximum and the sum of exp((x - ref) inv_t) (Sampler::m and Sampler::sum, src/sampling/sampler.h:37-38)
//     and puts every token above the threshold on a list in LDS, as its 64-bit order key (logit, then id);
//   * tokens the history or the bias list touch are left out by the sweep (a bitmap in LDS, built as in ws_sample.h's
//     phase 0) and come in afterwards with their adjusted logit;
//   * the list is sorted, and the reference's rules run on the sorted candidates: top-k, top-p on the mass of those, min-p
//     against the largest, the draw by inverse CDF with the row's uniform.
// A row for which a check fails, whose list runs over, or that has neither a top-k nor a min-p after all, is handed to the
// three-pass code of ws_sample.h inside the same call (WS_FLAG_ROUTE_HANDED_BACK).
// More rows than compute units are ws_twin.h's. Few rows are shared between workgroups by the kernel of ws_few.h, which ends with the same sort and rules; those it has no
// registers or lists for are shared here: each part lists its slice against its own threshold and leaves list, maximum and sum in
// the row's workspace, and the part that arrives last - a ticket, nobody waits - takes them all and finishes the row. The
// top_k largest of the merged list are the row's when the k-th of them lies above every part's threshold.
// A row without a top-k but with a min-p: what the floor min_p * p(max) lets through lies within -ln(min_p) / inv_t of the
// row's maximum, so the threshold needs no fitting - the head's maximum (never above the row's) minus that distance and
// a little more; the candidates are the whole list, the top-p cut compares with the row's normaliser (the sweep's sum,
// rounded to float as Sampler::sum is), and a cut that falls behind the list leaves the min-p floor to decide.
#pragma once
#include "ws_lean.h"

namespace ws {

constexpr uint32_t kShortMaxK = 1024u;  // largest top-k: one candidate a thread in the finish
constexpr uint32_t kShortHead = 8u;     // head of a slice: vectors a thread asked for before anything else
constexpr uint32_t kShortSample = 8u;   // of those, the vectors a thread whose tokens the threshold is fitted to (32768 tokens of fp32)
constexpr uint32_t kRouteShort = 0x2000u;
constexpr uint32_t kRowLeft = 0xffffffffu;  // in `flags`: a row left to another launch (WS_FLAGS_LEFT; no set of flags has every bit)
constexpr uint32_t kTwinRest = kRowLeft;  // in `flags`, between two kernels: a row of ws_twin.h's left to the three-pass code (no set of flags has every bit)


#ifdef WS_SHORT_TIMERS
#define WSS_MARK(k) \
    if (threadIdx.x == 0) S.marks[k] = static_cast<float>(clock64() - wss_t0)
#else
#define WSS_MARK(k)
#endif

struct ShortShared {
#ifdef WS_SHORT_TIMERS
    float marks[16];
#endif
    double red_d[WS_WAVES];
    double s_d[8];
    unsigned long long s_q[4];
    uint32_t s_w[16];
    uint32_t red_u[WS_WAVES];
    float red_f[WS_WAVES];
    alignas(16) uint32_t bcnt[64], bstart[64];  // the bucket sort's counts and starts
};

// How far the keys of a list lie below its largest: the largest such distance, and their sum (known: somebody has looked).
struct ShortSpan {
    float dmax = 0.f, total = 0.f;
    bool known = false;
};
// Puts the n_list (<= kShortCap) different keys in descending order. m: the largest of their logits. Every thread calls it.
__device__ __forceinline__ void short_sort(uint64_t* list, const uint32_t n_list, const float m, ShortShared& S, const ShortSpan span = {}) {
    const uint32_t t = threadIdx.x;
    if (n_list <= WS_BLOCK / 4u) {
        // A short list (a lone row's top-k 40 lists some 200 keys): every key against every other, four threads a key,
        // each counting the larger keys in a quarter of the list - two barriers, where the bucket sort takes seven.
        const uint32_t ki = t >> 2, qr = t & 3u;
        const uint32_t chunk = ((n_list + 7u) >> 3) << 1;  // keys a quarter, even: two keys a read
        const uint32_t lo = qr * chunk, hi = min(lo + chunk, n_list);
        const uint64_t own = ki < n_list ? list[ki] : 0ull;
        uint32_t above = 0;
        if (ki < n_list) {
            for (uint32_t j = lo; j < hi; j += 8u) {  // four reads on their way together (one past the quarter's end stays inside the list's 32 KiB and is not counted)
                ulonglong2 o[4];
#pragma unroll
                for (uint32_t r = 0; r < 4u; ++r) o[r] = *reinterpret_cast<const ulonglong2*>(&list[j + 2u * r]);
#pragma unroll
                for (uint32_t r = 0; r < 4u; ++r)
                    above += ((j + 2u * r < hi && o[r].x > own) ? 1u : 0u) + ((j + 2u * r + 1u < hi && o[r].y > own) ? 1u : 0u);
            }
        }
        above += __shfl_xor(above, 1);
        above += __shfl_xor(above, 2);
        __syncthreads();  // (every key has been read)
        if (ki < n_list && qr == 0u) list[above] = own;  // (the keys are all different: so are their ranks)
        __syncthreads();
    } else {
        // Buckets by how far a logit lies above the lowest listed one, on a logarithmic scale of the mean such distance: a
        // list is the tail of a row's logits, dense at its lower end, with a few tokens far above as a rule. (On a linear
        // scale a third of the keys could share a bucket, and each of them counts the others: 871 of 8 rows' keys took 12K
        // clocks, 8K of them there.)
        float dmax = span.dmax;
        double total = static_cast<double>(span.total);
        if (!span.known) {
            float dsum = 0.f;
            for (uint32_t k = t; k < n_list; k += WS_BLOCK) {
                const float d = fminf(__fsub_rn(m, unkey32(static_cast<uint32_t>(list[k] >> 32))), 3e38f);
                dmax = fmaxf(dmax, d);
                dsum += d;
            }
            dmax = wave_max(dmax);
            dsum = wave_sum(dsum);
            __syncthreads();  // (the row's maximum and sum were read from these words, and not every wave need have come by)
            if ((t & 63u) == 0u) {
                S.red_f[t >> 6] = dmax;
                S.red_d[t >> 6] = static_cast<double>(dsum);
            }
            __syncthreads();
            dmax = S.red_f[0];
            total = S.red_d[0];
#pragma unroll
            for (uint32_t w = 1; w < WS_WAVES; ++w) {
                dmax = fmaxf(dmax, S.red_f[w]);
                total += S.red_d[w];
            }
        }
        const float mean = fmaxf(dmax - static_cast<float>(total) / static_cast<float>(n_list), dmax * 1e-6f + 1e-30f);
        // (512 buckets, their counters behind the keys, while the list leaves that room; else 64 in the static words)
        const bool wide = n_list <= kShortCap - 512u;
        const uint32_t nbk = wide ? 512u : 64u;
        uint32_t* bc = wide ? reinterpret_cast<uint32_t*>(list + (kShortCap - 512u)) : S.bcnt;
        uint32_t* bs = wide ? bc + 512 : S.bstart;
        // the logarithm is the bit pattern of 1 + distance / mean: every step of it is monotonous, as the sort needs it
        const float per = 1.f / mean;
        auto level = [&](float d) { return static_cast<float>(__float_as_uint(__fadd_rn(1.f, __fmul_rn(fmaxf(__fsub_rn(dmax, d), 0.f), per))) - 0x3f800000u); };
        const float scale = static_cast<float>(nbk) / (level(0.f) + 1.f);
        bucket_sort_desc(list, n_list, bc, bs, nbk, [&](uint64_t key_) {
            const float d = fminf(__fsub_rn(m, unkey32(static_cast<uint32_t>(key_ >> 32))), 3e38f);
            return nbk - 1u - min(nbk - 1u, static_cast<uint32_t>(level(d) * scale));
        });
    }
}

// what the rules need to know of a row
struct ShortRow {
    double top_p, min_p, u, z;  // z: the row's normaliser against its maximum m
    float inv_t, m;
    uint32_t n_cand;  // candidates: the first n_cand keys of the list (1 .. kShortCap)
    bool by_k;        // they are the row's top_k largest; else everything the min-p floor may let through
};

// a distance to a decision, and what it is measured in (divided only where somebody asks for the quotient: a division is some 200 clocks of the chain)
struct ShortMargin {
    double d, of;
};
// The row's answer, written by the lane that has the drawn token: its id, its mass, the running mass with and without it; the kept set's size and mass
__device__ __forceinline__ void short_answer(const LeanArgPtr Ap, const uint32_t row, const ShortRow& R, uint32_t n3, uint32_t id, double e, double cin, double cex, double Zk, double target,
                                             bool drawn, ShortMargin mg_top_p, ShortMargin mg_min_p, uint32_t pos) {
    const ShortMargin mg = {drawn ? fmin(cin - target, pos > 0u ? target - cex : 1e300) : 0.0, Zk};
    const double tol = Ap->tol;
    uint32_t flags = kRouteShort;
    if (mg_top_p.d < tol * mg_top_p.of) flags |= kNearTopP;
    if (mg_min_p.d < tol * mg_min_p.of) flags |= kNearMinP;
    if (mg.d < tol * mg.of) flags |= kNearDraw;
    Ap->token[row] = static_cast<int32_t>(id);
    Ap->flags[row] = flags;
    if (Ap->prob) Ap->prob[row] = static_cast<float>(e / Zk);
    if (Ap->n_kept) Ap->n_kept[row] = n3;
    if (Ap->stats) {
        Ap->stats[2 * row] = R.m;
        Ap->stats[2 * row + 1] = static_cast<float>(R.z);
    }
    if (Ap->margin) {
        Ap->margin[3 * row] = mg_top_p.d / mg_top_p.of;
        Ap->margin[3 * row + 1] = mg_min_p.d / mg_min_p.of;
        Ap->margin[3 * row + 2] = mg.d / mg.of;
    }
}

// The same for a row with a top-k, without an order: the keys are dealt to 512 buckets as the sort would, with their masses, and one wave looks for the cuts and
// the draw - a bucket by the buckets' running counts and masses, then a place among its few keys, which alone are put in order. What bounds a wide top-k's
// finish where other rows sweep on the same unit (ws_twin.h) is the instructions: the rank and running mass of every key, sixteen waves in and out of a dozen barriers.
// Masses are added up in fixed point against the maximum's, in whole units of 2^-51 and what is left of each in units of 2^-77: the order of the additions does not
// matter, and a running mass is as good as exact until it becomes a 64-bit float. (Worked out on the CPU for 3000 lists of 600 to 2000 keys, the error of a running mass in
// units of 2^-53 of itself: 0.5 on average and 2.9 at most; short_rules' sums 1.3 and 9.3.)
// For 65 keys and more (n_list <= kShortCap - 1024: the buckets lie behind the list) of rows that are asked for neither a kept-set dump
// nor an entropy or a query. Every thread calls it. Returns false when a bucket has more than a wave's lanes of keys (equal logits; where logits were 16-bit
// floats once, hundreds are equal), which the counts tell before anybody has worked out a mass: the list still holds the same keys, and `span` is known.
// S.s_d[7]: the row's normaliser (R.z is not looked at: nobody has to keep it in registers meanwhile).
__device__ __forceinline__ bool short_pick(uint64_t* list, const uint32_t n_list, const uint32_t row, const ShortRow& R, ShortShared& S, ShortSpan& span) {
    constexpr uint32_t K = (kShortCap - 1024u) / WS_BLOCK, NB = 512u;
    static_assert(WS_BLOCK >= NB, "a thread a bucket");
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    unsigned long long* mass = reinterpret_cast<unsigned long long*>(list + (kShortCap - 1024u));
    uint32_t *rest = reinterpret_cast<uint32_t*>(mass + NB), *cnt = rest + NB, *start = cnt;  // (the buckets' first places, once their counts are read)
    const double inv_t = static_cast<double>(R.inv_t), min_p = R.min_p;
    const bool use_top_p = R.top_p < 1.0, use_min_p = min_p > 0.0;
    // (2^51 and 2^26: a mass is 1 at most, and there are 4096 of them; the rests of a bucket's 64 keys are 32 bits together)
    constexpr double kFix = 2251799813685248.0, kUnfix = 1.0 / kFix, kRest = 67108864.0, kUnrest = kUnfix / kRest;
    float d[K], dmax = 0.f, dsum = 0.f;
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        d[k] = 0.f;
        if (k * WS_BLOCK < n_list && k * WS_BLOCK + t < n_list) {
            d[k] = fminf(__fsub_rn(R.m, unkey32(static_cast<uint32_t>(list[k * WS_BLOCK + t] >> 32))), 3e38f);
            dmax = fmaxf(dmax, d[k]);
            dsum += d[k];
        }
    }
    if (t < NB) {
        mass[t] = 0ull;
        rest[t] = 0u;
        cnt[t] = 0u;
    }
    if (t == 0u) {
        S.s_w[6] = 0u;
        S.s_w[8] = 0u;
        S.s_q[0] = ~0ull;
    }
    dmax = wave_max(dmax);
    dsum = wave_sum(dsum);
    if (lane == 0u) {
        S.bcnt[wv] = __float_as_uint(dmax);
        S.bstart[wv] = __float_as_uint(dsum);
    }
    __syncthreads();  // (the buckets are clear as well)
    float total = 0.f;
    dmax = 0.f;
#pragma unroll
    for (uint32_t w = 0; w < WS_WAVES; ++w) {
        dmax = fmaxf(dmax, __uint_as_float(S.bcnt[w]));
        total += __uint_as_float(S.bstart[w]);
    }
    span = {dmax, total, true};
    const float mean = fmaxf(dmax - total / static_cast<float>(n_list), dmax * 1e-6f + 1e-30f);
    // (the scale of short_sort's buckets)
    const float per = 1.f / mean;
    auto level = [&](float d_) { return static_cast<float>(__float_as_uint(__fadd_rn(1.f, __fmul_rn(fmaxf(__fsub_rn(dmax, d_), 0.f), per))) - 0x3f800000u); };
    const float scale = static_cast<float>(NB) / (level(0.f) + 1.f);
    uint32_t at[K];  // bucket | place in it << 16
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n_list && k * WS_BLOCK + t < n_list) {
            const uint32_t b = NB - 1u - min(NB - 1u, static_cast<uint32_t>(level(d[k]) * scale)), place = atomicAdd(&cnt[b], 1u);
            at[k] = b | (place << 16);
            if (place >= 64u) S.s_w[8] = 1u;
        }
    __syncthreads();
    if (S.s_w[8] != 0u) return false;
    uint32_t pass = 0;
    double near = INFINITY;
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n_list && k * WS_BLOCK + t < n_list) {
            const double e = exp_down(static_cast<double>(d[k]) * inv_t), fixed = e * kFix, whole = floor(fixed);
            const uint32_t b = at[k] & 0xffffu;
            atomicAdd(&mass[b], static_cast<unsigned long long>(whole));
            atomicAdd(&rest[b], static_cast<uint32_t>((fixed - whole) * kRest));
            pass += e >= min_p ? 1u : 0u;
            near = fmin(near, fabs(e - min_p));
        }
    if (use_min_p) {
        pass = wave_sum(pass);
        if (lane == 0u && pass) atomicAdd(&S.s_w[6], pass);
        // The bits of numbers that are not negative, in their order; a wave's smallest by halves. (An atomic of every lane, which the compiler makes a 64-bit scan of, was
        // 2 to 8 us of a launch: top-k 600, min-p 0.09, 257 rows of 8206 29.4 -> 25.4, 300 of 8982 29.4 -> 24.6, 1024 of 57152 88.1 -> 80.4.)
        const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(near));
        const uint32_t high = wave_min_u32(static_cast<uint32_t>(bits >> 32)), low = wave_min_u32(static_cast<uint32_t>(bits >> 32) == high ? static_cast<uint32_t>(bits) : 0xffffffffu);
        if (lane == 0u) atomicMin(&S.s_q[0], (static_cast<unsigned long long>(high) << 32) | low);
    }
    uint32_t c8[8], n_in = 0;
    if (wv == 0u) {  // a lane has eight buckets
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            c8[k] = cnt[lane * 8u + k];
            n_in += c8[k];
        }
        uint32_t run = wave_incl_scan(n_in) - n_in;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            start[lane * 8u + k] = run;
            run += c8[k];
        }
        n_in = run;
    }
    uint64_t key[K];  // (read again: the exponentials have the registers)
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) key[k] = k * WS_BLOCK < n_list && k * WS_BLOCK + t < n_list ? list[k * WS_BLOCK + t] : 0ull;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        if (k * WS_BLOCK < n_list && k * WS_BLOCK + t < n_list) list[start[at[k] & 0xffffu] + (at[k] >> 16)] = key[k];
    __syncthreads();
    if (wv != 0u) return true;

    // ------------------------------------------------------------------ one wave
    double m8[8];  // the running mass with each of the lane's buckets
    {
        uint64_t g8[8], l8[8], g = 0, l = 0;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            g8[k] = g += mass[lane * 8u + k];
            l8[k] = l += rest[lane * 8u + k];
        }
        const uint64_t g0 = wave_incl_scan(g) - g, l0 = wave_incl_scan(l) - l;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) m8[k] = fma(static_cast<double>(l0 + l8[k]), kUnrest, static_cast<double>(g0 + g8[k]) * kUnfix);
    }
    // a bucket's keys in order, one a lane, with what is ranked before them
    struct Place {
        uint32_t n, before;  // keys in the bucket, and before it
        uint64_t key;
        double e, cin, cex;
    };
    // the first bucket with which the running count and mass satisfy `reached`; found: whether there is one
    auto look = [&](auto&& reached, bool& found) __attribute__((always_inline)) {
        Place R_;
        const uint64_t any = __ballot(reached(n_in, m8[7]));
        found = any != 0ull;
        const uint32_t f = found ? static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1) : 63u;
        uint32_t run = f ? lane_value(n_in, f - 1u) : 0u, n = 0, first = run;
        double sum = f ? lane_value(m8[7], f - 1u) : 0.0, before = sum;
        bool done = false;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t c = lane_value(c8[k], f);
            const double with = lane_value(m8[k], f);
            if (!done && c) {  // uniform
                n = c;
                first = run;
                before = sum;
                run += c;
                sum = with;
                done = reached(run, sum);
            }
        }
        const uint64_t own = lane < n ? list[first + lane] : 0ull;  // (the buckets lie one behind the other)
        uint32_t above = 0;
        for (uint32_t j = 0; j < n; ++j) above += lane_value(own, j) > own ? 1u : 0u;  // uniform
        uint64_t* sorted = reinterpret_cast<uint64_t*>(mass);  // (the masses are in registers)
        if (lane < n) sorted[above] = own;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        R_.n = n;
        R_.before = first;
        R_.key = lane < n ? sorted[lane] : 0ull;
        R_.e = lane < n ? exp_down(static_cast<double>(__fsub_rn(R.m, unkey32(static_cast<uint32_t>(R_.key >> 32)))) * inv_t) : 0.0;
        const double inc = wave_incl_scan(R_.e), up = __shfl_up(inc, 1);
        R_.cin = before + inc;
        R_.cex = before + (lane ? up : 0.0);
        __builtin_amdgcn_wave_barrier();
        return R_;
    };
    bool found;
    const uint32_t n_cand = R.n_cand;
    const double all = lane_value(m8[7], 63u);
    double Zk1 = all, e_last = -1.0;
    if (n_list > n_cand) {
        const Place at_k = look([&](uint32_t n, double) { return n >= n_cand; }, found);
        const uint32_t j = n_cand - 1u - at_k.before;
        Zk1 = lane_value(at_k.cin, j);
        e_last = lane_value(at_k.e, j);
    }
    const double X = R.top_p * Zk1;
    uint32_t n3 = n_cand;
    double M = Zk1;
    ShortMargin mg_top_p = {1.0, 1.0}, mg_min_p = {1.0, 1.0};
    if (use_top_p) {
        const Place at_p = look([&](uint32_t, double m_) { return m_ >= X; }, found);
        mg_top_p = {0.0, X};  // (rounding: the running mass never reaches top_p of itself)
        if (found) {
            const uint64_t is = __ballot(lane < at_p.n && at_p.cin >= X);
            const uint32_t j = is ? static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(is)) - 1) : at_p.n - 1u;
            if (at_p.before + j < n_cand) {
                n3 = at_p.before + j + 1u;
                M = lane_value(at_p.cin, j);
                const double ex = lane_value(at_p.cex, j);
                mg_top_p = {fmin(M - X, n3 > 1u ? X - ex : X), X};
            }
        }
    }
    if (use_min_p) {
        const uint32_t passed = S.s_w[6];
        const double nearest = passed >= n_cand && e_last >= 0.0 ? fabs(e_last - min_p) : __longlong_as_double(static_cast<long long>(S.s_q[0]));
        mg_min_p = {fmin(min_p, nearest), min_p};
        if (passed < n3) {
            n3 = max(passed, 1u);
            const Place at_n = look([&](uint32_t n, double) { return n >= n3; }, found);
            M = lane_value(at_n.cin, n3 - 1u - at_n.before);
        }
    }
    const double target = R.u * M;
    Place at_u = look([&](uint32_t, double m_) { return m_ > target; }, found);
    uint32_t j;
    {
        const uint64_t is = __ballot(lane < at_u.n && at_u.cin > target);
        j = is ? static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(is)) - 1) : at_u.n - 1u;
    }
    const bool drawn = found && at_u.before + j < n3;
    if (!drawn) {  // (rounding: the walk falls through to the last kept, src/sampling/sampler.cpp:131)
        at_u = look([&](uint32_t n, double) { return n >= n3; }, found);
        j = n3 - 1u - at_u.before;
    }
    const LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    ShortRow answer = R;
    answer.z = S.s_d[7];
    if (lane == j)
        short_answer(Ap, row, answer, n3, 0xffffffffu - static_cast<uint32_t>(at_u.key), at_u.e, at_u.cin, at_u.cex, M, target, drawn, mg_top_p, mg_min_p, at_u.before + j);
    return true;
}

// The reference's rules (src/sampling/sampler.cpp:31-74, :118-131) on the sorted candidates, and the row's results. Every
// thread of the workgroup calls it.
__device__ __forceinline__ void short_rules(uint64_t* list, const uint32_t row, const ShortRow& R, ShortShared& S) {
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    const double top_p = R.top_p, min_p = R.min_p, u = R.u;
    const bool use_top_p = top_p < 1.0, use_min_p = min_p > 0.0, by_k = R.by_k;
    const float inv_t = R.inv_t, m = R.m;
    const uint32_t n_cand = R.n_cand;
    // what the top-p cut compares with: the mass of the top_k candidates (src/sampling/sampler.cpp:45-48, a closed set),
    // or the row's normaliser as a float (Sampler::sum) when there is no top-k
    const double z_row = static_cast<double>(static_cast<float>(R.z));

    // ---- the rules (src/sampling/sampler.cpp:31-74) on the top_k candidates, one a thread: masses against the maximum,
    // running sums in sorted order
    const bool has = t < n_cand;
    const uint64_t key = has ? list[t] : 0ull;
    const float x = has ? unkey32(static_cast<uint32_t>(key >> 32)) : -INFINITY;
    const uint32_t id = 0xffffffffu - static_cast<uint32_t>(key);
    const LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t n3;
    typedef ShortMargin Margin;
    auto write_out = [&](uint32_t id_, double e_, double cin_, double cex_, double Zk_, double target_, bool drawn, Margin mg_top_p_, Margin mg_min_p_, uint32_t pos) {
        short_answer(Ap, row, R, n3, id_, e_, cin_, cex_, Zk_, target_, drawn, mg_top_p_, mg_min_p_, pos);
    };
    // optional outputs: -sum p ln p over the kept set with p = e / Zk and ln e = (x - m) / temperature, which is
    // ln Zk - (sum of e ln e) / Zk; and the share of one named token, 0 when it is not kept
    const bool more = Ap->entropy != nullptr || Ap->query_prob != nullptr;  // uniform
    const uint32_t query = (Ap->query_prob && Ap->query) ? static_cast<uint32_t>(Ap->query[row]) : 0xffffffffu;  // (none: no token's id)
    auto log_mass = [&](float x_) { return static_cast<double>(__fsub_rn(x_, m)) * static_cast<double>(inv_t); };
    auto write_more = [&](double e_ln_e, double e_query, double Zk_) {
        if (Ap->entropy) Ap->entropy[row] = log(Zk_) - e_ln_e / Zk_;
        if (Ap->query_prob) Ap->query_prob[row] = e_query / Zk_;
    };
    // more candidates than threads (a wide top-k, a wide min-p floor): thread t has those at places KC t .. KC t + KC - 1 of the order; the same rules.
    // (KC as small as will do: with eight a thread for all of them most waves had none. 512 threads: 8 rows of 32000, top-k 600, 18.5 us -> 16.3; 64 rows with
    // min-p floors that let 600 to 2000 through 33.7 -> 32.2)
    auto several = [&](auto kc) __attribute__((always_inline)) {
        constexpr uint32_t KC = decltype(kc)::value;
        uint64_t wkey[KC];
        double e[KC], cin[KC], cex[KC], tot = 0.0;
#pragma unroll
        for (uint32_t j = 0; j < KC; ++j) {
            const uint32_t pos = KC * t + j;
            wkey[j] = pos < n_cand ? list[pos] : 0ull;
            e[j] = pos < n_cand ? exp_down(static_cast<double>(__fsub_rn(m, unkey32(static_cast<uint32_t>(wkey[j] >> 32)))) * static_cast<double>(inv_t)) : 0.0;
            tot += e[j];
        }
        double Zk1;
        double run = block_excl_scan(tot, S.red_d, &Zk1);
#pragma unroll
        for (uint32_t j = 0; j < KC; ++j) {
            cex[j] = run;
            run += e[j];
            cin[j] = run;
        }
        if (t == 0) {
            S.s_q[0] = ~0ull;
            S.s_q[1] = ~0ull;
            S.s_w[6] = 0u;
            S.s_d[0] = 1.0;
            S.s_d[1] = 1.0;
            S.s_d[2] = 1.0;
        }
        __syncthreads();
        const double X = top_p * (by_k ? Zk1 : z_row);
        uint32_t pass_local = 0;
#pragma unroll
        for (uint32_t j = 0; j < KC; ++j) {
            const uint32_t pos = KC * t + j;
            if (use_top_p && pos < n_cand && cin[j] >= X && !(cex[j] >= X)) atomicMin(&S.s_q[0], static_cast<unsigned long long>(pos));
            pass_local += (pos < n_cand && e[j] >= min_p) ? 1u : 0u;
        }
        if (use_min_p) {
            const uint32_t wp = wave_sum(pass_local);
            if (lane == 0u && wp) atomicAdd(&S.s_w[6], wp);
        }
        __syncthreads();
        uint32_t n2 = n_cand;
        double mg_top_p = 1.0, mg_min_p = 1.0;
        bool cut_behind = false;
        const unsigned long long cq = use_top_p ? S.s_q[0] : ~0ull;
        if (use_top_p) {
            if (cq != ~0ull) n2 = static_cast<uint32_t>(cq) + 1u;
            else if (by_k) mg_top_p = 0.0;
            else cut_behind = true;
        }
        n3 = n2;
        const uint32_t passed = use_min_p ? S.s_w[6] : 0u;
        if (use_min_p) {
            n3 = min(n2, passed);
            if (n3 < 1u) n3 = 1u;
        }
#pragma unroll
        for (uint32_t j = 0; j < KC; ++j) {
            const uint32_t pos = KC * t + j;
            if (pos >= n_cand) continue;
            if (use_top_p && cq != ~0ull && pos == n2 - 1u) S.s_d[0] = fmin(cin[j] - X, pos > 0u ? X - cex[j] : X) / X;
            if (use_min_p && passed > 0u && pos == passed - 1u) S.s_d[1] = fabs(e[j] - min_p) / min_p;
            if (use_min_p && pos == passed && passed < n_cand) S.s_d[2] = fabs(e[j] - min_p) / min_p;
            if (pos == n3 - 1u) S.s_d[3] = cin[j];
        }
        __syncthreads();
        if (cut_behind) mg_top_p = (X - Zk1) / X;
        else if (use_top_p && mg_top_p != 0.0) mg_top_p = S.s_d[0];
        if (use_min_p) mg_min_p = fmin(S.s_d[1], S.s_d[2]);
        const double Zk = S.s_d[3];
        const double target = u * Zk;
#pragma unroll
        for (uint32_t j = 0; j < KC; ++j) {
            const uint32_t pos = KC * t + j;
            if (pos < n3 && cin[j] > target && !(cex[j] > target)) atomicMin(&S.s_q[1], static_cast<unsigned long long>(pos));
        }
        __syncthreads();
        const unsigned long long dq = S.s_q[1];
        const uint32_t d_pos = dq != ~0ull ? static_cast<uint32_t>(dq) : n3 - 1u;
#pragma unroll
        for (uint32_t j = 0; j < KC; ++j)
            if (KC * t + j == d_pos)
                write_out(0xffffffffu - static_cast<uint32_t>(wkey[j]), e[j], cin[j], cex[j], Zk, target, dq != ~0ull, {mg_top_p, 1.0}, {mg_min_p, 1.0}, d_pos);
        if (more) {
            double se = 0.0, sq = 0.0;
#pragma unroll
            for (uint32_t j = 0; j < KC; ++j)
                if (KC * t + j < n3) {
                    if (e[j] > 0.0) se += e[j] * log_mass(unkey32(static_cast<uint32_t>(wkey[j] >> 32)));
                    if (0xffffffffu - static_cast<uint32_t>(wkey[j]) == query) sq += e[j];
                }
            se = block_sum(se, S.red_d);
            sq = block_sum(sq, S.red_d);
            if (t == 0) write_more(se, sq, Zk);
        }
    };
    if (n_cand <= 64u) {
        // the usual case, a top-k of a few dozen: one wave, a candidate a lane, no barrier and no atomic
        if (wv == 0u) {
            const double e = has ? exp_down(static_cast<double>(__fsub_rn(m, x)) * static_cast<double>(inv_t)) : 0.0;
            const double cin = wave_incl_scan(e);
            const double up = __shfl_up(cin, 1);
            const double cex = lane ? up : 0.0;
            const double Zk1 = lane_value(cin, n_cand - 1u);
            const double X = top_p * (by_k ? Zk1 : z_row);
            uint32_t n2 = n_cand;
            Margin mg_top_p = {1.0, 1.0}, mg_min_p = {1.0, 1.0};
            if (use_top_p) {
                const uint64_t cm = __ballot(has && cin >= X && !(cex >= X));
                if (cm) {
                    const uint32_t jc = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(cm)) - 1);
                    n2 = jc + 1u;
                    const double ci = lane_value(cin, jc), ce = lane_value(cex, jc);
                    mg_top_p = {fmin(ci - X, jc > 0u ? X - ce : X), X};
                } else {
                    // a top-k row: rounding, the running mass never reaches top_p of itself. Else: the cut lies behind the list
                    mg_top_p = {by_k ? 0.0 : X - Zk1, X};
                }
            }
            n3 = n2;
            if (use_min_p) {
                const uint32_t passed = static_cast<uint32_t>(__popcll(__ballot(has && e >= min_p)));  // (a prefix of the order: masses do not rise along it)
                n3 = min(n2, passed);
                if (n3 < 1u) n3 = 1u;
                const double near = fabs(e - min_p);
                mg_min_p = {min_p, min_p};
                if (passed > 0u) mg_min_p.d = fmin(mg_min_p.d, lane_value(near, passed - 1u));
                if (passed < n_cand) mg_min_p.d = fmin(mg_min_p.d, lane_value(near, passed));
            }
            const double Zk = lane_value(cin, n3 - 1u);
            const double target = u * Zk;
            const uint64_t dm = __ballot(has && lane < n3 && cin > target && !(cex > target));
            const uint32_t d_pos = dm ? static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(dm)) - 1) : n3 - 1u;  // (src/sampling/sampler.cpp:131: the walk falls through to the last kept)
            if (lane == d_pos) write_out(id, e, cin, cex, Zk, target, dm != 0ull, mg_top_p, mg_min_p, d_pos);
            if (more) {
                const bool kept = has && lane < n3;
                const double se = wave_sum(kept && e > 0.0 ? e * log_mass(x) : 0.0), sq = wave_sum(kept && id == query ? e : 0.0);
                if (lane == 0u) write_more(se, sq, Zk);
            }
        }
    } else if (n_cand <= WS_BLOCK) {
        double e = 0.0;
        if (wv * 64u < n_cand) e = has ? exp_down(static_cast<double>(__fsub_rn(m, x)) * static_cast<double>(inv_t)) : 0.0;  // (per wave)
        double Zk1;
        const double cex = block_excl_scan(e, S.red_d, &Zk1);  // mass ranked before this candidate; Zk1: of all top_k
        const double cin = cex + e;
        if (t == 0) {
            S.s_q[0] = ~0ull;  // the top-p cut: first position whose running mass reaches X
            S.s_q[1] = ~0ull;  // the draw
            S.s_w[6] = 0u;     // candidates at or above the min-p floor
            S.s_d[0] = 1.0;    // margins: top-p, min-p (two neighbours)
            S.s_d[1] = 1.0;
            S.s_d[2] = 1.0;
        }
        __syncthreads();
        const double X = top_p * (by_k ? Zk1 : z_row);
        if (use_top_p && has && cin >= X && !(cex >= X)) atomicMin(&S.s_q[0], static_cast<unsigned long long>(t));
        if (use_min_p) {
            const uint64_t np = __ballot(has && e >= min_p);
            if (lane == 0u && np) atomicAdd(&S.s_w[6], static_cast<uint32_t>(__popcll(np)));
        }
        __syncthreads();
        uint32_t n2 = n_cand;
        double mg_top_p = 1.0, mg_min_p = 1.0;
        bool cut_behind = false;
        if (use_top_p) {
            const unsigned long long cq = S.s_q[0];
            if (cq != ~0ull) n2 = static_cast<uint32_t>(cq) + 1u;
            else if (by_k) mg_top_p = 0.0;  // rounding: the running mass never reaches top_p of itself
            else cut_behind = true;         // no top-k: the cut lies behind the list
            if (has && t == n2 - 1u && cq != ~0ull) S.s_d[0] = fmin(cin - X, t > 0u ? X - cex : X) / X;
        }
        n3 = n2;
        if (use_min_p) {
            const uint32_t passed = S.s_w[6];  // (a prefix of the order: masses do not rise along it)
            n3 = min(n2, passed);
            if (n3 < 1u) n3 = 1u;
            if (has && passed > 0u && t == passed - 1u) S.s_d[1] = fabs(e - min_p) / min_p;
            if (has && t == passed && passed < n_cand) S.s_d[2] = fabs(e - min_p) / min_p;
        }
        if (has && t == n3 - 1u) S.s_d[3] = cin;  // mass of the kept set
        __syncthreads();
        if (cut_behind) mg_top_p = (X - Zk1) / X;
        else if (use_top_p && mg_top_p != 0.0) mg_top_p = S.s_d[0];
        if (use_min_p) mg_min_p = fmin(S.s_d[1], S.s_d[2]);
        const double Zk = S.s_d[3];
        const double target = u * Zk;
        if (has && t < n3 && cin > target && !(cex > target)) atomicMin(&S.s_q[1], static_cast<unsigned long long>(t));
        __syncthreads();
        const unsigned long long dq = S.s_q[1];
        const uint32_t d_pos = dq != ~0ull ? static_cast<uint32_t>(dq) : n3 - 1u;  // (src/sampling/sampler.cpp:131: the walk falls through to the last kept)
        if (has && t == d_pos) write_out(id, e, cin, cex, Zk, target, dq != ~0ull, {mg_top_p, 1.0}, {mg_min_p, 1.0}, d_pos);
        if (more) {
            const bool kept = has && t < n3;
            const double se = block_sum(kept && e > 0.0 ? e * log_mass(x) : 0.0, S.red_d), sq = block_sum(kept && id == query ? e : 0.0, S.red_d);
            if (t == 0) write_more(se, sq, Zk);
        }
    } else if (n_cand <= 2u * WS_BLOCK) {
        several(std::integral_constant<uint32_t, 2u>{});
    } else if (WS_BLOCK < 1024 && n_cand <= 4u * WS_BLOCK) {
        several(std::integral_constant<uint32_t, 4u>{});
    } else {
        several(std::integral_constant<uint32_t, kShortCap / WS_BLOCK>{});
    }
    // ---- the kept set in ascending id order (the first kept_cap of it): of up to 64 by the wave that has them, else the same sort on (inverted
    // id, logit) pairs
    if (Ap->kept_ids && n_cand <= 64u) {
        if (wv == 0u) {
            uint32_t place = 0;
            for (uint32_t j = 0; j < n3; ++j) place += lane_value(id, j) < id ? 1u : 0u;  // uniform
            if (lane < n3 && place < Ap->kept_cap) {
                Ap->kept_ids[static_cast<size_t>(row) * Ap->kept_cap + place] = static_cast<int32_t>(id);
                if (Ap->kept_logits) Ap->kept_logits[static_cast<size_t>(row) * Ap->kept_cap + place] = x;
            }
        }
    } else if (Ap->kept_ids) {
        __syncthreads();
        if (n_cand > WS_BLOCK) {
            for (uint32_t k = t; k < n3; k += WS_BLOCK) {
                const uint64_t key_ = list[k];
                list[k] = (static_cast<uint64_t>(static_cast<uint32_t>(key_)) << 32) | __float_as_uint(unkey32(static_cast<uint32_t>(key_ >> 32)));
            }
        } else if (t < n3) {
            list[t] = (static_cast<uint64_t>(0xffffffffu - id) << 32) | __float_as_uint(x);
        }
        __syncthreads();
        const uint32_t per_bucket = (Ap->vocab + 63u) / 64u;
        bucket_sort_desc(list, n3, S.bcnt, S.bstart, 64u, [&](uint64_t key_) { return (0xffffffffu - static_cast<uint32_t>(key_ >> 32)) / per_bucket; });
        for (uint32_t k = t; k < n3 && k < Ap->kept_cap; k += WS_BLOCK) {
            const uint64_t e_ = list[k];
            Ap->kept_ids[static_cast<size_t>(row) * Ap->kept_cap + k] = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(e_ >> 32));
            if (Ap->kept_logits) Ap->kept_logits[static_cast<size_t>(row) * Ap->kept_cap + k] = __uint_as_float(static_cast<uint32_t>(e_));
        }
    }
}

// LDS of a row: [0, 32 KiB) the list (before the sweep: the head's bin counts), then at lds_ab the bitmap of the touched
// tokens, its 16-bit popcount prefixes, and at lds_cnt the per-rank words {history count | bias entries << 20 | claimed}
// and 16-bit indices of each rank's first bias entry.
// Returns false when the row has to go to the three-pass code (uniform over the workgroup; nothing has been written for it, and a
// shared row's workspace is as the launch found it); finisher: this workgroup is the one that would do that.
template <int DT, bool MASKED, bool SHARED>
__device__ __forceinline__ bool short_row(const BatchArgs& A, const uint32_t row, const uint32_t part, const uint32_t n_parts, ShortShared& S, bool& finisher) {
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
    uint16_t* wprefix = reinterpret_cast<uint16_t*>(lds + A.lds_ab + nW * 4u);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(lds + A.lds_cnt);
    uint16_t* first = reinterpret_cast<uint16_t*>(cnt + A.patch_cap);

    // The row in vectors: the whole ones, and the few tokens behind them (none, of most vocabularies) one by one after the sweep.
    // Masked fp32 rows: all of them, the last read where it ends with the row and moved down. (Either way for the registers'
    // sake, measured when batches of any size came here: moved vectors spill them in the bf16 kernels - unmasked, 1000 rows of 24896: 118 us against 72; masked, 300 rows of
    // 151936: 102 against 89, 1024 of 262144: 445 against 411 -, clamped whole ones in the masked fp32 kernel - 300 rows of
    // 151936: 99 us against 81, 1024 of 262144: 430 against 390.)
    constexpr bool MOVED = MASKED && DT == 0;
    const uint32_t nv = MOVED ? (V + TPV - 1u) / TPV : V / TPV, n_odd = MOVED ? 0u : V % TPV;
    const uint32_t j_part = MOVED && V % TPV ? nv - 1u : 0xffffffffu;
    // the vectors [j0, j1) and the tokens of this workgroup: the row, or a shared row's slice
    const uint32_t nvp = SHARED ? (nv + n_parts - 1u) / n_parts : nv, j0 = SHARED ? min(part * nvp, nv) : 0u, j1 = SHARED ? min(j0 + nvp, nv) : nv;
    const uint32_t tok0 = j0 * TPV, tok1 = SHARED && part != n_parts - 1u ? j1 * TPV : V, n_tok = tok1 - tok0;
    finisher = !SHARED;
    auto vector_at = [&](uint32_t j) __attribute__((always_inline)) {
        if (MOVED) return row_vector<DT>(base, SHARED ? min(j, j1 - 1u) : j, V);
        const LooseVec v = *reinterpret_cast<const LooseVec*>(base + min(j, j1 - 1u) * 16u);
        return make_uint4(v.x, v.y, v.z, v.w);
    };
    auto word_at = [&](uint32_t j) __attribute__((always_inline)) {
        return MOVED ? min((SHARED ? min(j, j1 - 1u) : j) * TPV, V - 1u) >> 5 : (min(j, j1 - 1u) * TPV) >> 5;
    };

    // the head of the slice is asked for before anything else
    // (every load of the row is unconditional, its index clamped to the slice, and brings the vector's word of the allow
    // mask with it: a load behind a branch makes the compiler wait for every load before it)
    uint4 hq[kShortHead];
    uint32_t hna[kShortHead];
#pragma unroll
    for (uint32_t k = 0; k < kShortHead; ++k) {
        const uint32_t j = j0 + k * WS_BLOCK + t;
        hq[k] = vector_at(j);
        hna[k] = MASKED ? allow[word_at(j)] : 0xffffffffu;
    }
    for (uint32_t b = t; b < 4096u; b += WS_BLOCK) head_cnt[b] = 0u;
    // (the tables of the touched tokens as well, while the parameters travel: their sizes are the launch's, not the row's)
    if (A.hist || A.bias_ids) {
        for (uint32_t w = t; w < nW; w += WS_BLOCK) touched[w] = 0u;
        for (uint32_t r = t; r < A.patch_cap; r += WS_BLOCK) {
            cnt[r] = 0u;
            first[r] = 0xffffu;
        }
    }

    const LeanRowParams P = load_row_params(A, row);
    WSS_MARK(0);  // parameters in
    const float inv_t = P.inv_t;
    const uint32_t top_k = P.top_k, nh = P.nh, nb = P.nb;
    const double top_p = P.top_p, min_p = P.min_p;
    // rows this code does not take
    const bool by_k = top_k >= 1u && top_k <= kShortMaxK && top_k <= V;  // the top_k largest decide
    const bool by_p = top_k == 0u && min_p > 0.0 && min_p <= 1.0;      // no top-k: what the min-p floor lets through decides
    const bool not_mine = !(by_k || by_p) || !(inv_t > 0.f) || nh + nb > A.patch_cap;
    const int32_t* hist_ids = A.hist + P.h0;
    const int32_t* bias_ids = A.bias_ids + P.b0;
    const float* bias_vals = A.bias_vals + P.b0;

    // ---- the bitmap of the touched tokens, their ranks, per-rank history counts and bias entries (phase 0 of ws_sample.h)
    uint32_t n_touched = 0;
    constexpr uint32_t kIds = 4u;  // ids a thread keeps in registers: the first 4096 of the history, the first 1024 bias entries
    uint32_t hid[kIds], bid = 0xffffffffu;
    if (!not_mine && nh + nb > 0u) {
#pragma unroll
        for (uint32_t k = 0; k < kIds; ++k) hid[k] = k * WS_BLOCK + t < nh ? static_cast<uint32_t>(hist_ids[k * WS_BLOCK + t]) : 0xffffffffu;
        if (t < nb) bid = static_cast<uint32_t>(bias_ids[t]);
        __syncthreads();  // (the tables were cleared at the top)
        auto mark = [&](uint32_t id) {
            if (id < V) atomicOr(&touched[id >> 5], 1u << (id & 31u));
        };
#pragma unroll
        for (uint32_t k = 0; k < kIds; ++k)
            if (k * WS_BLOCK < nh) mark(hid[k]);
        // (ids beyond those in registers: four loads on their way together, not one trip to memory each)
        auto four = [&](const int32_t* ids, uint32_t n, uint32_t j0, uint32_t (&e)[4]) {
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) e[k] = j0 + k * WS_BLOCK + t < n ? static_cast<uint32_t>(ids[j0 + k * WS_BLOCK + t]) : 0xffffffffu;
        };
        for (uint32_t j0 = kIds * WS_BLOCK; j0 < nh; j0 += 4u * WS_BLOCK) {
            uint32_t e[4];
            four(hist_ids, nh, j0, e);
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) mark(e[k]);
        }
        mark(bid);
        for (uint32_t j0 = WS_BLOCK; j0 < nb; j0 += 4u * WS_BLOCK) {
            uint32_t e[4];
            four(bias_ids, nb, j0, e);
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) mark(e[k]);
        }
        __syncthreads();
        // popcount prefixes: five consecutive words a thread and round (one round up to 163840 tokens)
        constexpr uint32_t kChunk = 5u;
        uint32_t run_total = 0;
        for (uint32_t w0 = 0; w0 < nW; w0 += kChunk * WS_BLOCK) {
            const uint32_t wb = w0 + t * kChunk;
            uint32_t wd[kChunk], local = 0;
#pragma unroll
            for (uint32_t k = 0; k < kChunk; ++k) {
                wd[k] = wb + k < nW ? touched[wb + k] : 0u;
                local += __popc(wd[k]);
            }
            uint32_t total;
            uint32_t run = run_total + block_excl_scan(local, S.red_u, &total);
#pragma unroll
            for (uint32_t k = 0; k < kChunk; ++k) {
                if (wb + k < nW) wprefix[wb + k] = static_cast<uint16_t>(run);
                run += __popc(wd[k]);
            }
            run_total += total;
        }
        __syncthreads();
        n_touched = run_total;
        auto rank = [&](uint32_t id) { return static_cast<uint32_t>(wprefix[id >> 5]) + __popc(touched[id >> 5] & ((1u << (id & 31u)) - 1u)); };
        auto count = [&](uint32_t id) {
            if (id < V) atomicAdd(&cnt[rank(id)], 1u);
        };
        auto bias_entry = [&](uint32_t id, uint32_t j) {
            if (id < V) {
                const uint32_t r = rank(id);
                atomicAdd(&cnt[r], 1u << 20);
                // (the smallest index: 16-bit atomics do not exist, so the word that holds two of them takes a minimum of its own half)
                uint32_t* w32 = reinterpret_cast<uint32_t*>(first) + (r >> 1);
                const uint32_t sh = (r & 1u) * 16u;
                uint32_t seen = *w32;
                while (((seen >> sh) & 0xffffu) > j) {
                    const uint32_t want_w = (seen & ~(0xffffu << sh)) | (j << sh);
                    const uint32_t got = atomicCAS(w32, seen, want_w);
                    if (got == seen) break;
                    seen = got;
                }
            }
        };
#pragma unroll
        for (uint32_t k = 0; k < kIds; ++k)
            if (k * WS_BLOCK < nh) count(hid[k]);
        for (uint32_t j0 = kIds * WS_BLOCK; j0 < nh; j0 += 4u * WS_BLOCK) {
            uint32_t e[4];
            four(hist_ids, nh, j0, e);
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) count(e[k]);
        }
        bias_entry(bid, t);
        for (uint32_t j0 = WS_BLOCK; j0 < nb; j0 += 4u * WS_BLOCK) {
            uint32_t e[4];
            four(bias_ids, nb, j0, e);
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) bias_entry(e[k], j0 + k * WS_BLOCK + t);
        }
        __syncthreads();
    }

    WSS_MARK(1);  // bitmap done
    // one vector: its tokens as floats, masked-out / touched / NaN ones as -inf
    auto unpack = [&](uint4 q, uint32_t na, uint32_t j, float (&x)[TPV]) {
        const uint32_t i0 = j * TPV;
        if (MOVED && j_part != 0xffffffffu && j == j_part) q = part_vector<DT>(q, TPV - V % TPV);  // (uniform before per lane)
        uint32_t invalid = 0u;  // bit e: token e does not count here
        if (MASKED) invalid = ~(na >> (i0 & 31u));
        if (n_touched) invalid |= touched[i0 >> 5] >> (i0 & 31u);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (uint32_t e = 0; e < TPV; ++e) {
            uint32_t bits = DT == 0 ? w[e] : ((e & 1u) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
            bits |= static_cast<uint32_t>(static_cast<int32_t>(invalid << (31u - e)) >> 31);  // -> NaN
            x[e] = fmaxf(__uint_as_float(bits), -INFINITY);
        }
    };

    // the first two batches behind the head are asked for now: they travel while the threshold is worked out
    constexpr uint32_t KB = 4;  // vectors a thread and batch, two batches in flight
    uint4 qa[KB], qb[KB];
    uint32_t naa[KB], nab[KB];
    const uint32_t jb = j0 + kShortHead * WS_BLOCK;
    auto load = [&](uint4 (&q)[KB], uint32_t (&na)[KB], uint32_t jbase) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t k = 0; k < KB; ++k) {
            const uint32_t j = jbase + k * WS_BLOCK + t;
            q[k] = vector_at(j);
            na[k] = MASKED ? allow[word_at(j)] : 0xffffffffu;
        }
    };
    load(qa, naa, jb);
    load(qb, nab, jb + KB * WS_BLOCK);

    // ---- the threshold: the head's logits counted in 4096 bins of 1/64 e-fold below the head's maximum
    float ref = -INFINITY;
    const uint32_t n_head_vec = min(j1 - j0, kShortSample * WS_BLOCK);
    {
        float x[TPV];
#pragma unroll
        for (uint32_t k = 0; k < kShortSample; ++k) {
            const uint32_t j = j0 + k * WS_BLOCK + t;
            if (j < j1) {
                unpack(hq[k], hna[k], j, x);
#pragma unroll
                for (uint32_t e = 0; e < TPV; ++e) ref = fmaxf(ref, x[e]);
            }
        }
        ref = block_max(ref, S.red_f);  // (its barriers also publish the zeroed counts)
    }
    const float c64 = inv_t * 64.f;
    float thr = -INFINITY;  // tokens above it are listed
    // tokens to list: the count above a threshold fitted to a sample of the row scatters like the square root of the
    // sample's rank: half of top_k on top, 150 at least; of a slice its share of those. (A slice that is the sample itself: the
    // count is exact but for a bin's tokens, and what matters is that no part holds more of the row's top_k than it lists.)
    const uint32_t n_head = n_head_vec == j1 - j0 ? n_tok : min(n_head_vec * TPV, n_tok);
    // (a head that is the whole row: the count is exact but for the tokens of a bin, and twice top_k will do. 156 rows of
    // 24896, Zipfian, top-k 25: 30.6 us with 191 tokens to list, most of them in a second round of counting, 21 with 56)
    const uint32_t want = !SHARED ? min(n_head >= V ? 2u * top_k + 6u : 0xffffffffu, top_k + max(top_k >> 1, 150u) + 16u)
                          : n_head >= n_tok ? 2u * ((top_k + n_parts - 1u) / n_parts) + 6u
                                            : (top_k + max(top_k >> 1, 150u) + n_parts - 1u) / n_parts + 16u;
    bool list_all = by_k && n_head >= n_tok && want >= n_tok;
    if (by_p && ref > -INFINITY) thr = __fadd_rn(ref, __fdiv_rn(static_cast<float>(log(min_p)) - 0.02f, inv_t));  // (0.02 e-folds below the floor: roundings)
    if (!not_mine && by_k && ref > -INFINITY && !list_all) {
        // rank in the head that about `want` tokens of the slice lie above
        const uint64_t r_star64 = (static_cast<uint64_t>(n_head) * want + n_tok - 1u) / n_tok;
        const uint32_t r_star = static_cast<uint32_t>(r_star64 < 4u ? 4u : r_star64);
        // The bins near the top are all that matters (the r_star-th largest of the head is one of its largest per cent
        // or so): first only the tokens within 8 e-folds of the head's maximum are counted - an LDS atomic each, and a
        // sixth of the tokens -, the others only when those turn out to be fewer than r_star.
        constexpr float kNear = 512.f;
        uint32_t b_star = 0xffffffffu;
        if (t == 0) S.s_w[0] = 0xffffffffu;  // (the bin, once found; the barrier behind the counting publishes this)
        for (int round = 0; round < 2; ++round) {  // uniform
            float x[TPV];
#pragma unroll
            for (uint32_t k = 0; k < kShortSample; ++k) {
                const uint32_t j = j0 + k * WS_BLOCK + t;
                if (j < j1) {
                    unpack(hq[k], hna[k], j, x);
#pragma unroll
                    for (uint32_t e = 0; e < TPV; ++e) {
                        const float d = fminf(__fmul_rn(__fsub_rn(ref, x[e]), c64), 4095.f);  // (-inf, and anything 64 e-folds down: the last bin)
                        // (the last bin - masked-out tokens, nine in ten of some rows - is nobody's threshold and is
                        // not counted: the additions of a wave to that one word would queue up sixty-four deep)
                        if (round == 0 ? d < kNear : (d >= kNear && d < 4095.f)) atomicAdd(&head_cnt[static_cast<uint32_t>(d)], 1u);
                    }
                }
            }
            __syncthreads();
            const uint4 c4 = *reinterpret_cast<const uint4*>(&head_cnt[4u * t]);
            const uint32_t mine = c4.x + c4.y + c4.z + c4.w;
            uint32_t total;
            const uint32_t before = block_excl_scan(mine, S.red_u, &total);
            if (before < r_star && before + mine >= r_star) {  // the bin in which the head's r_star-th largest lies
                uint32_t run = before, b = 4u * t;
                const uint32_t c[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    if (run < r_star && run + c[k] >= r_star) b = 4u * t + k;
                    run += c[k];
                }
                S.s_w[0] = b;
            }
            __syncthreads();
            b_star = S.s_w[0];
            if (b_star != 0xffffffffu) break;
        }
        if (b_star >= 4095u) list_all = true;  // (fewer than r_star tokens above the last bin: everything is listed)
        else thr = __fsub_rn(ref, __fdiv_rn(static_cast<float>(b_star + 1u), c64));
    }
    if (list_all) thr = -INFINITY;
    if (t == 0) {
        S.s_w[1] = 0u;  // tokens listed
        S.s_w[2] = 0u;  // the list ran over
    }
    __syncthreads();  // (the counts and the bin have been read: the list takes the counts' place)

    WSS_MARK(2);  // threshold known
    // ---- the sweep: maximum, sum of exp against `ref`, tokens above the threshold to the list
    const float k2 = inv_t * 1.44269504088896340736f;
    const float k2lo = static_cast<float>(static_cast<double>(inv_t) * 1.44269504088896340736 - static_cast<double>(k2));
    float m = -INFINITY, s = 0.f;
    auto push = [&](float x, uint32_t id, bool yes) {  // (one LDS atomic a listed token: they are few)
        if (yes) {
            const uint32_t slot = atomicAdd(&S.s_w[1], 1u);
            if (slot < kShortCap) list[slot] = key64(x, id);
            else S.s_w[2] = 1u;
        }
    };
    auto take = [&](const uint4& q, uint32_t na, uint32_t j) {
        float x[TPV];
        unpack(q, na, j, x);
        float vm = -INFINITY;
#pragma unroll
        for (uint32_t e = 0; e < TPV; ++e) {
            vm = fmaxf(vm, x[e]);
            const float a = fmaxf(__fsub_rn(x[e], ref), -1e30f);
            s += __builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2));  // (v_exp_f32: arguments below -126 give 0, which is what they are worth)
        }
        m = fmaxf(m, vm);
        if (__ballot(vm > thr)) {  // uniform: a vector with a token for the list (a few per thousand)
#pragma unroll
            for (uint32_t e = 0; e < TPV; ++e) push(x[e], j * TPV + e, x[e] > thr);
        }
    };
    if (!not_mine && ref > -INFINITY) {  // (a head without any token: the row goes the other way)
#pragma unroll
        for (uint32_t k = 0; k < kShortHead; ++k) {
            const uint32_t j = j0 + k * WS_BLOCK + t;
            if (j < j1) take(hq[k], hna[k], j);
        }
        auto eat = [&](const uint4 (&q)[KB], const uint32_t (&na)[KB], uint32_t jbase) __attribute__((always_inline)) {
#pragma unroll
            for (uint32_t k = 0; k < KB; ++k) {
                const uint32_t j = jbase + k * WS_BLOCK + t;
                if (j < j1) take(q[k], na[k], j);
            }
        };
        if (jb < j1) {
            for (uint32_t jc = jb; jc < j1; jc += 2u * KB * WS_BLOCK) {
                eat(qa, naa, jc);
                load(qa, naa, jc + 2u * KB * WS_BLOCK);
                eat(qb, nab, jc + KB * WS_BLOCK);
                load(qb, nab, jc + 3u * KB * WS_BLOCK);
            }
        }
    }

    if (n_odd && tok1 == V && !not_mine && ref > -INFINITY) {  // uniform: the tokens behind the last whole vector
        float x = -INFINITY;
        const uint32_t id = nv * TPV + t;
        if (t < n_odd && (!MASKED || ((allow[id >> 5] >> (id & 31u)) & 1u)) && !(n_touched && ((touched[id >> 5] >> (id & 31u)) & 1u)))
            x = fmaxf(DT == 0 ? reinterpret_cast<const float*>(base)[id] : bf16_to_f32(reinterpret_cast<const uint16_t*>(base)[id]), -INFINITY);
        if (t < n_odd) {
            const float a = fmaxf(__fsub_rn(x, ref), -1e30f);
            s += __builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2));
            m = fmaxf(m, x);
        }
        push(x, id, t < n_odd && x > thr);
    }
    WSS_MARK(3);  // sweep done
    // ---- the touched tokens: adjusted logit (bias entries in list order, then repetition, then frequency /
    // presence, as ws_sample.h applies them), into the maximum, the sum and - above the threshold - the list
    if (!not_mine && n_touched) {
        constexpr uint32_t kClaim = 0x80000000u;
        auto rank = [&](uint32_t id) { return static_cast<uint32_t>(wprefix[id >> 5]) + __popc(touched[id >> 5] & ((1u << (id & 31u)) - 1u)); };
        // History and bias entries are one sequence here (whoever claims a token applies both kinds), up to eight
        // entries a thread at a time: the ids not in registers asked for together, then the claims, then the claimed
        // tokens' logits asked for together, then the arithmetic - three trips to memory a round
        // (n_live: entries left in this round, so that empty slots issue nothing).
        const uint32_t n_all = nh + nb;
        auto some = [&](auto ks, uint32_t j0) {
            constexpr uint32_t KS = decltype(ks)::value;
            const uint32_t n_live = n_all - j0;
            uint32_t id[KS], old[KS], r[KS];
            float raw[KS];
#pragma unroll
            for (uint32_t k = 0; k < KS; ++k) {
                id[k] = 0xffffffffu;
                if (k * WS_BLOCK >= n_live) continue;  // uniform
                const uint32_t j = j0 + k * WS_BLOCK + t;
                if (j0 == 0u && k < kIds && (k + 1u) * WS_BLOCK <= nh) id[k] = hid[k];  // (uniform: a whole round of history ids in registers)
                else if (j < nh) id[k] = static_cast<uint32_t>(hist_ids[j]);
                else if (j < n_all) id[k] = static_cast<uint32_t>(bias_ids[j - nh]);
            }
#pragma unroll
            for (uint32_t k = 0; k < KS; ++k) {
                old[k] = kClaim;
                r[k] = 0u;
                if (k * WS_BLOCK < n_live && id[k] < tok1 && (!SHARED || id[k] >= tok0)) {
                    r[k] = rank(id[k]);
                    old[k] = atomicOr(&cnt[r[k]], kClaim);
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < KS; ++k) {
                raw[k] = -INFINITY;
                if (k * WS_BLOCK < n_live && !(old[k] & kClaim)) {
                    // (the logit only where the mask allows the token: nine in ten of a masked row's history ids would
                    // fetch a sector each for nothing, half as many bytes again as the row itself)
                    const bool allowed = !MASKED || ((allow[id[k] >> 5] >> (id[k] & 31u)) & 1u);
                    if (allowed)
                        raw[k] = DT == 0 ? reinterpret_cast<const float*>(base)[id[k]] : bf16_to_f32(reinterpret_cast<const uint16_t*>(base)[id[k]]);
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < KS; ++k) {
                if (k * WS_BLOCK >= n_live) continue;  // uniform
                const bool have = !(old[k] & kClaim);
                float x = -INFINITY;
                if (have) {
                    const uint32_t c = old[k] & 0xfffffu, n_bias = (old[k] >> 20) & 0x7ffu;
                    x = fmaxf(raw[k], -INFINITY);
                    if (__ballot(n_bias != 0u)) {  // uniform
                        const uint32_t j = n_bias ? first[r[k]] : 0u;
                        if (n_bias) x = __fadd_rn(x, bias_vals[j]);
                        x = add_other_bias(n_bias > 1u, id[k], j, x, bias_ids, bias_vals, nb);
                    }
                    if (c) {
                        x = x > 0.f ? __fdiv_rn(x, P.rep) : __fmul_rn(x, P.rep);
                        x = __fsub_rn(x, __fadd_rn(__fmul_rn(P.freq, static_cast<float>(c)), P.pres));
                    }
                    x = fmaxf(x, -INFINITY);
                    m = fmaxf(m, x);
                    const float a_ = fmaxf(__fsub_rn(x, ref), -1e30f);
                    s += __builtin_amdgcn_exp2f(fmaf(a_, k2lo, a_ * k2));
                }
                push(x, id[k], have && x > thr);
            }
        };
        // (four entries a thread when that is all there is: the wider code costs a short list a microsecond)
        if (n_all <= 4u * WS_BLOCK) some(std::integral_constant<uint32_t, 4u>{}, 0u);
        else
            for (uint32_t j0 = 0; j0 < n_all; j0 += 8u * WS_BLOCK) some(std::integral_constant<uint32_t, 8u>{}, j0);
    }
    WSS_MARK(4);  // touched tokens in
#ifdef WS_SHORT_TIMERS
    if (lane == 0u) atomicMax(reinterpret_cast<int*>(&S.marks[13]), __float_as_int(static_cast<float>(clock64() - wss_t0)));  // the slowest wave's
#endif
    double z;  // the sum against `ref`
    {          // the block's maximum and sum with one barrier between them
        const float wm_ = wave_max(m);
        const double ws_ = wave_sum(static_cast<double>(s));
        __syncthreads();
        if (lane == 0u) {
            S.red_f[wv] = wm_;
            S.red_d[wv] = ws_;
        }
        __syncthreads();
        m = S.red_f[0];
        z = S.red_d[0];
#pragma unroll
        for (uint32_t w = 1; w < WS_WAVES; ++w) {
            m = fmaxf(m, S.red_f[w]);
            z += S.red_d[w];
        }
    }
    WSS_MARK(9);
    uint32_t n_list = S.s_w[1];
    bool bad = not_mine || S.s_w[2] != 0u || n_list > kShortCap || !(ref > -INFINITY) || !(m > -INFINITY) || !(__fsub_rn(m, ref) * inv_t < 80.f);
    // Tokens above `ref` can be most of the sum, and the larger the exponent, the less of a fraction 32 bits leave it (1.2e-6 of
    // the normaliser where the maximum lies 60 units above the head's; 2e-7 up to the four units below which nothing is done):
    // they are all on the list, and their terms are taken out and put back in 64 bits.
    if (!bad && __fsub_rn(m, ref) * inv_t > 4.f) {  // uniform
        double more = 0.0;
        for (uint32_t k = t; k < n_list; k += WS_BLOCK) {
            const float x = unkey32(static_cast<uint32_t>(list[k] >> 32)), a = __fsub_rn(x, ref);
            if (a > 0.f) more += exp((static_cast<double>(x) - static_cast<double>(ref)) * static_cast<double>(inv_t)) - static_cast<double>(__builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2)));
        }
        z += block_sum(more, S.red_d);
    }
    float thr_max = thr;

    // ---- a shared row: the parts' lists, maxima and sums meet in the row's workspace; the last one to arrive goes on
    if constexpr (SHARED) {
        unsigned char* work = A.work + static_cast<size_t>(row) * kShortSplitRowBytes;
        unsigned long long* glist = reinterpret_cast<unsigned long long*>(work);
        uint32_t* ctrl = reinterpret_cast<uint32_t*>(work + kShortSplitCtrl);
        const uint32_t region = kShortCap / n_parts;  // every part has its own stretch of the list: nothing to reserve
        if (n_list > region) bad = true;
        if (t == 0) {
            uint32_t* mine = ctrl + 64u + 8u * part;
            __hip_atomic_store(&mine[0], key32(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&mine[1], key32(thr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // the sum as it is, against the part's `ref`, and `ref` with it (against the `ref` of a bad part it may not be a number)
            __hip_atomic_store(reinterpret_cast<unsigned long long*>(&mine[2]), static_cast<unsigned long long>(__double_as_longlong(bad ? 0.0 : z)), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&mine[4], bad ? 0xffffffffu : n_list, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&mine[5], key32(ref), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (!bad)
            for (uint32_t k = t; k < n_list; k += WS_BLOCK)
                __hip_atomic_store(&glist[part * region + k], static_cast<unsigned long long>(list[k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (device-scope accesses and this wait make the meeting sound without a release or an acquire, which would write back and
        // invalidate whole caches: as in ws_few.h)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // every wave's stores have arrived
        if (t == 0) S.s_w[5] = __hip_atomic_fetch_add(&ctrl[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (S.s_w[5] != n_parts - 1u) return true;  // not the last: done
        finisher = true;
        // The keys are asked for right away, every place of every stretch: which of them count is known when the parts' words
        // are in. Lane p of the first wave reads part p's.
        constexpr uint32_t kSlots = kShortCap / WS_BLOCK;
        uint64_t got[kSlots];
#pragma unroll
        for (uint32_t i = 0; i < kSlots; ++i) got[i] = __hip_atomic_load(&glist[i * WS_BLOCK + t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();  // (everybody is done with its own list)
        if (wv == 0u) {   // (one wave: sixteen doing the same arithmetic side by side take four times as long)
            float mp = -INFINITY, tp = -INFINITY, rp = -INFINITY;
            double zp = 0.0;
            uint32_t np = 0u;
            if (lane < n_parts) {
                const uint32_t* words = ctrl + 64u + 8u * lane;
                mp = unkey32(__hip_atomic_load(&words[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                tp = unkey32(__hip_atomic_load(&words[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                zp = __longlong_as_double(static_cast<long long>(__hip_atomic_load(reinterpret_cast<const unsigned long long*>(&words[2]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
                np = __hip_atomic_load(&words[4], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                rp = unkey32(__hip_atomic_load(&words[5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            }
            const bool any_bad = __ballot(np == 0xffffffffu) != 0ull;
            if (np == 0xffffffffu) np = 0u;
            const float mm = wave_max(mp), tt = wave_max(tp);
            const double zz = wave_sum(zp > 0.0 ? zp * exp((static_cast<double>(rp) - static_cast<double>(mm)) * static_cast<double>(inv_t)) : 0.0);
            const uint32_t upto = wave_incl_scan(np);  // where the part's keys end in the merged list
            if (lane < n_parts) {
                S.red_u[lane] = np;
                S.bcnt[lane] = upto - np;
            }
            if (lane == 63u) {
                S.red_f[0] = mm;
                S.red_f[1] = tt;
                S.s_d[0] = zz;
                S.bstart[0] = upto;
                S.bstart[1] = any_bad ? 1u : 0u;
            }
        }
        __syncthreads();
        m = S.red_f[0];
        thr_max = S.red_f[1];
        z = S.s_d[0];  // against the row's maximum from here on
        ref = m;
        n_list = S.bstart[0];
        bad = S.bstart[1] != 0u || !(m > -INFINITY);
        const uint32_t region_log2 = static_cast<uint32_t>(__ffs(region)) - 1u;  // (a power of two, as the number of parts is)
#pragma unroll
        for (uint32_t i = 0; i < kSlots; ++i) {
            const uint32_t slot = i * WS_BLOCK + t, p = slot >> region_log2, k = slot - (p << region_log2);
            if (k < S.red_u[p]) {
                list[S.bcnt[p] + k] = got[i];
                __hip_atomic_store(&glist[slot], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // the workspace as the next launch needs it
            }
        }
        if (t < 64u + 8u * n_parts) __hip_atomic_store(&ctrl[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
    }
    WSS_MARK(5);  // parts met
    const uint32_t n_cand = by_k ? top_k : n_list;  // candidates the rules look at
    if (bad || n_list < n_cand || n_cand == 0u || n_cand > kShortCap) return false;
    short_sort(list, n_list, m, S);
    WSS_MARK(6);  // sorted
    // the k-th largest has to lie above the threshold, every part's (below one, the sweep has left out tokens that rank before it);
    // a min-p row's threshold lies below its floor by construction
    const float x_k = unkey32(static_cast<uint32_t>(list[n_cand - 1u] >> 32));
    if ((by_k && !(x_k > thr_max)) || !(x_k > -INFINITY)) return false;
    ShortRow R;
    R.top_p = top_p;
    R.min_p = min_p;
    R.u = batch_uniform(A.rng, P.seed, row, P.step, 0);
    R.z = z * exp((static_cast<double>(ref) - static_cast<double>(m)) * static_cast<double>(inv_t));
    R.inv_t = inv_t;
    R.m = m;
    R.n_cand = n_cand;
    R.by_k = by_k;
    short_rules(list, row, R, S);
#ifdef WS_SHORT_TIMERS
    WSS_MARK(8);
    __syncthreads();
    if (t < 16 && A.kept_logits) A.kept_logits[static_cast<size_t>(row) * A.kept_cap + 100u + t] = t == 15 ? static_cast<float>(n_list) : S.marks[t];
#endif
    return true;
}

template <int DT, bool MASKED, bool SHARED>
__global__ void __launch_bounds__(WS_BLOCK) short_batch_kernel(BatchArgs A) {
    __shared__ ShortShared shared;
    const uint32_t lg = SHARED ? A.split_log2 : 0u, row = blockIdx.x >> lg, part = blockIdx.x & ((1u << lg) - 1u);
    bool finisher;
    if (!short_row<DT, MASKED, SHARED>(A, row, part, 1u << lg, shared, finisher) && finisher) {
        __syncthreads();
        LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(Ap));
        if (Ap->kept_ids) three_pass_row<true>(Ap, row);
        else three_pass_row<false>(Ap, row);
    }
}

}  // namespace ws
