// The sampler for bf16 rows: one workgroup of 1024 threads a row, which keeps the row in registers as it came and counts its
// tokens by their value.
//
// A bf16 logit is one of a few thousand values - 128 to an octave - so a row's histogram needs no arithmetic on the logits and
// loses nothing: a bin is a value, and its tokens tie. Cut and draw are then a bin and a place among its tied tokens, whatever their
// number, and the token at a place is found by comparing the row's registers with the value and counting in id order. Nothing is
// sorted, no bin is read again, and a row may have a top-k, a top-p and a min-p in any combination, or none: a top-k is a place in
// the order like the others (src/sampling/sampler.cpp:15-78, :118-146).
//
//   * 19 vectors of 128 bits a thread hold 155648 tokens, six of them on their way at a time. Longer rows are read again behind the
//     19th when the drawn token is looked for.
//   * A token's bin by packed 16-bit integer instructions, two tokens each: saturating subtractions, a maximum and a minimum
//     (code_pair), then one 32-bit LDS addition a token. Bins go from 512 down to 2^-23, one for everything nearer to zero, and from
//     -2^-23 down to -512. Masked-out tokens become NaN in place: the last bins, one to a lane, where nothing is looked at.
//   * The touched tokens (history, bias list) are counted like the others and taken out again afterwards. Their ids are ranked by a
//     bitmap and its prefix sums, in four steps between the row's rounds, so that the trips to memory for the ids and for their
//     logits pass meanwhile. Their adjusted logits are 32-bit floats: they are listed by the group of eight bins they fall in - count,
//     and mass in fixed point against the group's top or the row's maximum -, and those of the bin that a cut or the draw falls in are put in
//     order there.
//   * A thread has eight bins for the prefix sums; one wave then looks for the cuts and the draw, without a barrier.
//
// What bounds it: eight waves' worth of LDS additions at random words, some eight clocks an instruction of 64 lanes - 10 us for 151936
// tokens, about what 256 such rows take to read -, and behind it a chain of eight barriers, 13 us (clocks of a 64-row batch with
// 1024-id histories: 28 K until the last wave is through the row, 3 K touched tokens, 10 K prefix sums, 7 K cuts and draw, 7 K the
// token's id). Asking for the whole row at once made the first vector wait for the last to be asked for (+15 K); the registers'
// vectors and the search for the cuts together spilled (+10 K); a stretch of 64 bins at a time for the prefix sums, over all waves, was
// 5 K slower. Measured (151936 bf16, us): 256 rows of top-p 0.9, Zipfian, 2048-id histories 48.9 -> 40; 64 rows of which nothing is known
// 69 -> 28; 256 rows of top-k 50 52 -> 29; 256 of top-k 1000, masked 71 -> 32; 8 rows of top-p 43 -> 26; without a filter 77 -> 51;
// 100 rows of 50257 tokens 47 -> 19, 300 rows of 262144 with a mask 225 -> 102.
#pragma once
#include "ws_lean.h"

namespace ws {

constexpr uint32_t kCodeTop = (127u + 9u) << 7;   // bf16 code of 512: logits from there up are not for this kernel
constexpr uint32_t kCodeZero = (127u - 23u) << 7;  // code of 2^-23: everything up to it, of either sign, is one bin
constexpr uint32_t kCodeBins = 8192u, kCodeFold = kCodeTop - kCodeZero;  // bins, and the bin of zero: the middle one, [-2^-23, 2^-23)
static_assert(kCodeFold * 2u == kCodeBins, "as many bins above zero as from there down");
constexpr uint32_t kCodeTail = kCodeBins - 64u;   // the last 64 bins, from -384 down: masked, touched, and nothing that counts
constexpr uint32_t kCodeGroups = kCodeBins / 8u;  // eight bins each, one group to a thread
constexpr uint32_t kCodeSub = 512u;               // touched tokens in one bin, where a cut or the draw falls in it
constexpr uint32_t kCodeFixBits = 44u;            // fixed point of the groups' touched masses (65535 of them at most)
constexpr float kCodeWide = 4.f;                  // e-folds a group spans from which its touched masses are not taken against its top
constexpr uint32_t kCodeHeldVecs = 19u;           // vectors a thread holds
// Up to here the anchor of a row of logits below 512 lies at most 64 of its bins further above the maximum than it was put (anchor_product's 2^-21): 2900
// of them, 45 e-folds, are left below the maximum. Colder rows lose some to the tail.
constexpr float kCodeMaxInvT = 4096.f;

typedef uint16_t CodePair __attribute__((ext_vector_type(2)));
typedef int16_t CodePairS __attribute__((ext_vector_type(2)));

// the bins of two tokens (16 bits each): 0 the last value below 512 and everything above, the middle bin around zero, `last` bins below it at most
__device__ __forceinline__ CodePair code_pair(uint32_t y, CodePair last) {
    const CodePairS s = __builtin_bit_cast(CodePairS, y);
    const CodePair u = __builtin_bit_cast(CodePair, y);
    constexpr int16_t kZ = static_cast<int16_t>(kCodeZero - 1u);
    constexpr uint16_t kT = static_cast<uint16_t>(kCodeTop - 1u), kN = static_cast<uint16_t>(0x8000u + kCodeZero);
    const CodePair above = __builtin_elementwise_sub_sat(CodePair{kT, kT}, __builtin_bit_cast(CodePair, __builtin_elementwise_max(s, CodePairS{kZ, kZ})));
    const CodePair below = __builtin_elementwise_min(__builtin_elementwise_sub_sat(u, CodePair{kN, kN}), last);
    return above + below;
}
// a bin's value: its smallest logit, the only one but for touched tokens
__device__ __forceinline__ float code_value(uint32_t bin) {
    const uint32_t h = bin < kCodeFold ? kCodeTop - 1u - bin : (bin == kCodeFold ? 0u : 0x8000u + kCodeZero + (bin - kCodeFold));
    return __uint_as_float(h << 16);
}
// the bin of any logit: the one whose value is the largest that is not above it
__device__ __forceinline__ uint32_t code_bin(float x) {
    const uint32_t u = __float_as_uint(x);
    if (!(u >> 31)) {
        const uint32_t h = u >> 16;
        return h >= kCodeTop ? 0u : kCodeTop - 1u - max(h, kCodeZero - 1u);
    }
    const uint32_t h = ((u & 0x7fffffffu) + 0xffffu) >> 16;
    return kCodeFold + (h <= kCodeZero ? 0u : min(h - kCodeZero, kCodeFold - 1u));
}
// The eight values of a group lie in one octave, `step` apart; no logit of the group lies a step above the first.
__device__ __forceinline__ float code_group_step(uint32_t g) { return __fsub_rn(code_value(g * 8u), code_value(g * 8u + 1u)); }
__device__ __forceinline__ double code_group_top(uint32_t g) { return static_cast<double>(code_value(g * 8u)) + static_cast<double>(code_group_step(g)); }

// each half: zero stays zero, everything else is one
__device__ __forceinline__ CodePair code_one(uint32_t y) {
    CodePair d;  // (written out: the compiler makes two comparisons and a permutation of it)
    asm("v_pk_min_u16 %0, %1, 1 op_sel_hi:[1,0]" : "=v"(d) : "v"(y));
    return d;
}

// sum of a row of sixteen lanes up to and with the lane
template <class T>
__device__ __forceinline__ T row_incl_scan(T v) {
    v += dpp_or_zero<0x111, 0xf>(v);
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    return v;
}
// what lanes of a wave have stored in LDS is there for its other lanes (they run in step: the order of the code is all it takes)
__device__ __forceinline__ void lanes_meet() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

#ifdef WS_CODE_TIMERS  // (debug builds: clocks since the kernel began, to `margin`, 32 doubles a row)
#define WSC_MARK(k) \
    if (threadIdx.x == 0) S.marks[k] = clock64() - S.t0
#define WSC_MARK2(k) \
    if (lane == 0u) S.marks[k] = clock64() - S.t0
#else
#define WSC_MARK(k)
#define WSC_MARK2(k)
#endif
struct CodeShared {
#ifdef WS_CODE_TIMERS
    long long t0, marks[32];
#endif
    double s_exp[128];  // kExpHi, kExpLo
    double u, floor_below;  // the row's uniform; how far below the maximum the min-p floor lies
    double red_d[WS_WAVES];
    uint64_t sub[kCodeSub], sorted[kCodeSub];
    unsigned long long bin_mass[8];
    uint32_t bin_cnt[8];
    uint32_t red_u[WS_WAVES], red_v[WS_WAVES];
    uint32_t head_bin;  // first bin of the row's head
    uint32_t top_bin, top_key, bad;  // the first bin that holds a token; the touched tokens' largest logit; a logit this kernel does not take
    uint32_t n_out;    // masked-out tokens, where it matters
    uint32_t waiting;  // whether a touched token's mass waits for the largest of them
    // the drawn token, when it is one of a bin's tied tokens: their value (both halves), the place among them, the touched ones among
    // them (ids in ascending order in `sorted`), and the outcome
    uint32_t state, value2, place, n_eq, eq_at, token;  // state: 0 the row is handed back, 1 `token` it is, 2 it is to be found, 3 and 4 see walk
    // a row without a filter whose draw lies behind its 256 largest: the last of these is `token` (4: is to be found), its logit, and the mass to
    // walk over the others in id order
    float walk_below;
    double walk;
    // the other answers, and what the margins are made of
    uint32_t n_kept;
    double unit, kept_mass, gap_top_p, of_top_p, near_min_p, gap_draw;
    // running sums up to and with each wave's groups; the groups the first cut falls in (against the float normaliser, or by rank, and
    // against the exact one) and the draw, should the cut be where the running mass just reaches its target
    double wave_mass[WS_WAVES];
    uint32_t wave_cnt[WS_WAVES];
    uint32_t g_first[2], g_draw;
};

// what is looked for: a token's place; the first at which the running mass reaches a value; the first below a mass; the first that passes a
// running mass - and what is found: its rank, the running mass with and without it, its own, and the token, or its place among the
// tied ones of its bin
enum CodeLook { kByRank, kByMass, kByPassing, kPast };
struct CodeAt {
    bool ok;
    uint32_t rank, bin, token, place, n_eq, n_above;
    double cin, cex, unit, near;
    float logit;
    uint32_t first;  // rank of its bin's first token
};

// where everything lies in dynamic LDS (ws_abi.hip works out the same sizes: code_lds_bytes)
struct CodeLds {
    uint32_t groups, block, touched, wprefix, cnt, id, raw, pos, stash, total;
};
__host__ __device__ inline CodeLds code_lds(uint32_t V, uint32_t cap, uint32_t copies) {
    CodeLds L;
    const uint32_t nW = (V + 31u) / 32u;
    L.groups = copies * kCodeBins * 4u;
    L.block = L.groups + kCodeGroups * 16u;  // mass (8), count (4), list (4)
    L.touched = L.block + (((V + 511u) / 512u * 4u + 15u) & ~15u);  // tied tokens of 512 neighbours each
    const uint32_t maps = cap ? nW * 4u + ((nW * 2u + 15u) & ~15u) : 0u;
    L.wprefix = L.touched + (cap ? nW * 4u : 0u);
    L.cnt = (L.touched + maps + 15u) & ~15u;
    L.id = L.cnt + cap * 4u;
    L.raw = L.id + cap * 4u;
    L.pos = L.raw + cap * 2u;
    L.total = (L.pos + cap * 2u + 15u) & ~15u;
    // the last wave's vectors while it looks for the cuts (1 KiB each): over the second copy of the counts, which have been brought together by
    // then; with one copy they are read from memory again
    L.stash = kCodeBins * 4u;
    return L;
}

// One row. Returns false when it is left to the three-pass code (nothing has been written for it then). MASKED: the batch has an
// allow mask, TOUCHED: a history or a bias list; NV: vectors a thread holds, NV - 5 of them at least whole rounds of the row.
template <bool MASKED, bool TOUCHED, int NV>
__device__ __forceinline__ bool code_row(const BatchArgs& A, const uint32_t row, CodeShared& S) {
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    const uint32_t V = A.vocab, nW = (V + 31u) >> 5;
    const unsigned char* base = static_cast<const unsigned char*>(A.logits) + static_cast<size_t>(row) * A.row_stride * 2u;
    const uint32_t nv = (V + 7u) >> 3, drop = nv * 8u - V;
    const uint32_t* allow = MASKED ? A.allow + static_cast<size_t>(row) * A.allow_stride : nullptr;

    // ------------------------------------------------------------------ the first of the row's vectors
    uint32_t aw[MASKED ? (NV + 3) / 4 : 1];  // allow words: lane l of a wave holds word l % 16 of the wave's rounds l / 16, + 4, ..
    if (MASKED) {
#pragma unroll
        for (int k = 0; k < (NV + 3) / 4; ++k) aw[k] = allow[min((static_cast<uint32_t>(k) * 4u + (lane >> 4)) * (WS_BLOCK / 4u) + wv * 16u + (lane & 15u), nW - 1u)];
    }
    uint4 q[NV];
    auto load = [&](int c) __attribute__((always_inline)) { q[c] = row_vector<1>(base, static_cast<uint32_t>(c) * WS_BLOCK + t, V); };
    // Vectors of a thread on their way: six (with all of them at once the first would wait for the last to be asked for), and only two of them
    // before the parameters and the history ids, which would come behind them.
    constexpr int kAhead = NV < 6 ? NV : 6;
    load(0);
    load(1);

    const uint32_t cap = TOUCHED ? A.code_cap : 0u;
    const bool two = A.lds_tie != 0u;  // copies of the counts
    const CodeLds L = code_lds(V, cap, two ? 2u : 1u);
    uint32_t* count = reinterpret_cast<uint32_t*>(lds);  // (and, with a second copy, the odd lanes' kCodeBins words on)
    unsigned long long* g_mass = reinterpret_cast<unsigned long long*>(lds + L.groups);
    double* g_pre = reinterpret_cast<double*>(lds + L.groups);  // (later: the mass ranked before the group)
    uint32_t* g_cnt = reinterpret_cast<uint32_t*>(lds + L.groups + kCodeGroups * 8u);
    uint32_t* g_cpre = g_cnt;  // (later: the tokens ranked before it)
    uint32_t* g_list = g_cnt + kCodeGroups;  // (later: where its touched tokens are listed | how many << 16)
    uint32_t* touched = reinterpret_cast<uint32_t*>(lds + L.touched);
    uint16_t* wprefix = reinterpret_cast<uint16_t*>(lds + L.wprefix);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(lds + L.cnt);  // by rank: history count | bias entries << 20; later the adjusted logit
    float* adj = reinterpret_cast<float*>(lds + L.cnt);
    uint32_t* tid = reinterpret_cast<uint32_t*>(lds + L.id);   // by rank: the token
    uint16_t* raw = reinterpret_cast<uint16_t*>(lds + L.raw);  // by rank: its bf16 logit; later: the ranks, group by group
    uint16_t* pos = reinterpret_cast<uint16_t*>(lds + L.pos);  // by rank: its first bias entry; later its place in its group's list
    if (t < 128u) S.s_exp[t] = t < 64u ? kExpHi[t] : kExpLo[t - 64u];
    if (t == 0u) {
        S.top_bin = kCodeBins;
        S.head_bin = kCodeBins;
        S.top_key = 0u;
        S.bad = 0u;
        S.n_out = 0u;
        S.waiting = 0u;
        S.state = 0u;
        S.g_first[0] = S.g_first[1] = S.g_draw = kCodeGroups;
    }
    const LeanRowParams P = load_row_params(A, row);
    const float inv_t = P.inv_t;
    const double top_p = P.top_p, min_p = P.min_p;
    const bool use_top_p = top_p < 1.0, use_min_p = min_p > 0.0;
    // rows this code does not take: a top-p that keeps nothing, a min-p above 1, the race draw, parameters the three-pass code reports (more entries than
    // the batch declares: its tables may have room for up to three of them), temperatures below kCodeMaxInvT's
    const bool open = P.top_k == 0u && !use_top_p && !use_min_p;
    if (!(top_p > 0.0) || !(min_p <= 1.0) || P.race || !(inv_t > 0.f) || !(inv_t <= kCodeMaxInvT) || P.nh + P.nb > (TOUCHED ? A.patch_cap : 0u)) return false;
    if (wv == WS_WAVES - 1u) {  // (the seed by way of a vector register: as scalar arithmetic every wave would work the generator's rounds out)
        uint32_t seed_lo = static_cast<uint32_t>(P.seed);
        asm volatile("" : "+v"(seed_lo));
        const double u_ = batch_uniform(A.rng, (P.seed & 0xffffffff00000000ull) | seed_lo, row, P.step, 0);
        if (lane == 0u) S.u = u_;
    }
    if (wv == WS_WAVES - 2u && use_min_p) {
        const double below = -log(min_p) / static_cast<double>(inv_t);
        if (lane == 0u) S.floor_below = below;
    }
    const int32_t* hist_ids = A.hist + P.h0;
    const int32_t* bias_ids = A.bias_ids + P.b0;
    const float* bias_vals = A.bias_vals + P.b0;
    const uint32_t nh = P.nh, nb = P.nb;

    // ------------------------------------------------------------------ bitmap of the touched ids, prefix per word, count and first
    // bias entry by rank (the row travels meanwhile)
    uint32_t n_touched = 0;  // uniform
    constexpr int kIds = 2;  // history ids a thread keeps at hand
    int32_t hid[kIds] = {-1, -1}, bid = -1;
    uint32_t hraw[kIds] = {}, braw = 0;  // their logits
    if (TOUCHED) {
#pragma unroll
        for (int k = 0; k < kIds; ++k) hid[k] = t + k * WS_BLOCK < nh ? hist_ids[t + k * WS_BLOCK] : -1;
        bid = t < nb ? bias_ids[t] : -1;
    }
#pragma unroll
    for (int c = 2; c < kAhead; ++c) load(c);
    {
        const uint32_t words = L.touched / 4u;
        for (uint32_t i = t * 4u; i < words; i += WS_BLOCK * 4u) *reinterpret_cast<uint4*>(&count[i]) = make_uint4(0u, 0u, 0u, 0u);
        if (TOUCHED) {
            for (uint32_t w = t; w < nW; w += WS_BLOCK) touched[w] = 0u;
            for (uint32_t r = t; r < cap; r += WS_BLOCK) {
                cnt[r] = 0u;
                pos[r] = 0xffffu;
            }
        }
    }
    WSC_MARK(0);
    __syncthreads();  // the tables are clear

    // ------------------------------------------------------------------ every token's bin: the row's first rounds, while the ids are on their way
    const uint16_t last_ = static_cast<uint16_t>(kCodeFold - 1u - lane);
    const CodePair last = {last_, last_};  // (the tail: a bin of its own for each lane)
    typedef __attribute__((address_space(3))) uint32_t* LdsWord;
    const uint32_t my_count = static_cast<uint32_t>((uintptr_t)(LdsWord)(count + (two && (t & 1u) ? kCodeBins : 0u)));
    auto count_vector = [&](const uint4& v) __attribute__((always_inline)) {
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t at = __builtin_bit_cast(uint32_t, static_cast<CodePair>(code_pair(w4[k], last) << CodePair{2, 2}));
            uint32_t lo, hi;  // (each half to an address in one instruction)
            asm("v_add_u32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(lo) : "v"(my_count), "v"(at));
            asm("v_add_u32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(hi) : "v"(my_count), "v"(at));
            __hip_atomic_fetch_add((LdsWord)(uintptr_t)lo, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add((LdsWord)(uintptr_t)hi, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    // the row's last vector, where it ends inside one, and the lanes past it
    auto trim = [&](uint4& v, const uint32_t j) __attribute__((always_inline)) {
        if (j + 1u == nv && drop) v = part_vector<1>(v, drop);
        if (j >= nv) v = make_uint4(0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu);
    };
    auto mask_out = [&](uint4& v, const uint32_t allowed) __attribute__((always_inline)) {  // allowed: a bit for each of the eight
        const CodePair k2 = __builtin_bit_cast(CodePair, (~allowed & 0xffu) * 0x00010001u);
        auto nan_at = [&](uint32_t& w, uint16_t lo) {  // a token's bit to bit 15 of its half, then all over the half
            const CodePair up = k2 << CodePair{static_cast<uint16_t>(15u - lo), static_cast<uint16_t>(14u - lo)};
            w |= __builtin_bit_cast(uint32_t, __builtin_bit_cast(CodePairS, up) >> CodePairS{15, 15});
        };
        nan_at(v.x, 0);
        nan_at(v.y, 2);
        nan_at(v.z, 4);
        nan_at(v.w, 6);
    };
    auto held_allow = [&](int c) -> uint32_t {
        const uint32_t w = __shfl(aw[MASKED ? c >> 2 : 0], static_cast<int>((static_cast<uint32_t>(c & 3) << 4) + (lane >> 2)));
        return w >> ((lane & 3u) * 8u);
    };
    auto as_held = [&](uint4& v, uint32_t j) __attribute__((always_inline)) {  // what count_round makes of a held vector
        trim(v, j);
        if (MASKED) mask_out(v, allow[min(j >> 2, nW - 1u)] >> ((j * 8u) & 31u));
    };
    auto load_again = [&](uint32_t j) {
        uint4 v = row_vector<1>(base, j, V);
        as_held(v, j);
        return v;
    };
    // the row's vectors behind the held ones, one asked for while another is looked at (with every one waited for, rows of 262144 tokens took 1 us more)
    auto behind_held = [&](auto&& what) __attribute__((always_inline)) {
        if (NV != kCodeHeldVecs || NV * WS_BLOCK >= nv) return;  // uniform
        uint4 next = row_vector<1>(base, NV * WS_BLOCK + t, V);
        for (uint32_t j0 = NV * WS_BLOCK; j0 < nv; j0 += WS_BLOCK) {  // uniform
            uint4 v = next;
            next = row_vector<1>(base, j0 + WS_BLOCK + t, V);  // (past the row: its end)
            as_held(v, j0 + t);
            what(v, j0);
        }
    };
    // the first bin of the row's head (S.head_bin): the anchor of the masses, see mass_of
    auto look_at_head = [&](const uint4& v) __attribute__((always_inline)) {
        const CodePair a = __builtin_elementwise_min(code_pair(v.x, last), code_pair(v.y, last)), b = __builtin_elementwise_min(code_pair(v.z, last), code_pair(v.w, last));
        const CodePair c = __builtin_elementwise_min(a, b);
        const uint32_t first = wave_min_u32_apart(min(static_cast<uint32_t>(c.x), static_cast<uint32_t>(c.y)));
        if (lane == 0u) atomicMin(&S.head_bin, first);
    };
    auto count_round = [&](const int c) __attribute__((always_inline)) {
        const uint32_t j0 = static_cast<uint32_t>(c) * WS_BLOCK;
        if (c + kAhead < NV) load(c + kAhead < NV ? c + kAhead : 0);  // (not behind the branch: the compiler would wait there for every load before it)
        if (c < NV - 5 || j0 < nv) {  // uniform
            if (c >= NV - 6 && j0 + WS_BLOCK >= nv) trim(q[c], j0 + t);  // uniform
            if (c < 2 && A.code_head == 2u) look_at_head(q[c]);
            if (MASKED) mask_out(q[c], held_allow(c));
            if (!TOUCHED && c == 0 && A.code_head == 1u) look_at_head(q[c]);
            count_vector(q[c]);
        }
    };
    // The touched tokens: bitmap of their ids, prefix per word (a token's rank among them), count, logit and first bias entry by rank. Four
    // steps with a barrier before each, between the row's rounds: the trips to memory of the ids and then of their logits pass meanwhile.
    auto logit_at = [&](int32_t id_) -> uint32_t {
        const uint32_t id = min(static_cast<uint32_t>(id_), V - 1u);
        const uint32_t h = reinterpret_cast<const uint16_t*>(base)[id];
        return !MASKED || ((allow[id >> 5] >> (id & 31u)) & 1u) ? h : 0xff80u;  // (masked out: -inf)
    };
    auto rank = [&](uint32_t id) { return static_cast<uint32_t>(wprefix[id >> 5]) + static_cast<uint32_t>(__popc(touched[id >> 5] & ((1u << (id & 31u)) - 1u))); };
    constexpr uint32_t kWords = (NV * 8u * WS_BLOCK / 32u + WS_BLOCK - 1u) / WS_BLOCK;  // words of the bitmap a thread, of a row the registers hold
    const uint32_t per_ = NV < kCodeHeldVecs ? kWords : max(kWords, (nW + WS_BLOCK - 1u) / WS_BLOCK), w0_ = t * per_, w1_ = min(w0_ + per_, nW);
    uint32_t before_ = 0;  // touched tokens of the wave up to and with this thread's words
    auto touch = [&](const int step) __attribute__((always_inline)) {
        if (!TOUCHED || (nh + nb == 0u && A.code_head != 1u)) return;  // uniform
        if (step == 0) {
            auto mark = [&](int32_t id) {
                if (static_cast<uint32_t>(id) < V) atomicOr(&touched[static_cast<uint32_t>(id) >> 5], 1u << (id & 31));
            };
#pragma unroll
            for (int k = 0; k < kIds; ++k)
                if (static_cast<uint32_t>(k) * WS_BLOCK < nh) {
                    mark(hid[k]);
                    hraw[k] = logit_at(hid[k]);
                }
            for (uint32_t j = t + kIds * WS_BLOCK; j < nh; j += WS_BLOCK) mark(hist_ids[j]);
            if (nb) {
                mark(bid);
                braw = logit_at(bid);
            }
            for (uint32_t j = t + WS_BLOCK; j < nb; j += WS_BLOCK) mark(bias_ids[j]);
        } else if (step == 1) {
            __syncthreads();
            if (A.code_head == 1u) {  // uniform: the head without its touched tokens
                uint4 v = q[0];
                mask_out(v, ~(touched[min(t >> 2, nW - 1u)] >> ((t & 3u) * 8u)));
                look_at_head(v);
            }
            uint32_t local = 0, wd[kWords];
#pragma unroll
            for (uint32_t k = 0; k < kWords; ++k) wd[k] = touched[min(w0_ + k, nW - 1u)];
#pragma unroll
            for (uint32_t k = 0; k < kWords; ++k) local += w0_ + k < nW ? static_cast<uint32_t>(__popc(wd[k])) : 0u;
            for (uint32_t w = w0_ + kWords; w < w1_; ++w) local += static_cast<uint32_t>(__popc(touched[w]));
            before_ = wave_incl_scan(local);
            if (lane == 63u) S.red_u[wv] = before_;
            before_ -= local;
        } else if (step == 2) {
            __syncthreads();
            const uint32_t all = row_incl_scan(S.red_u[lane & (WS_WAVES - 1u)]);
            uint32_t run = (wv ? lane_value(all, wv - 1u) : 0u) + before_;
            n_touched = lane_value(all, WS_WAVES - 1u);
            uint32_t wd[kWords];
#pragma unroll
            for (uint32_t k = 0; k < kWords; ++k) wd[k] = touched[min(w0_ + k, nW - 1u)];
#pragma unroll
            for (uint32_t k = 0; k < kWords; ++k) {
                if (w0_ + k < nW) wprefix[w0_ + k] = static_cast<uint16_t>(run);
                run += static_cast<uint32_t>(__popc(wd[k]));
            }
            for (uint32_t w = w0_ + kWords; w < w1_; ++w) {
                wprefix[w] = static_cast<uint16_t>(run);
                run += static_cast<uint32_t>(__popc(touched[w]));
            }
        } else {
            __syncthreads();
            auto heard = [&](int32_t id_, uint32_t h) {
                const uint32_t id = static_cast<uint32_t>(id_);
                if (id < V) {
                    const uint32_t r = rank(id);
                    atomicAdd(&cnt[r], 1u);
                    tid[r] = id;
                    raw[r] = static_cast<uint16_t>(h);
                }
            };
#pragma unroll
            for (int k = 0; k < kIds; ++k)
                if (static_cast<uint32_t>(k) * WS_BLOCK < nh) heard(hid[k], hraw[k]);
            for (uint32_t j0 = kIds * WS_BLOCK; j0 < nh; j0 += 4u * WS_BLOCK) {  // uniform: four at a time, asked for together
                int32_t id[4];
                uint32_t h[4];
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) id[k] = j0 + k * WS_BLOCK + t < nh ? hist_ids[j0 + k * WS_BLOCK + t] : -1;
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) h[k] = logit_at(id[k]);
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) heard(id[k], h[k]);
            }
            for (uint32_t j = t; j < nb; j += WS_BLOCK) {
                const int32_t id_ = j == t ? bid : bias_ids[j];
                const uint32_t id = static_cast<uint32_t>(id_);
                if (id < V) {
                    const uint32_t r = rank(id);
                    atomicAdd(&cnt[r], 1u << 20);
                    tid[r] = id;
                    raw[r] = static_cast<uint16_t>(j == t ? braw : logit_at(id_));
                    // (the smallest entry number of the id: 16-bit words have no atomic minimum, so a pair of them goes by compare and swap)
                    uint32_t* word = reinterpret_cast<uint32_t*>(pos) + (r >> 1);
                    const uint32_t sh = (r & 1u) * 16u;
                    for (uint32_t seen = *word; ((seen >> sh) & 0xffffu) > j;) {
                        const uint32_t was = atomicCAS(word, seen, (seen & ~(0xffffu << sh)) | (j << sh));
                        if (was == seen) break;
                        seen = was;
                    }
                }
            }
        }
    };
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        count_round(c);
        constexpr int kStep = (NV + 4) / 5;
        if ((c + 1) % kStep == 0 && (c + 1) / kStep <= 4) touch((c + 1) / kStep - 1);
    }
    WSC_MARK(2);
    behind_held([&](const uint4& v, uint32_t) { count_vector(v); });
    __syncthreads();

    WSC_MARK(3);
    // ------------------------------------------------------------------ the touched tokens' adjusted logits, by group
    // A token's mass, e^(x - m). In a batch that the single-sweep kernels would take (code_head != 0) it is theirs to the last bit but a few:
    // a bin of 1/64 below an anchor above the row's head, and a quadratic inside the bin (bin_coord, bin_word) - good to 5e-7, and a row is
    // cut at the same token whichever kernel its batch gets. In the other batches it is the host sampler's own formula in 64 bits.
    const bool by_bins = A.code_head != 0u;
    const float c64 = inv_t * 64.f;
    const float anchor0 = code_value(min(S.head_bin, kCodeTail)) + A.code_above / inv_t;
    const float aq0 = anchor_product(anchor0, c64);
    auto inside = [&](float tc) { return static_cast<double>(0x40000000u - static_cast<uint32_t>(bin_word(tc))); };  // of a bin's mass at its upper end, in units of 2^-30
    const double kFix = static_cast<double>(1ull << kCodeFixBits), kUnfix = 1.0 / kFix;
    // A touched token's mass in fixed point against that of `top`, and (unfix_of) the other way round. `top` is that of the token's group; in a wide
    // one no more than the largest touched token: an octave's eighth is 0.5 from 8 to 16 and 2 from 32 to 64, 10 to 40 e-folds at a temperature of 0.05, and
    // against a top so far above it the largest token of the row would weigh nothing. (Each is off by 2^-45 e^4 of the normaliser at most.)
    // The largest is known behind a barrier, so those of wide groups wait for a loop of their own - and in the kernel whose vectors leave no registers for
    // this code beside the bias search all of them (256 rows, 2048 ids, us, those of narrow groups at once and all of them later: of 50257 26.6 / 27.4, of 151936
    // 41.7 with 63 registers spilled / 40.9).
    // (The row's 64-bit values are kept in scalar registers there for the same reason; in the others, where vector registers are left, that only
    // lengthens the chain: 250 rows with 500 ids, us, scalar / vector: of 80000 24.8 / 24.0, of 41000 21.3 / 21.0.)
    auto row_value = [](double v) __attribute__((always_inline)) { return NV == kCodeHeldVecs ? lane_value(v, 0u) : v; };
    const double inv_t_d = row_value(static_cast<double>(inv_t));
    auto group_waits = [&](uint32_t g) { return NV == kCodeHeldVecs || code_group_step(g) * inv_t > kCodeWide / 8.f; };
    auto group_by_bins = [&](uint32_t g, double top) {  // (none of them above the anchor, or in the tail)
        return by_bins && top <= static_cast<double>(anchor0) && bin_coord(aq0, c64, code_value(g * 8u + 7u)) < 4000.f;
    };
    auto top_bin_of = [&](double top) { return static_cast<uint32_t>(bin_coord(aq0, c64, static_cast<float>(top))); };
    auto fix_of = [&](float x, uint32_t g, double top) {
        double e;
        if (group_by_bins(g, top)) {
            const float tc = bin_coord(aq0, c64, x);
            const uint32_t d = static_cast<uint32_t>(tc) - top_bin_of(top);
            e = S.s_exp[d >> 6] * S.s_exp[64u + (d & 63u)] * (inside(tc) * kFixInv);
        } else {
            e = code_exp((top - static_cast<double>(x)) * inv_t_d);
        }
        return static_cast<unsigned long long>(e * kFix + 0.5);
    };
    if (TOUCHED) {
        uint32_t best = 0u;
        for (uint32_t r = t; r < n_touched; r += WS_BLOCK) {
            const uint32_t cw = cnt[r], c = cw & 0xfffffu, n_bias = (cw >> 20) & 0x7ffu;
            float x = fmaxf(bf16_to_f32(raw[r]), -INFINITY);
            const uint32_t was = code_bin(x);  // (out of the raw logits' counts)
            if (was < kCodeTail) atomicSub(&count[was], 1u);
            if (__ballot(n_bias != 0u)) {  // uniform
                const uint32_t j = n_bias ? pos[r] : 0u;
                if (n_bias) x = __fadd_rn(x, bias_vals[j]);
                if (__ballot(n_bias > 1u)) x = add_other_bias(n_bias > 1u, tid[r], j, x, bias_ids, bias_vals, nb);
            }
            if (c) {
                x = x > 0.f ? __fdiv_rn(x, P.rep) : __fmul_rn(x, P.rep);
                x = __fsub_rn(x, __fadd_rn(__fmul_rn(P.freq, static_cast<float>(c)), P.pres));
            }
            adj[r] = x;
            const uint32_t bin = x == x ? code_bin(x) : 0u;  // (NaN out of the penalties: the three-pass code's)
            if (bin < 8u) S.bad = 1u;
            if (bin < kCodeTail && bin >= 8u) {
                const uint32_t g = bin >> 3;
                best = max(best, key32(x));
                if (group_waits(g)) S.waiting = 1u;
                else atomicAdd(&g_mass[g], fix_of(x, g, code_group_top(g)));
                pos[r] = static_cast<uint16_t>(atomicAdd(&g_cnt[g], 1u));
            }
        }
        best = ~wave_min_u32_apart(~best);
        if (lane == 0u && best) atomicMax(&S.top_key, best);
    }
    if (TOUCHED) __syncthreads();
    WSC_MARK(4);
    const double touched_max = TOUCHED && S.top_key ? static_cast<double>(unkey32(S.top_key)) : -INFINITY;
    auto top_of = [&](uint32_t g) { return group_waits(g) ? fmin(code_group_top(g), touched_max) : code_group_top(g); };
    if (TOUCHED && S.waiting)  // uniform
        for (uint32_t r = t; r < n_touched; r += WS_BLOCK) {
            const float x = adj[r];
            const uint32_t bin = code_bin(x), g = bin >> 3;
            if (bin < kCodeTail && bin >= 8u && group_waits(g)) atomicAdd(&g_mass[g], fix_of(x, g, top_of(g)));
        }
    // ------------------------------------------------------------------ this thread's eight bins, and the prefix sums over the groups: tokens,
    // mass, touched tokens
    uint32_t c8[8], own = 0, first = kCodeBins;
    {
        const uint4 a = *reinterpret_cast<const uint4*>(&count[t * 8u]), b = *reinterpret_cast<const uint4*>(&count[t * 8u + 4u]);
        c8[0] = a.x, c8[1] = a.y, c8[2] = a.z, c8[3] = a.w, c8[4] = b.x, c8[5] = b.y, c8[6] = b.z, c8[7] = b.w;
        if (two) {
            const uint4 e = *reinterpret_cast<const uint4*>(&count[kCodeBins + t * 8u]), f = *reinterpret_cast<const uint4*>(&count[kCodeBins + t * 8u + 4u]);
            c8[0] += e.x, c8[1] += e.y, c8[2] += e.z, c8[3] += e.w, c8[4] += f.x, c8[5] += f.y, c8[6] += f.z, c8[7] += f.w;
            *reinterpret_cast<uint4*>(&count[t * 8u]) = make_uint4(c8[0], c8[1], c8[2], c8[3]);
            *reinterpret_cast<uint4*>(&count[t * 8u + 4u]) = make_uint4(c8[4], c8[5], c8[6], c8[7]);
        }
        if (t >= kCodeTail / 8u)
#pragma unroll
            for (int k = 0; k < 8; ++k) c8[k] = 0u;
#pragma unroll
        for (int k = 7; k >= 0; --k) {
            own += c8[k];
            first = c8[k] ? t * 8u + static_cast<uint32_t>(k) : first;
        }
    }
    const uint32_t ext = TOUCHED ? g_cnt[t] : 0u;
    const bool wave_has = __ballot(own + ext != 0u) != 0ull;
    first = wave_has ? wave_min_u32_apart(first) : kCodeBins;
    if (lane == 0u && first < kCodeBins) atomicMin(&S.top_bin, first);
    __syncthreads();
    const float m = fmaxf(S.top_bin < kCodeTail ? code_value(S.top_bin) : -INFINITY, S.top_key ? unkey32(S.top_key) : -INFINITY);
    // (a touched token that is not for this kernel, a token above the bins, or none in them)
    WSC_MARK(5);
    if (S.bad || S.top_bin < 8u || !(m > -INFINITY)) return false;
    // The last bins are not looked at. Where they do not lie 50 e-folds below the maximum, or not below the min-p floor, nothing but masked-out tokens
    // may be in them: those are counted, and the row is handed back further down if there are others.
    const bool tail_matters = !(__fsub_rn(m, code_value(kCodeTail)) * inv_t >= 50.f) ||
                              (use_min_p && code_bin(static_cast<float>(static_cast<double>(m) - S.floor_below)) >= kCodeTail);  // uniform
    if (MASKED && tail_matters) {
        uint32_t out = 0;
        for (uint32_t w = t; w < nW; w += WS_BLOCK) out += static_cast<uint32_t>(__popc(~allow[w] & (w + 1u < nW ? 0xffffffffu : 0xffffffffu >> (nW * 32u - V))));
        out = wave_sum(out);
        if (lane == 0u) atomicAdd(&S.n_out, out);
    }
    // (an anchor that lies below the maximum, or wastefully far above it, gives way to the maximum itself)
    const float aq = m <= anchor0 && (anchor0 - m) * c64 <= 1024.f ? aq0 : anchor_product(m, c64);
    const double m_d = row_value(static_cast<double>(m));
    const double lift = row_value(static_cast<double>(aq) * (1.0 / 64.0) - m_d * inv_t_d);
    auto exact_mass = [&](float x) { return code_exp(static_cast<double>(__fsub_rn(m, x)) * inv_t_d); };
    auto mass_of = [&](float x) {
        if (!by_bins) return exact_mass(x);  // uniform
        const float tc = bin_coord(aq, c64, x);
        return code_exp(static_cast<double>(static_cast<uint32_t>(tc)) * (1.0 / 64.0) - lift) * (inside(tc) * kFixInv);
    };
    auto unfix_of = [&](unsigned long long sum, uint32_t g) {
        const double top = top_of(g);
        const double down = group_by_bins(g, top) ? (static_cast<double>(top_bin_of(top)) - static_cast<double>(aq0)) * (1.0 / 64.0) + m_d * inv_t_d : (m_d - top) * inv_t_d;
        return static_cast<double>(sum) * kUnfix * code_exp(down);
    };
    double Z;
    uint32_t n_all;
    {
        double mass = 0.0;
        if (own) {
            if (by_bins) {  // uniform: every value's bin is its own
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float tc = bin_coord(aq, c64, code_value(t * 8u + static_cast<uint32_t>(k)), 4031.f);
                    const uint32_t b = static_cast<uint32_t>(tc);
                    mass = fma(static_cast<double>(c8[k]), S.s_exp[b >> 6] * S.s_exp[64u + (b & 63u)] * inside(tc), mass);
                }
                mass *= kFixInv * code_exp(-lift);
            } else {  // equal steps: eight masses from the first one's and the factor of a step
                // (the first that holds a token: a group may reach above the maximum, where masses have no bound)
                const double f = code_exp(static_cast<double>(code_group_step(t)) * inv_t_d);
                uint32_t k0 = 7u;
                mass = static_cast<double>(c8[7]);
#pragma unroll
                for (int k = 6; k >= 0; --k) k0 = c8[k] ? static_cast<uint32_t>(k) : k0;
#pragma unroll
                for (int k = 6; k >= 0; --k) mass = static_cast<uint32_t>(k) >= k0 ? fma(mass, f, static_cast<double>(c8[k])) : mass;
                mass *= exact_mass(code_value(t * 8u + k0));
            }
        }
        if (TOUCHED && ext) mass += unfix_of(g_mass[t], t);
        const uint32_t n = own + ext;
        uint32_t ni = 0u, ei = 0u;
        double mi = 0.0, up = 0.0;
        if (wave_has) {  // uniform
            ni = wave_incl_scan(n);
            if (TOUCHED) ei = wave_incl_scan(ext);
            mi = wave_incl_scan(mass);
            up = __shfl_up(mi, 1);
        }
        if (lane == 63u) {
            S.red_d[wv] = mi;
            S.red_u[wv] = ni;
            S.red_v[wv] = ei;
        }
        __syncthreads();
        const double wm = row_incl_scan(S.red_d[lane & (WS_WAVES - 1u)]);
        const uint32_t wn = row_incl_scan(S.red_u[lane & (WS_WAVES - 1u)]), we = TOUCHED ? row_incl_scan(S.red_v[lane & (WS_WAVES - 1u)]) : 0u;
        Z = lane_value(wm, WS_WAVES - 1u);
        n_all = lane_value(wn, WS_WAVES - 1u);
        if (tail_matters && n_all + S.n_out < V) return false;  // uniform
        if (!(Z > 0.5 && Z < INFINITY)) return false;  // uniform (the maximum's own mass is 1: it has not been counted as it should)
        if (wave_has) {  // uniform
            const double base_m = wv ? lane_value(wm, wv - 1u) : 0.0;
            const uint32_t base_n = wv ? lane_value(wn, wv - 1u) : 0u;
            const double pre = base_m + (lane ? up : 0.0), end = lane == 63u ? lane_value(wm, wv) : base_m + mi;  // (where the next group begins, bit for bit)
            const uint32_t cend = base_n + ni, cpre = cend - n;
            if (TOUCHED) g_list[t] = ((wv ? lane_value(we, wv - 1u) : 0u) + ei - ext) | (ext << 16);
            g_pre[t] = pre;
            g_cpre[t] = cpre;
            // the groups the searches below begin with
            if (P.top_k != 0u) {
                if (cpre < P.top_k && cend >= P.top_k) S.g_first[0] = t;
            } else if (use_top_p) {
                const double Xf = top_p * static_cast<double>(static_cast<float>(Z)), Xz = top_p * Z, at = S.u * Xf;
                if (pre < Xf && end >= Xf) S.g_first[0] = t;
                if (pre < Xz && end >= Xz) S.g_first[1] = t;
                if (pre <= at && end > at) S.g_draw = t;
            }
        } else {
            g_pre[t] = lane_value(wm, wv);
            g_cpre[t] = lane_value(wn, wv);
            g_list[t] = 0u;
        }
        if (wv == 0u && lane < WS_WAVES) {
            S.wave_mass[lane] = wm;
            S.wave_cnt[lane] = wn;
        }
    }
    __syncthreads();
    if (TOUCHED && n_touched) {
        uint16_t* order = raw;
        for (uint32_t r = t; r < n_touched; r += WS_BLOCK) {
            const uint32_t bin = code_bin(adj[r]);
            if (bin < kCodeTail) order[(g_list[bin >> 3] & 0xffffu) + pos[r]] = static_cast<uint16_t>(r);
        }
        __syncthreads();
    }
    constexpr uint32_t kSolver = WS_WAVES - 1u;  // the wave that looks for the cuts: its vectors wait in LDS - they and that code together would not fit the registers
    uint4* stash = reinterpret_cast<uint4*>(lds + L.stash) + lane;
    if (wv == kSolver && two) {
#pragma unroll
        for (int c = 0; c < NV; ++c)
            if (c < NV - 5 || static_cast<uint32_t>(c) * WS_BLOCK < nv) stash[c * 64] = q[c];  // uniform
    }

    // ------------------------------------------------------------------ one wave: the cuts and the draw, one after the other
    // (the arguments again, through a pointer the compiler cannot see through: none of them sits in a register across the sweep)
    LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    if (wv == kSolver) {
        WSC_MARK2(10);
        const uint16_t* order = raw;
        uint32_t n = V;  // kept so far, and their mass
        double M = Z, gap_top_p = 1.0, of_top_p = 1.0, mg_min_p = 1.0, gap_draw = 0.0;
        bool ok = true, fell = false;
        // the group that holds a token's place, or the token at which the running mass reaches X (passes X): a wave's 64 groups, then the one
        // of them; kCodeGroups where rounding puts it past the last one
        auto find = [&](auto mode_, uint32_t K, double X) __attribute__((always_inline)) {
            constexpr CodeLook mode = decltype(mode_)::value;
            const double ws = S.wave_mass[lane & (WS_WAVES - 1u)];
            const uint32_t wc = S.wave_cnt[lane & (WS_WAVES - 1u)];
            const uint64_t any = __ballot(lane < WS_WAVES && (mode == kByRank ? wc >= K : (mode == kByMass ? ws >= X : ws > X)));
            if (any == 0ull) return kCodeGroups;
            const uint32_t w = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1);
            const uint32_t next = min(w * 64u + lane + 1u, kCodeGroups - 1u);  // (where the lane's group ends the next begins)
            bool is;
            if (mode == kByRank) {
                const uint32_t c = g_cpre[next];
                is = (lane == 63u ? lane_value(wc, w) : c) >= K;
            } else {
                const double s_ = g_pre[next], s = lane == 63u ? lane_value(ws, w) : s_;
                is = mode == kByMass ? s >= X : s > X;
            }
            return w * 64u + static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(__ballot(is))) - 1);
        };
        // the token in group g (kByPassing: in bin k_of of it, where the floor lies; rank: how many pass)
        auto look = [&](auto mode_, uint32_t g, uint32_t K, double X, uint32_t k_of) __attribute__((always_inline)) {
            constexpr CodeLook mode = decltype(mode_)::value;
            CodeAt R;
            R.ok = false;
            if (g >= kCodeGroups) return R;
            const uint32_t listed = TOUCHED ? g_list[g] : 0u, list = listed & 0xffffu, n_ext = listed >> 16;
            const uint32_t b_ = g * 8u + (lane & 7u);  // lane k < 8 has the group's k-th bin
            uint32_t c = count[b_], e = 0;
            const double pre = g_pre[g];
            const uint32_t cpre = g_cpre[g];
            if (n_ext) {  // uniform
                if (lane < 8u) {
                    S.bin_cnt[lane] = 0u;
                    S.bin_mass[lane] = 0ull;
                }
                lanes_meet();
                for (uint32_t i = lane; i < n_ext; i += 64u) {
                    const float x = adj[order[list + i]];
                    const uint32_t k = code_bin(x) & 7u;
                    atomicAdd(&S.bin_cnt[k], 1u);
                    atomicAdd(&S.bin_mass[k], fix_of(x, g, top_of(g)));
                }
                lanes_meet();
                if (lane < 8u) e = S.bin_cnt[lane];
            }
            const double w = mass_of(code_value(b_));
            double mass = c ? static_cast<double>(c) * w : 0.0;  // (an empty bin may lie above the maximum: no bound to its w)
            if (e) mass += unfix_of(S.bin_mass[lane], g);
            if (lane >= 8u) c = 0u, mass = 0.0;
            const uint32_t ci = wave_incl_scan(c + e) + cpre;
            const double mi = wave_incl_scan(mass) + pre;
            uint32_t k = k_of;
            if (mode != kByPassing) {
                const bool here = c + e != 0u && (mode == kByRank || mass > 0.0);
                const uint64_t any = __ballot(here && (mode == kByRank ? ci >= K : (mode == kByMass ? mi >= X : mi > X))), some = __ballot(here);
                if (some == 0ull) return R;
                k = any ? static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1)
                        : 63u - static_cast<uint32_t>(__clzll(static_cast<long long>(some)));  // (rounding: the group's last bin)
            }
            const uint32_t bin = g * 8u + k, c_tied = lane_value(c, k), n_bin = lane_value(e, k);
            const double w_tied = lane_value(w, k);
            uint32_t rank = lane_value(ci, k) - c_tied - n_bin;            // of the bin's first token
            double run = k ? lane_value(mi, k - 1u) : pre;                 // mass ranked before it
            if (bin == kCodeFold || n_bin > kCodeSub) return R;            // (around zero values differ inside a bin)
            const float v = code_value(bin);
            uint32_t n_eq = 0, n_above = 0;  // touched tokens at the bin's value, and above it: these come first
            bool hit = false;
            R.near = 1.0;
            R.first = rank;
            R.token = 0xffffffffu;
            R.place = 0u;
            if (n_bin) {  // uniform: the bin's touched tokens in order
                uint32_t put = 0;
                for (uint32_t i0 = 0; i0 < n_ext; i0 += 64u) {
                    uint64_t key = 0ull;
                    if (i0 + lane < n_ext) {
                        const uint32_t r = order[list + i0 + lane];
                        const float x = adj[r];
                        if (code_bin(x) == bin) key = key64(x, tid[r]);
                    }
                    const uint64_t mk = __ballot(key != 0ull);
                    if (key) S.sub[put + static_cast<uint32_t>(__popcll(mk & ((1ull << lane) - 1ull)))] = key;
                    put += static_cast<uint32_t>(__popcll(mk));
                }
                lanes_meet();
                for (uint32_t i = 0; i < n_bin; i += 64u) {
                    const uint64_t key = i + lane < n_bin ? S.sub[i + lane] : 0ull;
                    uint32_t above = 0;
                    for (uint32_t j0 = 0; j0 < n_bin; j0 += 64u) {
                        const uint64_t other = j0 == i ? key : (j0 + lane < n_bin ? S.sub[j0 + lane] : 0ull);
                        for (uint32_t j = 0; j < min(64u, n_bin - j0); ++j) above += lane_value(other, j) > key ? 1u : 0u;
                    }
                    if (key) S.sorted[above] = key;
                    n_eq += key && static_cast<uint32_t>(key >> 32) == key32(v) ? 1u : 0u;
                }
                n_eq = wave_sum(n_eq);
                lanes_meet();
                n_above = n_bin - n_eq;
                for (uint32_t i0 = 0; i0 < n_above && !hit; i0 += 64u) {
                    const bool on = i0 + lane < n_above;
                    const uint64_t key = on ? S.sorted[i0 + lane] : 0ull;
                    const double wl = on ? mass_of(unkey32(static_cast<uint32_t>(key >> 32))) : 0.0;
                    const double cum = run + wave_incl_scan(wl);
                    const double own_ = mode == kByPassing && on ? exact_mass(unkey32(static_cast<uint32_t>(key >> 32))) : 0.0;
                    const bool is = on && (mode == kByRank ? rank + lane + 1u >= K : (mode == kByMass ? cum >= X : (mode == kPast ? cum > X : own_ < X)));
                    if (mode == kByPassing && on) R.near = fmin(R.near, fabs(own_ - X) / X);
                    uint64_t any = __ballot(is);
                    const uint32_t here = min(64u, n_above - i0);
                    if (any == 0ull && mode != kByPassing && i0 + here == n_above && c_tied + n_eq == 0u) any = 1ull << (here - 1u);  // (rounding: the bin's last)
                    if (any) {
                        const uint32_t f = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1);
                        hit = true;
                        rank += f;
                        R.unit = lane_value(wl, f);
                        R.logit = unkey32(static_cast<uint32_t>(lane_value(key, f) >> 32));
                        R.cin = lane_value(cum, f);
                        R.cex = f ? lane_value(cum, f - 1u) : run;
                        R.token = 0xffffffffu - static_cast<uint32_t>(lane_value(key, f));
                    } else {
                        rank += here;
                        run = lane_value(cum, here - 1u);
                    }
                }
            }
            if (!hit) {
                const uint32_t tied = c_tied + n_eq;
                R.unit = w_tied;
                R.logit = v;
                if (mode == kByPassing) {
                    const double own_ = exact_mass(v);
                    R.place = own_ >= X ? tied : 0u;
                    if (tied) R.near = fmin(R.near, fabs(own_ - X) / X);
                } else if (mode == kByRank) {
                    R.place = K - 1u - rank;
                } else if (tied > 1u) {
                    double inv = __builtin_amdgcn_rcp(w_tied);
                    inv = fma(fma(-w_tied, inv, 1.0), inv, inv);
                    const double want = (X - run) * inv;
                    uint32_t p = want > 0.0 ? (want < static_cast<double>(tied) ? static_cast<uint32_t>(want) : tied - 1u) : 0u;
                    auto there = [&](uint32_t p_) {
                        const double s = run + static_cast<double>(p_ + 1u) * w_tied;
                        return mode == kByMass ? s >= X : s > X;
                    };
                    while (p > 0u && there(p - 1u)) --p;
                    while (p + 1u < tied && !there(p)) ++p;
                    R.place = p;
                }
                rank += R.place;
                R.cex = run + static_cast<double>(R.place) * w_tied;
                R.cin = R.cex + w_tied;
            }
            R.rank = rank;
            R.bin = bin;
            R.n_eq = n_eq;
            R.n_above = n_above;
            R.ok = true;
            return R;
        };
        typedef std::integral_constant<CodeLook, kByRank> ByRank;
        typedef std::integral_constant<CodeLook, kByMass> ByMass;
        typedef std::integral_constant<CodeLook, kByPassing> ByPassing;
        typedef std::integral_constant<CodeLook, kPast> Past;
        if (open) {
            // the engine's short list, its 256 largest, by shares of the whole row; behind them the others in id order (src/sampling/sampler.cpp:118-146)
            const uint32_t K = min(kOpenList, V);
            n = K;
            M = static_cast<double>(static_cast<float>(Z));
            const double X = S.u * M;
            CodeAt at;
            double listed = Z;
            at.ok = true;
            if (n_all > K) {
                at = look(ByRank{}, find(ByRank{}, K, 0.0), K, 0.0, 0u);
                listed = at.cin;
            }
            const bool walk = at.ok && !(X < listed);
            if (at.ok && !walk) {
                at = look(Past{}, find(Past{}, 0u, X), 0u, X, 0u);
                at.ok = at.ok && at.rank < K;
                gap_draw = fmin(at.cin - X, at.rank > 0u ? X - at.cex : 1e300);
            }
            if (lane == 0u && at.ok && (!walk || n_all > K)) {
                S.state = (at.token != 0xffffffffu ? 1u : 2u) + (walk ? 2u : 0u);
                S.token = at.token;
                S.value2 = (__float_as_uint(code_value(at.bin)) >> 16) * 0x00010001u;
                S.place = at.place;
                S.n_eq = at.n_eq;
                S.eq_at = at.n_above;
                S.n_kept = n;
                S.unit = by_bins ? exact_mass(at.logit) : at.unit;
                S.kept_mass = M;
                S.gap_top_p = S.of_top_p = S.near_min_p = 1.0;
                S.gap_draw = gap_draw;
                S.walk_below = at.logit;
                S.walk = X - listed;
            }
            ok = false;  // (nothing else to do)
        }
        if (!open && P.top_k != 0u && P.top_k < V) {
            n = P.top_k;
            if (n < n_all) {  // (else the row's last tokens carry no mass)
                const CodeAt at = look(ByRank{}, S.g_first[0], n, 0.0, 0u);
                ok = at.ok;
                M = at.cin;
            }
        }
        if (ok && use_top_p) {
            // (the float normaliser - Sampler::sum, src/sampling/sampler.h:38 - while the cut is among the first 16384 tokens, as the reference's
            // lists have it)
            const double Xf = top_p * static_cast<double>(static_cast<float>(Z)), Xz = top_p * Z;
            bool exact_z = P.top_k == 0u && Xf > Z;
            uint32_t g;
            if (P.top_k != 0u) {
                g = find(ByMass{}, 0u, top_p * M);
            } else {
                g = S.g_first[exact_z ? 1 : 0];
                if (!exact_z && g < kCodeGroups && g_cpre[g] >= 16384u) {
                    exact_z = true;
                    g = S.g_first[1];
                }
            }
            for (;;) {
                const double X = P.top_k != 0u ? top_p * M : (exact_z ? Xz : Xf);
                const CodeAt at = look(ByMass{}, g, 0u, X, 0u);
                ok = at.ok;
                if (ok && P.top_k == 0u && !exact_z && at.first >= 16384u) {
                    exact_z = true;
                    g = S.g_first[1];
                    continue;
                }
                gap_top_p = fmin(at.cin - X, at.rank > 0u ? X - at.cex : X);
                of_top_p = X;
                if (at.rank < n) {
                    n = at.rank + 1u;
                    M = at.cin;
                }
                break;
            }
        }
        if (ok && use_min_p) {
            const float fx = static_cast<float>(static_cast<double>(m) - S.floor_below);
            const uint32_t bin = code_bin(fx);
            if (bin < kCodeTail) {  // (else all passes that is not masked out)
                const CodeAt at = look(ByPassing{}, bin >> 3, 0u, min_p, bin & 7u);
                ok = at.ok;
                // (a floor within a rounding of the bin's ends may have a neighbour's token near it)
                const float eps = 1e-6f * fabsf(fx) + 1e-6f / inv_t;
                mg_min_p = code_bin(fx + eps) != bin || code_bin(fx - eps) != bin ? 0.0 : static_cast<double>(-wave_max(-static_cast<float>(at.near)));
                if (at.rank < n) {
                    n = max(at.rank, 1u);
                    M = at.rank ? at.cex : 1.0;
                }
            } else {
                n = min(n, n_all);
            }
        }
        if (ok) {
            const double X = S.u * M;
            const uint32_t guess = S.g_draw;
            uint32_t g = kCodeGroups;
            if (guess < kCodeGroups) {
                const double next = guess + 1u < kCodeGroups ? g_pre[guess + 1u] : Z;
                if (g_pre[guess] <= X && next > X) g = guess;
            }
            if (g == kCodeGroups) g = find(Past{}, 0u, X);
            CodeAt at = look(Past{}, g, 0u, X, 0u);
            fell = g == kCodeGroups || (at.ok && at.rank >= n);  // (rounding: past the kept tokens - the last of them)
            if (fell) {
                const uint32_t K = min(n, n_all);
                at = look(ByRank{}, find(ByRank{}, K, 0.0), K, 0.0, 0u);
            } else {
                gap_draw = fmin(at.cin - X, at.rank > 0u ? X - at.cex : 1e300);
            }
            if (lane == 0u && at.ok) {
                S.state = at.token != 0xffffffffu ? 1u : 2u;
                S.token = at.token;
                S.value2 = (__float_as_uint(code_value(at.bin)) >> 16) * 0x00010001u;
                S.place = at.place;
                S.n_eq = at.n_eq;
                S.eq_at = at.n_above;
                S.n_kept = n;
                S.unit = by_bins ? exact_mass(at.logit) : at.unit;
                S.kept_mass = M;
                S.gap_top_p = gap_top_p;
                S.of_top_p = of_top_p;
                S.near_min_p = mg_min_p;
                S.gap_draw = gap_draw;
            }
        }
        WSC_MARK2(14);
        lanes_meet();
        if (two) {  // uniform
#pragma unroll
            for (int c = 0; c < NV; ++c) {
                q[c] = make_uint4(0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu);
                if (c < NV - 5 || static_cast<uint32_t>(c) * WS_BLOCK < nv) q[c] = stash[c * 64];
            }
        } else {
#pragma unroll
            for (int c = 0; c < NV; ++c) {
                q[c] = load_again(static_cast<uint32_t>(c) * WS_BLOCK + t);
                __builtin_amdgcn_sched_barrier(0);  // (one after the other: all at once they need more registers than there are)
            }
        }
    }
    __syncthreads();
    WSC_MARK(7);
    if (S.state == 0u) return false;
    // (one lane writes the answers)
    auto write_answers = [&]() __attribute__((always_inline)) {
        const double M = S.kept_mass, tol = Ap->tol;
        uint32_t flags = Ap->code_route | (open ? kOpen : 0u);
        if (S.gap_top_p < tol * S.of_top_p) flags |= kNearTopP;
        if (S.near_min_p < tol) flags |= kNearMinP;
        if (S.gap_draw < tol * M) flags |= kNearDraw;
        Ap->flags[row] = flags;
        if (Ap->prob) Ap->prob[row] = static_cast<float>(S.unit / M);
        if (Ap->n_kept) Ap->n_kept[row] = S.n_kept;
        if (Ap->stats) {
            Ap->stats[2 * row] = m;
            Ap->stats[2 * row + 1] = static_cast<float>(Z);
        }
#ifndef WS_CODE_TIMERS
        if (Ap->margin) {
            Ap->margin[3 * row] = S.gap_top_p / S.of_top_p;
            Ap->margin[3 * row + 1] = S.near_min_p;
            Ap->margin[3 * row + 2] = S.gap_draw / M;
        }
#endif
    };
    const uint32_t state = S.state;
    if (state == 1u) {
        if (t == 0u) {
            Ap->token[row] = static_cast<int32_t>(S.token);
            write_answers();
        }
        return true;
    }

    // ------------------------------------------------------------------ the tied token at that place in id order: how many there are in
    // every 512 neighbouring tokens (a wave's round), the block the place falls in, then its vectors
    uint32_t* block = reinterpret_cast<uint32_t*>(lds + L.block);
    const uint32_t value2 = S.value2;
    // which of a vector's eight tokens have the value and are not touched (bit for bit); j: the vector's number
    auto tied = [&](const uint4& v, uint32_t j) __attribute__((always_inline)) {
        const uint32_t a = __builtin_bit_cast(uint32_t, code_one(v.x ^ value2)), b = __builtin_bit_cast(uint32_t, code_one(v.y ^ value2));
        const uint32_t c = __builtin_bit_cast(uint32_t, code_one(v.z ^ value2)), d = __builtin_bit_cast(uint32_t, code_one(v.w ^ value2));
        const uint32_t differ = a | (b << 2) | (c << 4) | (d << 6);  // even tokens in the lower half, odd ones in the upper
        uint32_t bits = ~(differ | (differ >> 15)) & 0xffu;
        if (TOUCHED && n_touched) bits &= ~reinterpret_cast<const uint8_t*>(touched)[min(j, nv - 1u)];
        return bits;
    };
    auto tally = [&](const uint4& v, uint32_t j0) __attribute__((always_inline)) {
        auto low = [](uint32_t x, uint32_t y) { return __builtin_elementwise_min(__builtin_bit_cast(CodePair, x), __builtin_bit_cast(CodePair, y)); };
        const uint32_t least = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(low(v.x ^ value2, v.y ^ value2), low(v.z ^ value2, v.w ^ value2)));
        if ((least & 0xffffu) == 0u || (least >> 16) == 0u) {
            // (the address by way of a vector register: for one the compiler knows to be the wave's it adds the lanes up first, at many times the cost)
            uint32_t at = (j0 >> 6) + wv;
            asm volatile("" : "+v"(at));
            atomicAdd(&block[at], static_cast<uint32_t>(__popc(tied(v, j0 + t))));
        }
    };
    const uint32_t n_blocks = (nv + 63u) / 64u, per = (n_blocks + 63u) / 64u;
    // the block in which the running count passes `left` (which goes down to what is left in the block); none: 0xffffffff. Every wave for itself: a
    // lane adds up its share of the blocks, then the share it falls in is looked at one by one
    auto find_block = [&](auto* counts, auto& left) __attribute__((always_inline)) {
        typedef std::remove_reference_t<decltype(left)> Count;
        Count n = 0;
        for (uint32_t i = 0; i < per; ++i) n += lane * per + i < n_blocks ? counts[lane * per + i] : 0u;
        Count inc = wave_incl_scan(n);
        uint64_t any = __ballot(inc > left);
        if (any == 0ull) return 0xffffffffu;
        uint32_t f = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1);
        left -= lane_value(inc, f) - lane_value(n, f);
        const uint32_t at = f * per;
        n = lane < per && at + lane < n_blocks ? counts[at + lane] : 0u;
        inc = wave_incl_scan(n);
        any = __ballot(inc > left);
        f = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(any)) - 1);
        left -= lane_value(inc, f) - lane_value(n, f);
        return at + f;
    };
    auto vector_of = [&](uint32_t round) __attribute__((always_inline)) {  // this thread's of a round (the same for the wave)
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int c = 0; c < NV; ++c)
            if (static_cast<uint32_t>(c) == round) v = q[c];  // uniform
        if (NV == kCodeHeldVecs && round >= static_cast<uint32_t>(NV)) v = load_again(round * WS_BLOCK + t);
        return v;
    };
    if (state != 3u) {  // uniform
#pragma unroll
        for (int c = 0; c < NV; ++c)
            if (c < NV - 5 || static_cast<uint32_t>(c) * WS_BLOCK < nv) {  // uniform
                tally(q[c], static_cast<uint32_t>(c) * WS_BLOCK);
            }
        behind_held(tally);
        if (wv == kSolver)
            for (uint32_t i = lane; i < S.n_eq; i += 64u) atomicAdd(&block[(0xffffffffu - static_cast<uint32_t>(S.sorted[S.eq_at + i])) >> 9], 1u);
        __syncthreads();
        WSC_MARK(8);
        uint32_t left = S.place;
        const uint32_t at = find_block(block, left);
        if (at == 0xffffffffu) return false;  // (the counts and the histogram disagree)
        const uint32_t owner = at % WS_WAVES, round = at / WS_WAVES;
        if (state == 2u && t == (owner == 0u ? 64u : 0u)) write_answers();
        if (wv == owner) {
            const uint4 v = vector_of(round);
            uint32_t bits = tied(v, round * WS_BLOCK + t);
            for (uint32_t i = 0; i < S.n_eq; ++i) {
                const uint32_t id = 0xffffffffu - static_cast<uint32_t>(S.sorted[S.eq_at + i]);
                if ((id >> 9) == at && ((id >> 3) & 63u) == lane) bits |= 1u << (id & 7u);
            }
            const uint32_t mine = static_cast<uint32_t>(__popc(bits)), before = wave_incl_scan(mine) - mine;
            if (left >= before && left < before + mine) {
                for (uint32_t i = before; i < left; ++i) bits &= bits - 1u;
                const uint32_t id = (round * WS_BLOCK + t) * 8u + static_cast<uint32_t>(__ffs(bits)) - 1u;
                if (state == 2u) Ap->token[row] = static_cast<int32_t>(id);
                else S.token = id;
            }
        }
        if (state == 2u) return true;
    }

    // ------------------------------------------------------------------ an open row whose draw lies behind its 256 largest (the last of them is S.token by
    // now): a walk over the others in id order. The masses of every 512 neighbours in fixed point, the 512 the walk ends in, then its tokens.
    unsigned long long* mass_at = reinterpret_cast<unsigned long long*>(lds + L.groups);
    for (uint32_t i = t; i < n_blocks; i += WS_BLOCK) mass_at[i] = 0ull;
    __syncthreads();
    const float below = S.walk_below;
    const uint32_t last_id = S.token;
    auto behind = [&](float x, uint32_t id) { return !(x > below || (x == below && id <= last_id)); };  // not one of the 256
    const float k2 = inv_t * 1.44269504088896340736f;  // e^(a inv_t) = 2^(a k2 + a k2lo)
    const float k2lo = static_cast<float>(static_cast<double>(inv_t) * 1.44269504088896340736 - static_cast<double>(k2));
    constexpr double kWalkFix = 1099511627776.0;  // 2^40: a token's mass is 1 at most, and there are 2^20 of them
    auto add_block = [&](const uint4& v, uint32_t j0) __attribute__((always_inline)) {
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
        uint32_t gone = 0u;
        if (TOUCHED) gone = reinterpret_cast<const uint8_t*>(touched)[min(j0 + t, nv - 1u)];
        float s = 0.f;
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) {
            const float x = __uint_as_float(e & 1u ? w4[e >> 1] & 0xffff0000u : w4[e >> 1] << 16);
            const float a = fmaxf(__fsub_rn(x, m), -1e30f);  // (NaN: nothing)
            const float mass = __builtin_amdgcn_exp2f(fmaf(a, k2lo, a * k2));
            s += behind(x, (j0 + t) * 8u + e) && !((gone >> e) & 1u) ? mass : 0.f;
        }
        s = wave_sum(s);
        if (lane == 0u) atomicAdd(&mass_at[(j0 >> 6) + wv], static_cast<unsigned long long>(static_cast<double>(s) * kWalkFix));
    };
    // (from memory again: with the registers' vectors in this code as well, the rows that do not get here would pay for it)
    uint4 ahead[3];
#pragma unroll
    for (uint32_t k = 0; k < 3u; ++k) ahead[k] = row_vector<1>(base, k * WS_BLOCK + t, V);
    for (uint32_t j0 = 0; j0 < nv; j0 += 3u * WS_BLOCK) {  // uniform
#pragma unroll
        for (uint32_t k = 0; k < 3u; ++k) {
            const uint32_t j1 = j0 + k * WS_BLOCK;
            uint4 v = ahead[k];
            ahead[k] = row_vector<1>(base, j1 + 3u * WS_BLOCK + t, V);
            trim(v, j1 + t);
            if (MASKED) mask_out(v, allow[min((j1 + t) >> 2, nW - 1u)] >> ((t & 3u) * 8u));
            if (j1 < nv) add_block(v, j1);  // uniform
        }
    }
    if (TOUCHED)
        for (uint32_t r = t; r < n_touched; r += WS_BLOCK)
            if (behind(adj[r], tid[r])) atomicAdd(&mass_at[tid[r] >> 9], static_cast<unsigned long long>(exact_mass(adj[r]) * kWalkFix));
    __syncthreads();
    uint64_t left = static_cast<uint64_t>(S.walk * kWalkFix);
    const uint32_t at = find_block(mass_at, left);
    if (at == 0xffffffffu) return false;  // (rounding: behind the last one)
    if (wv != at % WS_WAVES) return true;
    const uint32_t round = at / WS_WAVES;
    const uint4 v = load_again(round * WS_BLOCK + t);
    const uint32_t w4[4] = {v.x, v.y, v.z, v.w}, id0 = (round * WS_BLOCK + t) * 8u;
    uint32_t gone = 0u;
    if (TOUCHED && n_touched) gone = reinterpret_cast<const uint8_t*>(touched)[min(id0 >> 3, nv - 1u)];
    double mass[8], mine = 0.0;
#pragma unroll
    for (uint32_t e = 0; e < 8u; ++e) {
        float x = __uint_as_float(e & 1u ? w4[e >> 1] & 0xffff0000u : w4[e >> 1] << 16);
        if (TOUCHED && ((gone >> e) & 1u)) x = id0 + e < V ? adj[rank(id0 + e)] : -INFINITY;
        x = fmaxf(x, -INFINITY);
        mass[e] = x > -INFINITY && behind(x, id0 + e) ? exact_mass(x) : 0.0;
        mine += mass[e];
    }
    const double inc = wave_incl_scan(mine), rest = static_cast<double>(left) * (1.0 / kWalkFix);
    const uint64_t past = __ballot(mine > 0.0 && inc > rest), some = __ballot(mine > 0.0);
    if (some == 0ull) return true;  // (a block with a sum has a token)
    // (rounding: the block's last)
    const uint32_t f = past ? static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(past)) - 1) : 63u - static_cast<uint32_t>(__clzll(static_cast<long long>(some)));
    if (lane == f) {
        double run = inc - mine, unit = 0.0, gap = 0.0;
        uint32_t id = 0;
        bool hit = false;
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e)
            if (!hit && mass[e] > 0.0) {
                const double next = run + mass[e];
                id = id0 + e;
                unit = mass[e];
                gap = fmin(fabs(next - rest), fabs(rest - run));
                hit = next > rest;
                run = next;
            }
        Ap->token[row] = static_cast<int32_t>(id);
        S.unit = unit;
        S.gap_draw = gap;
        write_answers();
    }
    return true;
}

template <bool MASKED, bool TOUCHED, int NV>
__global__ void __launch_bounds__(WS_BLOCK) code_batch_kernel(BatchArgs A) {
    __shared__ CodeShared shared;
    const uint32_t row = blockIdx.x;
#ifdef WS_CODE_TIMERS
    if (threadIdx.x == 0) shared.t0 = clock64();
    if (threadIdx.x < 32) shared.marks[threadIdx.x] = 0;
    __syncthreads();
    const bool done_ = code_row<MASKED, TOUCHED, NV>(A, row, shared);
    if (threadIdx.x == 0) shared.marks[15] = clock64() - shared.t0;
    __syncthreads();
    if (threadIdx.x < 32) A.margin[row * 32 + threadIdx.x] = static_cast<double>(shared.marks[threadIdx.x]);
    if (done_) return;
#else
    if (code_row<MASKED, TOUCHED, NV>(A, row, shared)) return;
#endif
    __syncthreads();  // whatever it left in LDS is dead
    LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    three_pass_row<false>(Ap, row);
}

}  // namespace ws
