// draft_sample_rows for gfx950: the draft distribution q of a draft-head row and the race draw coupled to the
// target sampler (reference: kernels/spec_sample.hip:34-205, same arguments, control-area and q-buffer layout;
// host statement of q: src/common/spec_sample.cpp:34-81).
// One pass for {max, sum exp((x - max) * inv_t)} (NaN adds nothing, kernels/spec_sample.hip:63-66) and the
// K = min(top_k, 32) largest logits (ties at the cut: lowest ids) - the short-list route of ws_topk.h -, then one wave
// finishes in the reference's arithmetic: f32 probabilities and filters in the reference's order, double-precision race keys.
#pragma once

#include "ws_common.h"
#include "ws_pick.h"
#include "ws_topk.h"

struct DSampArgs {
    int on[32];
    int top_k[32];
    int qoff[32];
    float inv_t[32];
    float top_p[32];
    float min_p[32];
    unsigned key_lo[32];
    unsigned key_hi[32];
};

namespace ws {
constexpr int kDraftMax = 32;  // candidates of a draft distribution
// whether a row is drawn at draft position r (c: its control area), and with how many candidates
__device__ __forceinline__ int draft_candidates(const int* c, int r, int tk, int n) {
    if (c[49] != 0 && c[48] <= r) return 0;  // chain stopped by the p-min cutoff at or before r
    return min((tk > 0 && tk < kDraftMax) ? tk : kDraftMax, n);
}
// a row's parameters
struct DraftRow {
    int top_k, qoff;
    float inv_t, top_p, min_p;
    uint64_t key;
    __device__ __forceinline__ static DraftRow of(const DSampArgs& a, int b) {
        return {a.top_k[b], a.qoff[b], a.inv_t[b], a.top_p[b], a.min_p[b], (static_cast<uint64_t>(a.key_hi[b]) << 32) | a.key_lo[b]};
    }
};
// ln(1 - U) of a token's race key (src/common/spec_sample.cpp:83-101)
__device__ __forceinline__ double draft_race(uint64_t key, int id) {
    return log(1.0 - ws::unit53(ws::mix64(key + (static_cast<uint64_t>(static_cast<uint32_t>(id)) + 1ull) * 0xE7037ED1A0B428DBull)));
}
// The draw of a row from its K largest logits (LDS: s_id, s_lg; any order that puts the lower of two equal logits' ids first),
// maximum and normaliser. One wave calls it. race(id, place): draft_race of the lane's candidate, which the list has at `place`; it is asked for last.
template <bool SORTED, class RACE>  // s_id, s_lg: in order (logit desc, id asc)
__device__ __forceinline__ void draft_finish(int* c, const DraftRow& D, int r, const int* map, int* qbuf, int K, const int* s_id, const float* s_lg, float top,
                                             float sum, RACE&& race) {
    constexpr int QMAX = kDraftMax;
    const int tk = D.top_k;
    // ---- one wave, lane i = candidate i (QMAX = 32 <= 64 lanes). What the reference's single thread does in a fixed order -
    // the running float sums of the filters - is done in that order by every lane for itself, with the candidates' values
    // read from their lanes (v_readlane, a few clocks a term; through the LDS crossbar the loops below took 7 us); what is
    // independent per candidate (its place in the order, its probability and its share, its race key with a
    // double-precision logarithm) is done by the candidate's lane.
    const int lane = threadIdx.x;
    const bool live = lane < K;
    auto value_at = [](float v, int j_) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j_)); };
    constexpr int kStep = 4;  // terms between two looks at whether any are left
    // front to back over the first n lanes (x + 0 is x)
    auto sum_of = [&](float v, int n) {
        const float own = lane < n ? v : 0.f;
        float z = 0.f;
#pragma unroll
        for (int i0 = 0; i0 < QMAX; i0 += kStep)
            if (i0 < n)  // uniform
#pragma unroll
                for (int i = i0; i < i0 + kStep; ++i) z = __fadd_rn(z, value_at(own, i));
        return z;
    };
    const int my_id = live ? (map ? map[s_id[lane]] : s_id[lane]) : 0x7fffffff;
    const float my_lg = live ? s_lg[lane] : -INFINITY;
    int id = my_id, from = lane;  // the lane's candidate, and its place in the list
    float lg = my_lg;
    if (!SORTED || map) {  // uniform
        int place = 0;  // logit desc, (mapped) id asc, then the position in the list
        for (int j = 0; j < K; ++j) {
            const float lj = value_at(my_lg, j);
            const int ij = __builtin_amdgcn_readlane(my_id, j);
            place += (lj > my_lg || (lj == my_lg && (ij < my_id || (ij == my_id && j < lane)))) ? 1 : 0;
        }
        // lane r takes the candidate of place r
        const int dst = (live ? place : lane) << 2;
        id = __builtin_amdgcn_ds_permute(dst, my_id);
        lg = __int_as_float(__builtin_amdgcn_ds_permute(dst, __float_as_int(my_lg)));
        from = __builtin_amdgcn_ds_permute(dst, lane);
    }
    float p = live ? __fdiv_rn(expf(__fmul_rn(__fsub_rn(lg, top), D.inv_t)), sum) : 0.f;
    int nk = K;
    const bool closed = tk > 0 && tk <= K;
    if (closed) nk = tk;
    const float top_p = D.top_p;
    if (top_p < 1.f) {
        const float z = closed ? sum_of(p, nk) : 1.f;
        const float share = lane < nk ? __fdiv_rn(p, z) : 0.f;
        float cum = 0.f;
        int before = 0;  // candidates at which the running share has not reached top_p
#pragma unroll
        for (int j0 = 0; j0 < QMAX; j0 += kStep)
            if (j0 < nk)  // uniform
#pragma unroll
                for (int j = j0; j < j0 + kStep; ++j) {
                    cum = __fadd_rn(cum, value_at(share, j));
                    before += cum >= top_p ? 0 : 1;
                }
        nk = min(nk, before + 1);
    }
    const float min_p = D.min_p;
    if (min_p > 0.f && nk > 0) {
        const float floor_p = __fmul_rn(min_p, value_at(p, 0));
        const uint64_t below = __ballot(lane < nk && !(p >= floor_p));  // the first of them ends the kept candidates
        if (below) nk = max(1, __ffsll(static_cast<unsigned long long>(below)) - 1);
    }
    const float z = sum_of(p, nk);
    p = lane < nk ? __fdiv_rn(p, z) : 0.f;
    // race: argmin E(v) / q(v), E(v) = -ln(1 - U(key, v)) (src/common/spec_sample.cpp:83-101); the earlier candidate on
    // equal keys, candidate 0 when none has a probability
    const double ln = race(id, from);
    double k = __longlong_as_double(0x7FF0000000000000ll);
    if (lane < nk && p > 0.f) k = __builtin_fabs(ln / static_cast<double>(p));  // (the logarithm is not above 0; and no -0)
    // (keys are not negative: their order is that of their bits)
    const uint64_t kb = static_cast<uint64_t>(__double_as_longlong(k));
    const uint32_t k_hi = static_cast<uint32_t>(kb >> 32), least_hi = wave_min_u32(k_hi);
    const uint32_t k_lo = k_hi == least_hi ? static_cast<uint32_t>(kb) : 0xffffffffu, least_lo = wave_min_u32(k_lo);
    const int pick = least_hi < 0x7FF00000u ? __ffsll(static_cast<unsigned long long>(__ballot(k_hi == least_hi && k_lo == least_lo))) - 1 : 0;
    const int picked = __builtin_amdgcn_readlane(id, pick);
    int* q = qbuf + D.qoff;
    if (lane == 0) {
        c[16 + r] = picked;
        q[0] = nk;
    }
    if (lane < nk) {
        q[1 + lane] = id;
        q[1 + QMAX + lane] = __float_as_int(p);
    }
}

__device__ __forceinline__ void draft_sample_row(const float* x, int n, int* ctl_all, const RowIdx& area, int r, const int* map,
                                                 const DSampArgs& a, int* qbuf, int b, int K) {
    __shared__ int s_id[kDraftMax];
    __shared__ float s_lg[kDraftMax];
    __shared__ float s_stats[2];
    // one pass over the row: {max, sum exp((x - max) * inv_t)} and the K largest logits in id order, ties at the cut to
    // the lowest ids (the short-list route of topk_rows)
    ws::topk_one_row(x + static_cast<size_t>(b) * n, n, K, a.inv_t[b], s_id, s_lg, s_stats);
    __syncthreads();
    const DraftRow D = DraftRow::of(a, b);
    if (threadIdx.x < 64)
        draft_finish<false>(ctl_all + area.v[b], D, r, map, qbuf, K, s_id, s_lg, s_stats[0], s_stats[1], [&](int id, int) { return draft_race(D.key, id); });
}
}  // namespace ws

#ifndef WS_NO_NAMED_KERNELS
extern "C" __global__ void __launch_bounds__(WS_BLOCK)
    draft_sample_rows(const float* x, int n, int* ctl_all, RowIdx area, int r, const int* map, DSampArgs a, int* qbuf) {
    const int b = static_cast<int>(blockIdx.x);
    if (a.on[b] == 0) return;
    const int K = ws::draft_candidates(ctl_all + area.v[b], r, a.top_k[b], n);
    if (K > 0) ws::draft_sample_row(x, n, ctl_all, area, r, map, a, qbuf, b, K);
}
#endif
