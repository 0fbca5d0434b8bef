// topk_rows, dflash_topk and draft_sample_rows for few rows, every row shared by up to sixteen workgroups that hold their share of
// it in registers: the waves list and sum as in ws_few.h (no history, no mask), the part that arrives last sorts about as many
// keys as are asked for. No counterpart in the reference, whose kernels give a row to one workgroup. What bounds it is the
// chain of dependent steps (see ws_few.h). Against shared rows whose parts fitted a histogram to the head of the row and
// whose last part counted the merged list once more (151936 fp32, microseconds a launch): 8 rows, K = 256: 19.6 -> 13.3;
// a draft draw of 8 rows: 26.0 -> 11.6, of which the draw's one wave took 7 and takes 2.5.
#pragma once
#include "ws_draft.h"
#include "ws_few.h"

namespace ws {

struct TopSplit {
    uint32_t parts, chunk_log2;
    unsigned char* work;  // kFewRowBytes a row
};

// The K largest logits of this row, by the part of it that arrives last: `list` in descending order (value desc, id asc), F.sum()
// the normaliser. Returns 0: another part's business; 1: listed; 2: this part has to do the row without the list.
template <int NV, bool SUM>
__device__ __forceinline__ int top_share(const float* x, int n, int K, float inv_t, const TopSplit& sp, uint32_t row, FewShared& F, uint64_t*& list) {
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t V = static_cast<uint32_t>(n);
#ifdef WS_SHORT_TIMERS
    if (threadIdx.x == 0) F.t0 = clock64();
#endif
    const FewShare L = FewShare::of<0>(V, sp.parts, blockIdx.x, sp.chunk_log2);
    const uint32_t j_part = V % 4u ? L.nv - 1u : 0xffffffffu;
    const unsigned char* base = reinterpret_cast<const unsigned char*>(x);
    uint4 q[NV];
#pragma unroll
    for (uint32_t k = 0; k < NV; ++k) q[k] = row_vector<0>(base, L.vec_of(k), V);
    float v[NV][4], lm = -INFINITY;
#pragma unroll
    for (uint32_t k = 0; k < NV; ++k) {
        const uint32_t j = L.vec_of(k);
        if (j_part != 0xffffffffu && j == j_part) q[k] = part_vector<0>(q[k], 4u - V % 4u);
        const uint32_t w[4] = {q[k].x, q[k].y, q[k].z, q[k].w};
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) {
            v[k][e] = j < L.nv ? fmaxf(__uint_as_float(w[e]), -INFINITY) : -INFINITY;
            lm = fmaxf(lm, v[k][e]);
        }
    }
    FewWant W;
    W.by_k = true;
    W.by_p = false;
    W.top_k = static_cast<uint32_t>(K);
    W.inv_t = inv_t;
    W.min_p = 0.0;
    unsigned char* work = sp.work + static_cast<size_t>(row) * kFewRowBytes;
    if (!few_publish<0, NV, SUM>(L, W, v, lm, nullptr, 0u, !SUM || inv_t > 0.f, work, F)) return 0;
    list = reinterpret_cast<uint64_t*>(lds);
    const uint32_t n_keys = few_collect<SUM>(L, W, work, F, list, []() {});
    if (n_keys < W.top_k || n_keys > kShortCap) return 2;
    list = few_sort(list, n_keys, F);
#ifdef WS_SHORT_TIMERS
    if (threadIdx.x == 0) reinterpret_cast<long long*>(work + 64512)[10] = n_keys;
#endif
    WSF_MARK(8);
    return 1;
}

template <int NV>
__global__ void __launch_bounds__(WS_BLOCK) topk_rows_shared(const float* x, int n, int K, float inv_t, int* ids, float* vals, float* stats, TopSplit sp) {
    __shared__ FewShared F;
    const size_t row = blockIdx.y;
    x += row * n;
    ids += row * K;
    vals += row * K;
    uint64_t* list;
    const int how = top_share<NV, true>(x, n, K, inv_t, sp, static_cast<uint32_t>(row), F, list);
    if (how == 0) return;
    if (how == 2) {
        __syncthreads();
        topk_one_row(x, n, K, inv_t, ids, vals, stats + 2 * row);
        return;
    }
    // ascending id: every kept entry counts the kept ids below its own, two threads an entry
    const uint32_t t = threadIdx.x, kk = static_cast<uint32_t>(K);
    __shared__ __align__(16) uint32_t kid[512];
    for (uint32_t i = t; i < ((kk + 15u) & ~15u); i += WS_BLOCK) kid[i] = i < kk ? 0xffffffffu - static_cast<uint32_t>(list[i]) : 0xffffffffu;
    __syncthreads();
    if (t == 0) {
        stats[2 * row] = F.red_f[0];
        stats[2 * row + 1] = static_cast<float>(F.sum());
    }
    const uint32_t half = ((kk + 15u) >> 4 << 3);  // ids each of the two looks at: eight or a multiple
    for (uint32_t i0 = 0; i0 < 2u * kk; i0 += WS_BLOCK) {
        const uint32_t i = (i0 + t) >> 1, lo = (t & 1u) * half;
        const uint32_t id = kid[min(i, kk - 1u)];
        const float logit = x[id];  // as it stands in the row (a key does not tell -0 from +0); never NaN here
        uint32_t place = 0;
        for (uint32_t j = lo; j < lo + half; j += 8u) {
            const uint4 a = *reinterpret_cast<const uint4*>(kid + j), b = *reinterpret_cast<const uint4*>(kid + j + 4u);
            place += (a.x < id ? 1u : 0u) + (a.y < id ? 1u : 0u) + (a.z < id ? 1u : 0u) + (a.w < id ? 1u : 0u) + (b.x < id ? 1u : 0u) + (b.y < id ? 1u : 0u) +
                     (b.z < id ? 1u : 0u) + (b.w < id ? 1u : 0u);
        }
        place += __shfl_xor(place, 1);
        if (i < kk && (t & 1u) == 0u) {
            ids[place] = static_cast<int>(id);
            vals[place] = logit;
        }
    }
#ifdef WS_SHORT_TIMERS
    unsigned char* work = sp.work + row * kFewRowBytes;
    WSF_MARK(9);
#endif
}

template <int NV>
__global__ void __launch_bounds__(WS_BLOCK) dflash_topk_shared(const float* x, int n, int ld, int k, int* ids, float* vals, TopSplit sp) {
    __shared__ FewShared F;
    const size_t row = blockIdx.y;
    x += row * ld;
    ids += row * k;
    vals += row * k;
    uint64_t* list;
    const int how = top_share<NV, false>(x, n, k, 1.f, sp, static_cast<uint32_t>(row), F, list);
    if (how == 0) return;
    if (how == 2) {
        __syncthreads();
        dflash_topk_row(x, n, k, ids, vals);
        return;
    }
    const int t = static_cast<int>(threadIdx.x);
    if (t < k) {
        const uint32_t id = 0xffffffffu - static_cast<uint32_t>(list[t]);
        ids[t] = static_cast<int>(id);
        vals[t] = x[id];
    }
}

template <int NV>
__global__ void __launch_bounds__(WS_BLOCK)
    draft_sample_rows_shared(const float* x, int n, int* ctl_all, RowIdx area, int r, const int* map, DSampArgs a, int* qbuf, TopSplit sp) {
    __shared__ FewShared F;
    const int b = static_cast<int>(blockIdx.y), K = draft_candidates(ctl_all, area, r, a, n, b);
    if (K == 0) return;  // (every part of the row sees the same words)
    uint64_t* list;
    const int how = top_share<NV, true>(x + static_cast<size_t>(b) * n, n, K, a.inv_t[b], sp, static_cast<uint32_t>(b), F, list);
    if (how == 0) return;
    if (how == 2) {
        __syncthreads();
        draft_sample_row(x, n, ctl_all, area, r, map, a, qbuf, b, K);
        return;
    }
    __shared__ int s_id[kDraftMax];
    __shared__ float s_lg[kDraftMax];
    const int t = static_cast<int>(threadIdx.x);
    if (t >= 64) return;
    if (t < K) {
        s_id[t] = static_cast<int>(0xffffffffu - static_cast<uint32_t>(list[t]));
        s_lg[t] = unkey32(static_cast<uint32_t>(list[t] >> 32));
    }
    __builtin_amdgcn_wave_barrier();  // (one wave: its LDS stores are done before its loads)
    draft_finish<true>(ctl_all, area, r, map, a, qbuf, b, K, s_id, s_lg, F.red_f[0], static_cast<float>(F.sum()));
#ifdef WS_SHORT_TIMERS
    unsigned char* work = sp.work + static_cast<size_t>(b) * kFewRowBytes;
    WSF_MARK(9);
#endif
}

// ---- greedy picks of few rows: every part leaves the largest {logit, lowest index} of its stretch as an order key in the row's
// scratch, once as it is and once mixed with a tag that no other launch has, waits until both have arrived and looks at all
// parts' places: where the two words of every part differ by the tag, everybody is there, and whoever sees that picks. The one
// whose words come last sees it, others may as well and write the same. So the scratch may hold anything when the launch
// begins, a caller need not clear or keep it, and no counter has to be reset. (What it holds by chance makes a pair of this tag
// once in 2^64; the picker breaks the row's pairs, for a captured launch has its tag again at every replay.) What bounds it: the
// stretch's loads (76 KB a compute unit at 32 rows of 151936) and two trips to memory; 32 rows took 10.4 us with a compute unit a
// row, and take 6.5.
struct PickArgs {  // (one argument of the launch: ten of them take the host 0.7 us longer)
    const float* x;
    int* out;
    unsigned long long* scratch;
    unsigned long long tag;
    unsigned n, parts;
    int* ids;
    int* pos;
    int advance;
};
struct PickArgsTo : PickArgs {
    RowIdx dst;  // argmax_rows_to: where each row's pick goes
};
template <int MODE>  // 0: out[row]; 1: out[dst.v[row]]; 2: one row, out[0], ids[0] and pos[0] += advance
__global__ void __launch_bounds__(WS_BLOCK) argmax_shared(std::conditional_t<MODE == 1, PickArgsTo, PickArgs> A) {
    __shared__ unsigned long long red[WS_WAVES];
    const uint32_t row = blockIdx.y, part = blockIdx.x, t = threadIdx.x, lane = t & 63u, V = A.n, parts = A.parts;
    const unsigned long long tag = A.tag;
    const unsigned char* base = reinterpret_cast<const unsigned char*>(A.x + static_cast<size_t>(row) * V);
    unsigned long long* scratch = A.scratch + static_cast<size_t>(row) * (2u * parts);
    const uint32_t nv = (V + 3u) / 4u, per = (nv + parts - 1u) / parts, j0 = min(part * per, nv), j1 = min(j0 + per, nv);
    float best = -INFINITY;
    uint32_t at = 0xffffffffu;
    auto take = [&](const uint4& q, uint32_t j) {  // (a last vector that overlaps the one before it offers tokens twice: no harm, but their places count from the row's end)
        const float v[4] = {fmaxf(__uint_as_float(q.x), -INFINITY), fmaxf(__uint_as_float(q.y), -INFINITY), fmaxf(__uint_as_float(q.z), -INFINITY),
                            fmaxf(__uint_as_float(q.w), -INFINITY)};
        const float m = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
        if (m > best) {
            best = m;
            at = min(4u * j, V - 4u) + (v[0] == m ? 0u : (v[1] == m ? 1u : (v[2] == m ? 2u : 3u)));
        }
    };
    constexpr uint32_t kU = 10u;  // loads of a thread on their way together
    for (uint32_t jb = j0; jb < j1; jb += kU * WS_BLOCK) {
        uint4 q[kU];
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) q[u] = row_vector<0>(base, min(jb + u * WS_BLOCK + t, j1 - 1u), V);
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) take(q[u], min(jb + u * WS_BLOCK + t, j1 - 1u));  // (past the stretch: its last vector once more)
    }
    auto wave_pick = [&](float v, uint32_t i) {  // the wave's largest, lowest index on ties, as a key
        const float m = wave_max(v);
        const uint32_t first = wave_min_u32(v == m ? i : 0xffffffffu);
        return (static_cast<unsigned long long>(key32(m)) << 32) | (0xffffffffu - first);
    };
    const unsigned long long mine = wave_pick(best, at);
    if (lane == 0u) red[t >> 6] = mine;
    __syncthreads();
    if (t >= 64u) return;
    auto word = [&](uint32_t p, uint32_t second) { return &scratch[2u * p + second]; };
    if (t == 0) {
        unsigned long long k = red[0];
#pragma unroll
        for (uint32_t w = 1; w < WS_WAVES; ++w) k = k > red[w] ? k : red[w];
        __hip_atomic_store(word(part, 0u), k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(word(part, 1u), k ^ tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the wave's: both words have arrived before it looks at the others')
    unsigned long long k = 0ull, k2 = tag;
    if (lane < parts) {
        k = __hip_atomic_load(word(lane, 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        k2 = __hip_atomic_load(word(lane, 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (__ballot((k ^ k2) != tag) != 0ull) return;  // somebody is still to come
    if (MODE == 2) {  // (pos moves once: of several who see everybody, the one who takes the first pair apart)
        bool mine_to_do = false;
        if (lane == 0u) {
            unsigned long long was = k2;
            mine_to_do = __hip_atomic_compare_exchange_strong(word(0u, 1u), &was, 0ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (__ballot(mine_to_do) == 0ull) return;
    }
    if (lane < parts) {  // no pair of this tag is left behind
        __hip_atomic_store(word(lane, 0u), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(word(lane, 1u), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool some = lane < parts;
    const unsigned long long r = wave_pick(some ? unkey32(static_cast<uint32_t>(k >> 32)) : -INFINITY, some ? 0xffffffffu - static_cast<uint32_t>(k) : 0xffffffffu);
    if (lane == 0u) {
        const uint32_t i = 0xffffffffu - static_cast<uint32_t>(r);
        const int id = i == 0xffffffffu ? 0 : static_cast<int>(i);  // (a row without a number: the first index)
        if constexpr (MODE == 1) A.out[A.dst.v[row]] = id;
        else A.out[row] = id;
        if (MODE == 2) {
            A.ids[0] = id;
            A.pos[0] += A.advance;
        }
    }
}

}  // namespace ws
