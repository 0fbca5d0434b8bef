// topk_rows, dflash_topk and draft_sample_rows for few rows, every row shared by up to sixteen workgroups that hold their share of
// it in registers: the waves list and sum as in ws_few.h (no history, no mask), the part that arrives last sorts about as many
// keys as are asked for. No counterpart in the reference, whose kernels give a row to one workgroup. What bounds it is the
// chain of dependent steps (see ws_few.h). Against shared rows whose parts fitted a histogram to the head of the row and
// whose last part counted the merged list once more (151936 fp32, microseconds a launch): 8 rows, K = 256: 19.6 -> 13.3;
// a draft draw of 8 rows: 26.0 -> 11.6, of which the draw's one wave took 7 and takes 2.5. Since then 13.3 -> 11.8 (top_select, and what ws_few.h names), and of
// the draw's one wave 6.5 K clocks -> 4.4 K: its parameters are asked for at the start, its sums end with the candidates, and the logarithms of the race
// keys are another wave's. (A cycle of 8 sequences and 4 drafts, with its verification: 81.1 us -> 68.3, and 61.4 with ws_accept.h's kernels as they are.)
#pragma once
#include "ws_draft.h"
#include "ws_few.h"

namespace ws {

struct TopSplit {
    uint32_t parts, chunk_log2, rows, together, vecs, slots;  // (together: few_place)
    unsigned char* work;  // kFewRowBytes a row
};

// The K largest logits of this row, by the part of it that arrives last: `list` in descending order (value desc, id asc), F.sum()
// the normaliser. K_of() says how many, once the share is on its way (0: the row is not looked at). Returns 0: another part's business; 1: listed;
// 2: this part has to do the row without the list; and with ORDER false 3: more keys are listed than are sorted by comparing all, n_keys of them, in no order.
template <int NV, bool SUM, bool ORDER, class KOF>
__device__ __forceinline__ int top_share(const float* x, int n, KOF&& K_of, float inv_t, const TopSplit& sp, uint32_t row, uint32_t part, FewShared& F, uint64_t*& list, uint32_t& n_keys) {
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t V = static_cast<uint32_t>(n);
#ifdef WS_SHORT_TIMERS
    if (threadIdx.x == 0) F.t0 = clock64();
#endif
    const FewShare L = FewShare::of<0>(V, sp.parts, part, sp.chunk_log2, sp.vecs, sp.slots);
    const uint32_t j_part = V % 4u ? L.nv - 1u : 0xffffffffu;
    const unsigned char* base = reinterpret_cast<const unsigned char*>(x);
    uint4 q[NV];
#pragma unroll
    for (uint32_t k = 0; k < NV; ++k) q[k] = row_vector<0>(base, L.vec_of(k), V);
    const int K = K_of();
    if (K == 0) return 0;  // (every part of the row sees the same words)
    float v[NV][4], vm[NV], lm = -INFINITY;
#pragma unroll
    for (uint32_t k = 0; k < NV; ++k) {
        if (k + 1u >= L.n_vec) {  // uniform: the round the row ends in, and those behind it
            const uint32_t j = L.vec_of(k);
            if (j == j_part) q[k] = part_vector<0>(q[k], 4u - V % 4u);
            if (j >= L.nv) q[k] = make_uint4(0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu);
        }
        const uint32_t w[4] = {q[k].x, q[k].y, q[k].z, q[k].w};
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) v[k][e] = few_logit(w[e]);
        vm[k] = few_max_of<4u>(v[k]);
        lm = fmaxf(lm, vm[k]);
    }
    FewWant W;
    W.by_k = true;
    W.by_p = false;
    W.top_k = static_cast<uint32_t>(K);
    W.inv_t = inv_t;
    W.min_p = 0.0;
    unsigned char* work = sp.work + static_cast<size_t>(row) * kFewRowBytes;
    if (!few_publish<0, NV, SUM>(L, W, v, vm, lm, nullptr, 0u, !SUM || inv_t > 0.f, work, F)) return 0;
    list = reinterpret_cast<uint64_t*>(lds);
    n_keys = few_collect<SUM>(L, W, work, F, list, []() {});
    if (n_keys < W.top_k || n_keys > kShortCap) return 2;
    const bool sorts = ORDER || n_keys <= WS_BLOCK / 4u;
    if (sorts) list = few_sort(list, n_keys, F);
#ifdef WS_SHORT_TIMERS
    if (threadIdx.x == 0) reinterpret_cast<long long*>(work + 64512)[10] = n_keys;
#endif
    WSF_MARK(8);
    return sorts ? 1 : 3;
}

// The ids of the K largest of the n listed keys (n > K, n <= kShortCap), in no order, to `ids`: the buckets of short_sort, of which only the one that the
// K-th falls in has to be put in order. (8 rows of 151936, K = 256, some 700 keys: the whole list sorted took 7.5 K clocks.)
__device__ __forceinline__ void top_select(uint64_t* list, uint32_t n, uint32_t K, uint32_t* ids, FewShared& F) {
    constexpr uint32_t KPT = kShortCap / WS_BLOCK, NBK = 512u;
    static_assert(NBK == WS_BLOCK, "a bucket a thread");
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6)));
    uint32_t* bc = reinterpret_cast<uint32_t*>(list + kShortCap);  // (behind the list: its sorted copy's place)
    uint32_t* bs = bc + NBK;
    const float m = F.red_f[0];
    uint64_t key[KPT];
    uint32_t bk[KPT], pos[KPT];
    float dmax = 0.f, dsum = 0.f;
    auto down = [&](uint64_t k) { return fminf(__fsub_rn(m, unkey32(static_cast<uint32_t>(k >> 32))), 3e38f); };
#pragma unroll
    for (uint32_t k = 0; k < KPT; ++k)
        if (k * WS_BLOCK < n) {  // uniform
            key[k] = k * WS_BLOCK + t < n ? list[k * WS_BLOCK + t] : 0ull;
            const float d = key[k] ? down(key[k]) : 0.f;
            dmax = fmaxf(dmax, d);
            dsum += d;
        }
    dmax = wave_max(dmax);
    dsum = wave_sum(dsum);
    if (lane == 0u) {
        F.sh.red_f[wv] = dmax;
        F.sh.red_d[wv] = static_cast<double>(dsum);
    }
    bc[t] = 0u;
    __syncthreads();
    dmax = F.sh.red_f[0];
    double total = F.sh.red_d[0];
#pragma unroll
    for (uint32_t w = 1; w < WS_WAVES; ++w) {
        dmax = fmaxf(dmax, F.sh.red_f[w]);
        total += F.sh.red_d[w];
    }
    // (short_sort's logarithmic scale)
    const float mean = fmaxf(dmax - static_cast<float>(total) / static_cast<float>(n), dmax * 1e-6f + 1e-30f), per = 1.f / mean;
    auto level = [&](float d) { return static_cast<float>(__float_as_uint(__fadd_rn(1.f, __fmul_rn(fmaxf(__fsub_rn(dmax, d), 0.f), per))) - 0x3f800000u); };
    const float scale = static_cast<float>(NBK) / (level(0.f) + 1.f);
#pragma unroll
    for (uint32_t k = 0; k < KPT; ++k)
        if (k * WS_BLOCK + t < n) {
            bk[k] = NBK - 1u - min(NBK - 1u, static_cast<uint32_t>(level(down(key[k])) * scale));
            pos[k] = atomicAdd(&bc[bk[k]], 1u);
        }
    __syncthreads();
    if (wv == 0u) {  // eight consecutive counts a lane
        const uint4 a = *reinterpret_cast<const uint4*>(&bc[lane * 8u]), b = *reinterpret_cast<const uint4*>(&bc[lane * 8u + 4u]);
        const uint32_t c[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t own = 0u;
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) own += c[i];
        uint32_t run = wave_incl_scan(own) - own;
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            bs[lane * 8u + i] = run;
            if (run < K && run + c[i] >= K) F.w[6] = lane * 8u + i;  // the K-th falls in this one
            run += c[i];
        }
    }
    __syncthreads();
    const uint32_t last = F.w[6], b0 = bs[last], c0 = bc[last];
#pragma unroll
    for (uint32_t k = 0; k < KPT; ++k)
        if (k * WS_BLOCK + t < n) {
            if (bk[k] < last) ids[bs[bk[k]] + pos[k]] = 0xffffffffu - static_cast<uint32_t>(key[k]);
            else if (bk[k] == last) list[pos[k]] = key[k];  // (every key is in a register)
        }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < KPT; ++k)
        if (k * WS_BLOCK + t < n && bk[k] == last) {
            uint32_t place = b0;
            for (uint32_t i = 0; i < c0; i += 4u) {  // four reads on their way together
                uint64_t o[4];
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) o[q] = list[min(i + q, c0 - 1u)];
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) place += (i + q < c0 && o[q] > key[k]) ? 1u : 0u;
            }
            if (place < K) ids[place] = 0xffffffffu - static_cast<uint32_t>(key[k]);
        }
}

template <int NV>
__global__ void __launch_bounds__(WS_BLOCK) topk_rows_shared(const float* x, int n, int K, float inv_t, int* ids, float* vals, float* stats, TopSplit sp) {
    __shared__ FewShared F;
    uint32_t row_, part;
    if (!few_place(sp.together, sp.rows, row_, part)) return;
    const size_t row = row_;
    x += row * n;
    ids += row * K;
    vals += row * K;
    uint64_t* list;
    uint32_t n_keys;
    const int how = top_share<NV, true, false>(x, n, [&]() { return K; }, inv_t, sp, row_, part, F, list, n_keys);
    if (how == 0) return;
    if (how == 2) {
        __syncthreads();
        topk_one_row(x, n, K, inv_t, ids, vals, stats + 2 * row);
        return;
    }
    // ascending id: every kept entry counts the kept ids below its own, two threads an entry
    const uint32_t t = threadIdx.x, kk = static_cast<uint32_t>(K);
    __shared__ __align__(16) uint32_t kid[512];
    for (uint32_t i = t; i < ((kk + 15u) & ~15u); i += WS_BLOCK) kid[i] = how == 1 && i < kk ? 0xffffffffu - static_cast<uint32_t>(list[i]) : 0xffffffffu;
    if (how == 3) {
        if (n_keys > kk) top_select(list, n_keys, kk, kid, F);
        else if (t < n_keys) kid[t] = 0xffffffffu - static_cast<uint32_t>(list[t]);
    }
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
    uint32_t row_, part;
    if (!few_place(sp.together, sp.rows, row_, part)) return;
    const size_t row = row_;
    x += row * ld;
    ids += row * k;
    vals += row * k;
    uint64_t* list;
    uint32_t n_keys;
    const int how = top_share<NV, false, true>(x, n, [&]() { return k; }, 1.f, sp, row_, part, F, list, n_keys);
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
    uint32_t row, part;
    if (!few_place(sp.together, sp.rows, row, part)) return;
    const int b = static_cast<int>(row);
    if (a.on[b] == 0) return;
    // (all of the row's parameters now: at the end each would be a trip of its own)
    DraftRow D = DraftRow::of(a, b);
    int at = area.v[b];
    asm volatile("" : "+s"(D.top_k), "+s"(D.qoff), "+s"(D.inv_t), "+s"(D.top_p), "+s"(D.min_p), "+s"(D.key), "+s"(at));
    int* c = ctl_all + at;
    uint64_t* list;
    uint32_t n_keys;
    int K = 0;
    const int how = top_share<NV, true, true>(x + static_cast<size_t>(b) * n, n, [&]() { return K = draft_candidates(c, r, D.top_k, n); }, D.inv_t, sp, row, part, F,
                                              list, n_keys);
    if (how == 0) return;
    if (how == 2) {
        __syncthreads();
        draft_sample_row(x, n, ctl_all, area, r, map, a, qbuf, b, K);
        return;
    }
    __shared__ int s_id[kDraftMax];
    __shared__ float s_lg[kDraftMax];
    __shared__ double s_race[kDraftMax];
    const int t = static_cast<int>(threadIdx.x);
    if (t >= 64) {  // another wave works out the logarithms of the candidates' race keys, which depend on nothing that this one does
        const int i = t - 64;
        if (i < K) {
            const int id = static_cast<int>(0xffffffffu - static_cast<uint32_t>(list[i]));
            s_race[i] = draft_race(D.key, map ? map[id] : id);
        }
        __syncthreads();
        return;
    }
    if (t < K) {
        s_id[t] = static_cast<int>(0xffffffffu - static_cast<uint32_t>(list[t]));
        s_lg[t] = unkey32(static_cast<uint32_t>(list[t] >> 32));
    }
    __builtin_amdgcn_wave_barrier();  // (one wave: its LDS stores are done before its loads)
    draft_finish<true>(c, D, r, map, qbuf, K, s_id, s_lg, F.red_f[0], static_cast<float>(F.sum()), [&](int, int from) {
        __syncthreads();
        return s_race[from < K ? from : 0];
    });
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
