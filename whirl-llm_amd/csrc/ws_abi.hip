// C ABI of libwhirl_sampling_hip.so (include/whirl_sampling_abi.h): argument checks on the host, launch geometry,
// by-value launch structs. No allocation, no synchronisation, no host copies of device data.
#include "../../include/whirl_sampling_abi.h"

#include <hip/hip_runtime.h>

#include <atomic>

#include <cstring>

#include "ws_accept.h"
#include "ws_adjust.h"
#include "ws_common.h"
#include "ws_draft.h"
#include "ws_pick.h"
#include "ws_sample.h"
#include "ws_spec.h"
#include "ws_lds_limit.h"
#include "ws_topk.h"

namespace ws {
// ws_fused.hip: the fused-sweep kernel, built for 512-thread workgroups
int launch_fused(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit);
// ws_split.hip: the same with rows split over several workgroups
int launch_split(hipStream_t stream, const BatchArgs& a, unsigned blocks, unsigned lds_bytes, unsigned lds_limit);
// ws_fused_kept.hip, ws_split_kept.hip: the builds of the two that can write the kept-set dump
int launch_fused_kept(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit);
int launch_split_kept(hipStream_t stream, const BatchArgs& a, unsigned blocks, unsigned lds_bytes, unsigned lds_limit);
// ws_lean.hip: the lean single-sweep kernel (1024 threads a row) for batches of unsplit rows without a top-k
int launch_lean(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit);
// each of them raises its kernels' dynamic LDS limit on the current device (once; the launchers call them too)
int prepare_fused(unsigned lds_limit);
int prepare_split(unsigned lds_limit);
int prepare_fused_kept(unsigned lds_limit);
int prepare_split_kept(unsigned lds_limit);
int prepare_lean(unsigned lds_limit);
// ws_short.hip: the short-list kernel for batches whose rows all have a bounded top-k
int launch_short(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit);
int prepare_short(unsigned lds_limit);
int launch_short_rest(hipStream_t stream, const BatchArgs& a, unsigned blocks, unsigned lds_bytes, unsigned lds_limit);
// ws_twin.hip: the same for rows that are not shared, two of them a compute unit
int launch_twin(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit);
int prepare_twin(unsigned lds_limit);
// ws_code.hip: bf16 rows, held in registers and counted by value
int launch_code(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit);
int prepare_code(unsigned lds_limit);
uint64_t code_lds_bytes(uint32_t vocab, uint32_t cap, uint32_t copies);
// ws_few.hip: the same rows shared between workgroups that hold them in registers
// (leave: a row that `own` takes along may be left undone, marked in its flags)
int launch_few(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit, const OwnRow* own, bool leave);
int prepare_few(unsigned lds_limit);
// ws_top.hip: topk_rows, dflash_topk and draft_sample_rows with rows shared between workgroups
int launch_topk_shared(hipStream_t stream, const float* x, int n, int K, float inv_t, int* ids, float* vals, float* stats, unsigned rows, unsigned parts,
                       unsigned chunk_log2, unsigned together, unsigned char* work);
int launch_dflash_shared(hipStream_t stream, const float* x, int n, int ld, int k, int* ids, float* vals, unsigned rows, unsigned parts, unsigned chunk_log2,
                         unsigned together, unsigned char* work);
int launch_draft_shared(hipStream_t stream, const float* x, int n, int* ctl_all, const void* area, int r, const int* map, const void* args, int* qbuf,
                        unsigned rows, unsigned parts, unsigned chunk_log2, unsigned together, unsigned char* work);
int launch_argmax_shared(hipStream_t stream, int mode, const float* x, int n, int* out, const void* dst, int* ids, int* pos, int advance, unsigned rows,
                         unsigned parts, unsigned long long* scratch, unsigned long long tag);
int prepare_top();
}  // namespace ws

namespace {

inline hipStream_t S(void* s) { return static_cast<hipStream_t>(s); }
inline int done() { return static_cast<int>(hipGetLastError()); }

constexpr uint32_t kMaxLds = 160u * 1024u;  // LDS per workgroup on gfx950
// what the sampler kernel declares statically (reduction scratch, exponent tables, the exact path's words), rounded up
#ifdef WS_PHASE_TIMERS
constexpr uint32_t kStaticLds = 4096u + 512u;  // + the phase marks
#else
constexpr uint32_t kStaticLds = 4096u;
#endif
// the short-list kernel's own words and those of both builds of the three-pass code it calls (8.2 KiB)
constexpr uint32_t kStaticShort = 9216u;
// the same for the kernel of two rows a compute unit, which calls nothing
constexpr uint32_t kStaticTwin = 1024u;
// the same for the kernel of few rows
constexpr uint32_t kStaticFew = 8192u;
// the same for the kernel of bf16 rows
constexpr uint32_t kStaticCode = 14336u;
// the lean kernel's own tables and those of the three-pass code it calls
#ifdef WS_PHASE_TIMERS
constexpr uint32_t kStaticLean = 11776u + 768u;
#else
constexpr uint32_t kStaticLean = 11776u;
#endif

struct BatchPlan {
    uint32_t patch_cap;
    uint32_t lds_ab;
    uint32_t lds_cnt;
    uint32_t lds_tie;
    uint32_t lds_total;
    bool fused;
    bool lean;            // the lean kernel can take the batch when its rows are not split (no top-k, no optional outputs)
    uint32_t lean_tie;    // its second histogram copy (0: none), its dynamic LDS, and the spare LDS of the three-pass code it calls
    uint32_t lean_total;
    uint32_t lean_fb_tie;
    bool shortlist;       // the short-list kernel takes the batch: every row has a top-k of at most top_k_max (the caller's word)
    uint32_t short_ab, short_cnt, short_total, short_fb_tie, short_fb_ab;  // its LDS: bitmap at short_ab, rank words at short_cnt
    bool twin;            // its rows go two a compute unit (ws_twin.h)
    uint32_t twin_ab, twin_tabs, twin_total;  // LDS of those: the bitmap, the tables, all
    uint32_t few_parts, few_total;  // short-list rows shared between this many workgroups each (0: not), and the dynamic LDS of those
    bool code;            // the kernel of bf16 rows takes the batch
    uint32_t code_head;   // its masses (BatchArgs)
    float code_above;
    uint32_t code_cap, code_copies, code_total, code_fb_tie, code_fb_ab;  // entries its tables take, copies of its counts, its dynamic LDS, and the three-pass code's layout in it
    uint32_t split_log2;  // the most parts per row that pay for this batch
    uint64_t workspace_min;  // split rows: the least that lets them split (no staging areas), 0 when nothing is split
    uint64_t workspace;   // bytes for that
    int err;
};

// compute units of the current device (one workgroup of the sampler per unit)
int compute_units() {
    static std::atomic<int> known[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = known[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = -1;
        known[dev].store(n, std::memory_order_relaxed);
    }
    return n > 0 ? n : 0;
}

// Whether a shared row's parts go to one chiplet: where its compute units take all parts of its rows at once. (What the parts leave for each other and
// the ids and parameters they all read then come from one L2. Apart and together, us: one row of 20000 9.9 / 9.7, of 151936 10.6 / 10.2, of 262144 11.5 / 11.3, a
// decode step with parameters in host memory 20.7 / 20.1; 5 rows level.)
uint32_t parts_together(uint32_t parts, uint32_t rows) {
    return (rows + ws::kChiplets - 1u) / ws::kChiplets * parts <= static_cast<uint32_t>(compute_units()) / ws::kChiplets ? 1u : 0u;
}

// Short-list rows that ws_few.h does not take - too long for the registers of as many workgroups as there are compute units
// for, or with histories too long for its lists - shared by the short-list kernel's own workgroups, which sweep a slice each: 2^n
// of them, 16 at most, of at least 8192 tokens, within the compute units (a second round of workgroups is not worth it).
// Unshared and shared microseconds, top-k 50 with 1000-id histories: 60 rows of 262144 fp32 47.0 / 35.0, 90 of 151936 36.7 /
// 33.4, 120 of 262144 48.9 / 44.0; min-p alone: 90 of 262144 65.7 / 48.0; 64 of 151936 with 8192 ids each 42.3 / 34.1.
uint32_t short_split_log2(const ws_batch* b) {
    if (b->max_split == 1u) return 0u;
    const uint32_t cus = static_cast<uint32_t>(compute_units()), most = b->max_split ? b->max_split : 16u;
    uint32_t lg = 0;
    while (lg < 4u && (2u << lg) <= most && uint64_t{b->rows} * (2u << lg) <= cus && b->vocab / (2u << lg) >= 8192u) ++lg;
    return lg;
}

// Few rows of the short-list kind: how many workgroups share a row. A share fits the registers of 512 threads (80 tokens
// each) and has 2048 tokens at least; as many parts as the compute units allow, up to 16 - a wide top-k gets 8 at most, its
// waves' lists need the room. Where the compute units allow fewer parts than that takes, shares of 112 tokens a thread are
// tried (two parts hold 114688 tokens, three 172032: unshared and shared microseconds, top-k 40: 90 rows of 82000 fp32
// 23.3 / 18.9, 70 of 151936 33.2 / 25.3, 90 of 92736 bf16 32 / 17). More workgroups than compute units: nobody waits for
// anybody, but the second round of them costs more than it saves (181 rows of 44992 fp32 22.4 / 32.7, 160 of 82000 bf16
// 29 / 32), bf16 rows aside whose slices in the short-list kernel would be longer than 90000 tokens: two rounds take 35 to 39 us
// whatever the length, such a slice more and more (bf16, top-k 50, its slices and two rounds here: 86 rows of 131072 30.3 / 37.3, 86
// of 151936 35.4 / 36.3, 66 of 200000 38.5 / 34.5, 86 of 200000 38.9 / 38.2, 64 of 262144 - slices of 65536 - 32.0 / 37.3, 73
// of 262144 42.7 / 39.2).
void few_plan(const ws_batch* b, uint64_t cap, uint64_t maps, BatchPlan& p) {
    p.few_parts = 0;
    if (b->max_split == 1u || cap > ws::kFewLists) return;
    const uint32_t cus = static_cast<uint32_t>(compute_units());
    const uint32_t share = ws::kFewShare;
    uint32_t most = b->top_k_max > 512u ? 8u : ws::kFewMaxParts;
    if (b->max_split && b->max_split < most) most = b->max_split;
    const uint32_t least = (b->vocab + share - 1u) / share;
    uint32_t parts = cus / b->rows;
    if (parts > most) parts = most;
    if (parts > b->vocab / 2048u) parts = b->vocab / 2048u;
    if (parts < least && (parts < 2u || uint64_t{parts} * ws::kFewWide < b->vocab)) parts = least;
    if (cap > uint64_t{parts} * 1600u) return;  // (touched tokens of a share: room for 2048)
    const bool twice = b->dtype == WS_DTYPE_BF16 && b->vocab >> short_split_log2(b) > 90000u;
    if (parts < 2u || parts > most || static_cast<uint64_t>(b->rows) * parts > (twice ? 2ull : 1ull) * cus) return;
    const uint64_t three = (cap * 8u > 65536u ? ((cap * 8u + 15u) & ~uint64_t{15}) : 65536u) + maps;
    const uint32_t room = parts < least ? ws::kFewWide : ws::kFewShare;
    const uint64_t own = 32768u + room * 2u + ws::few_bit_words(room / 512u) * 2048u;
    const uint64_t total = own > three ? own : three;
    if (total + kStaticFew > kMaxLds) return;
    p.few_parts = parts;
    p.few_total = static_cast<uint32_t>(total);
    p.workspace = p.workspace_min = uint64_t{b->rows} * ws::kFewRowBytes;
}

// bf16 rows of ws_code.h: any filters, any alignment; no optional outputs and no race. Two copies of the counts where there is room for
// them beside the tables of the history and bias entries: with one, rows of tied logits queue up at its words.
void code_plan(const ws_batch* b, uint64_t cap, uint64_t maps, uint64_t spare_bytes, BatchPlan& p) {
    p.code = false;
    if (b->dtype != WS_DTYPE_BF16 || b->mode != WS_MODE_AUTO || b->vocab < 8u || b->kept_ids || b->query_prob || b->entropy || b->race ||
        (b->bias_ids && b->max_bias > 2047u))
        return;
    p.code_cap = (static_cast<uint32_t>(cap) + 3u) & ~3u;
    // The masses of rows that are not of the short-list kind go by the bins of the other kernels such rows can get - with another dump, draw
    // or address - so that a cut among thousands of tokens falls on the same one: ws_sample.h's anchor, or for unshared rows without a top-k
    // ws_lean.h's.
    const bool shared = b->max_split != 1u && uint64_t{b->rows} * 4u <= static_cast<uint64_t>(compute_units()) && b->vocab >= 65536u;
    p.code_head = p.shortlist ? 0u : (p.fused ? 2u : 1u);
    p.code_above = p.fused && !b->top_k && !shared ? 12.f : 8.f;
    const uint64_t three = (cap * 8u > 65536u ? ((cap * 8u + 15u) & ~uint64_t{15}) : 65536u) + maps;
    for (p.code_copies = 2; p.code_copies > 0; --p.code_copies) {
        uint64_t total = ws::code_lds_bytes(b->vocab, p.code_cap, p.code_copies);
        if (total < three) total = three;
        if (total + kStaticCode > kMaxLds) continue;
        p.code = true;
        p.code_fb_ab = static_cast<uint32_t>(three - maps);
        p.code_fb_tie = three + spare_bytes <= total ? static_cast<uint32_t>((three + 15u) & ~uint64_t{15}) : 0u;
        p.code_total = static_cast<uint32_t>(total);
        return;
    }
}

// Rows of the short-list kind that go two a compute unit (ws_twin.h): more of them than compute units. Its sweep is no faster than ws_short.h's, one
// row a unit, and the kernel behind it that looks for rows left over takes 3 us: 256 rows of 151936, ws_short.h and ws_twin.h, 44.7 / 48.6; 300 rows
// 77.0 / 65.0, 512 82.2 / 73.2, 1000 of 8000 55.8 / 38.5.
bool twin_rows(const ws_batch* b) {
    const int cus = compute_units();
    return cus > 0 && b->rows > static_cast<uint32_t>(cus);
}

// bf16 rows with a top-k, more of them than compute units: whether ws_twin.h takes them or ws_code.h. ws_twin.h sorts a list of some 1.5 top-k keys, the time of
// which grows with the top-k, and its sweep costs more a token; touched tokens are cheaper in it. So it takes short rows with touched tokens and a list that is
// not long, and rows so long that ws_code.h reads two fifths of them twice, where two of its own fit a compute unit. Microseconds, ws_twin.h and ws_code.h (N(0, 2) rows;
// histories of 1000 ids but where it says so):
//   1000 rows of    8000: top-k 50 37.8 / 62.6, 128 44.8 / 63.3, 300 49.6 / 64.6; without histories 30.5 / 36.4, 37.4 / 36.4, 41.5 / 36.4
//               of 12288: 42.0 / 61.8, 50.5 / 65.4, 55.5 / 65.2
//               of 16384: 45.6 / 61.6, 55.3 / 65.2, 61.2 / 66.6; 16 ids 43.3 / 54.0, 52.4 / 54.9, 59.8 / 54.8; no ids 37.2 / 38.2 (rows of raised tokens 44.1 / 37.9), 47.2 / 38.5
//   512 rows of  24000: 29.3 / 33.3, 36.4 / 35.0, 41.5 / 36.6; 16 ids 28.3 / 29.5, 36.0 / 29.4; no ids 25.1 / 21.4
//            of  28032: 32.3 / 33.6, 37.4 / 34.7; 16 ids 30.9 / 30.0; raised tokens (600 rows) 55.8 / 46.2
//            of 151936: 63.0 / 56.7, 66.7 / 57.1       of 220032: 74.3 / 71.2, 80.2 / 70.5
//            of 245760: 78.5 / 80.5, 82.6 / 80.2       of 262144: 84.2 / 88.1, 88.9 / 88.2; no ids (400 rows) 74.5 / 65.0
//   400 masked rows (three tokens in ten) of 200000: 70.4 / 71.1, 73.4 / 71.8; of 262144 83.4 / 96.1, 87.6 / 96.0, top-k 300 97.1 / 97.1
//   300 rows of 360000, two a unit: 91.6 / 99.2, 98.9 / 99.7; of 400000, one: 134.7 / 109.1
bool twin_pays(const ws_batch* b, uint64_t cap, const BatchPlan& p) {
    const uint32_t k = b->top_k_max, V = b->vocab;
    if (cap == 0) return k <= 64u && V <= 8192u;
    if (V >= 245760u) return p.twin_total <= kMaxLds / 2u - kStaticTwin && k <= (b->allow ? 128u : 64u);
    return V <= (k <= 64u ? 24576u : k <= 128u ? 16384u : k <= 256u ? 12288u : 0u);
}

// bf16 rows of the short-list kind: ws_code.h, ws_few.h or ws_short.h. Few rows are ws_few.h's: it shares them, and its lists are short -
// but a list of some hundred keys has to be sorted, which costs more than counting a row that is not long, and two workgroups a row
// are not much of a share. Microseconds, ws_few.h and ws_code.h (1000-id histories): top-k 50: 64 rows of 50257 16.0 / 18.4, 100 rows 19.9 /
// 17.9, 100 of 80000 21.2 / 18.9, 100 of 32000 16.1 / 16.4, 64 of 151936 21.5 / 24.2; top-k 300: 1 of 32000 16.9 / 14.8, 8 of 151936 18.6 / 23.7;
// top-k 600 and 1000: 8 of 32000 20.5 / 16.3 and 22.2 / 16.6, 8 of 151936 24.8 / 24.7 and 29.2 / 24.6, 16 of 262144 29.5 / 35.5 and 34.8 / 35.9;
// min-p alone: 100 of 50257 18.2 / 18.5, 128 of 60000 18.9 / 19.5. What ws_few.h does not take: top-k 50, ws_short.h and ws_code.h: 200 of 32000 24.9 /
// 16.5, 1000 of 8000 with a min-p 62.2 / 59.1, 256 of 151936 52.2 / 29.4, 400 of 262144 118.6 / 90.0. Rows without a top-k have a short list and nothing to
// estimate: 150 of 20000 14.3 / 16.5, 1000 of 8000 46.2 / 56.3, 300 of 40000 31.9 / 31.2, 256 of 50257 22.5 / 20.0, 256 of 151936 45.1 / 30.4; longer than the
// registers hold and in four slices or more: 60 of 262144 32.0 / 37.9, in two: 100 of 262144 44.7 / 38.2. More rows than compute units: see twin_pays.
void code_or_short(const ws_batch* b, uint64_t cap, BatchPlan& p) {
    const bool by_k = b->top_k && b->top_k_max >= 1u;
    if (p.few_parts) {
        const bool long_lists = b->top_k_max > 512u ? b->vocab <= 163840u : b->top_k_max > 256u && b->vocab <= 40960u;
        p.code = by_k && (long_lists || (p.few_parts <= 2u && b->vocab > 32768u));
        if (p.code) p.few_parts = 0;
    } else if (by_k) {
        p.code = !(twin_rows(b) && twin_pays(b, cap, p));
    } else {
        p.code = b->vocab > 40960u && !(b->vocab > 163840u && short_split_log2(b) >= 2u);
    }
    if (p.code) p.workspace = p.workspace_min = 0;
}

// LDS of a row of ws_twin.h: the list and its spare places, the bitmap, the tables behind it; or, where that is more than half a compute unit's and the
// other way is not, the tables below the bitmap, in the upper part of the list's place as far as they have to (not over the sample's bin
// counts, which are in use with them; the touched tokens above the threshold are listed in what is left below the tables). Two rows a unit
// come before spare places: without them the sweep takes its places one by one.
void twin_plan(uint32_t nW, uint64_t cap, BatchPlan& p) {
    const uint64_t map = uint64_t{nW} * 4u, tabs = ((uint64_t{nW} * 2u + 3u) & ~uint64_t{3}) + ((cap * 2u + 3u) & ~uint64_t{3});
    const uint64_t half = kMaxLds / 2u - kStaticTwin, list = 32768u;
    uint64_t ab = list, total = list + map + tabs;
    const uint64_t spare = ws::kTwinSpare * 8u, room = total <= half ? half - total : spare;  // (a row that has the unit to itself: plan_batch has seen to more than this)
    ab += room < spare ? room & ~uint64_t{15} : spare;
    uint64_t tabs_at = ab + map;
    total = tabs_at + tabs;
    if (total > half && map + list <= half) {
        const uint64_t low_ab = (half - map) & ~uint64_t{15}, counts = ws::kTwinBins * 4u;
        if (low_ab >= tabs + counts + 3u) {
            ab = low_ab;
            tabs_at = (ab - tabs) & ~uint64_t{3};
            total = ab + map;
        }
    }
    p.twin_ab = static_cast<uint32_t>(ab);
    p.twin_tabs = static_cast<uint32_t>(tabs_at);
    p.twin_total = static_cast<uint32_t>(total);
}

// few: whether ws_few.h is considered
BatchPlan plan_batch(const ws_batch* b, bool few = true) {
    BatchPlan p{};
    p.err = WS_E_INVALID;
    if (!b || !b->logits || !b->inv_t || !b->seed || !b->step || !b->token || !b->flags) return p;
    if (b->rows == 0 || b->vocab == 0 || b->vocab > 1048575u || b->row_stride < b->vocab) return p;
    if (b->dtype != WS_DTYPE_F32 && b->dtype != WS_DTYPE_BF16) return p;
    if (b->rng != WS_RNG_SPLITMIX && b->rng != WS_RNG_PHILOX) return p;
    if (b->hist && !b->hist_off) return p;
    if (b->bias_ids && (!b->bias_off || !b->bias_vals)) return p;
    if (b->kept_ids && b->kept_cap == 0) return p;
    if (b->mode != WS_MODE_AUTO && b->mode != WS_MODE_EXACT && b->mode != WS_MODE_FUSED) return p;
    const uint64_t cap = (b->hist ? uint64_t{b->max_hist} : 0) + (b->bias_ids ? uint64_t{b->max_bias} : 0);
    const uint32_t nW = (b->vocab + 31u) / 32u;
    const uint64_t maps = uint64_t{nW} * 4u + ((uint64_t{nW} * 2u + 15u) & ~uint64_t{15}) + ((cap * 4u + 15u) & ~uint64_t{15});
    p.err = WS_E_UNSUPPORTED;
    if (cap > 65535u) return p;
    // fused sweep: rows of whole 128-bit vectors that fit the register cache, and LDS room for the per-rank counters
    // next to the histogram (the exact path reuses the histogram's LDS for them)
    const uint64_t esz = b->dtype == WS_DTYPE_F32 ? 4 : 2;
    const bool vec_rows = b->vocab % 8u == 0 && (b->row_stride * esz) % 16u == 0 && reinterpret_cast<uintptr_t>(b->logits) % 16u == 0;
    const uint64_t fused_total = 65536u + maps + cap * 8u;
    // (a token's bias entries are counted in 11 bits of its rank word)
    const bool can_fuse = vec_rows && b->vocab <= 163840u && fused_total + kStaticLds <= kMaxLds && (!b->bias_ids || b->max_bias <= 2047u);
    if (b->mode == WS_MODE_FUSED && !can_fuse) return p;
    p.fused = b->mode != WS_MODE_EXACT && can_fuse;
    uint64_t ab, total;
    if (p.fused) {
        ab = 65536u;
        total = fused_total;
        p.lds_cnt = static_cast<uint32_t>(65536u + maps);
    } else {
        ab = cap * 8u > 65536u ? ((cap * 8u + 15u) & ~uint64_t{15}) : 65536u;
        total = ab + maps;
        p.lds_cnt = 0;
    }
    if (total + kStaticLds > kMaxLds) return p;  // history + bias too long for the LDS rank tables
    // spare room, when there is any, for a second copy of the histogram during the single sweep (odd lanes add there,
    // which halves the collisions of a wave's atomics on a crowded bin) and later for the tie bitmap of the sort
    // (vocab / 32 words + 16-bit prefixes)
    const uint64_t tie_bytes = uint64_t{nW} * 4u + ((uint64_t{nW} * 2u + 15u) & ~uint64_t{15});
    const uint64_t spare_bytes = tie_bytes > 32768u ? tie_bytes : 32768u;
    p.lds_tie = 0;
    if (total + spare_bytes + kStaticLds <= kMaxLds) {
        p.lds_tie = static_cast<uint32_t>((total + 15u) & ~uint64_t{15});
        total = p.lds_tie + spare_bytes;
    }
    p.patch_cap = static_cast<uint32_t>(cap ? cap : 1);
    p.lds_ab = static_cast<uint32_t>(ab);
    p.lds_total = static_cast<uint32_t>(total);
    // The lean kernel shares the single-sweep layout (its static LDS is larger, so the second histogram copy fits less
    // often); the three-pass code it hands rows back to lays its tables over the same allocation.
#ifdef WS_PHASE_TIMERS
    const bool wants_entropy = false;  // (debug builds: `entropy` takes the lean kernel's phase marks, 16 doubles a row)
#else
    const bool wants_entropy = b->entropy != nullptr;
#endif
    // Its rows are those without a top-k, and a batch says so by leaving `top_k` out: a row with one would be handed
    // back to the three-pass code inside the launch, at twice the time of the kernel that takes a top-k in its stride.
    // It reads rows at any address. Rows that are not whole aligned vectors, which the other single-sweep kernels do not take, are swept three times otherwise, and short ones are. The
    // lines below were drawn when the one build of this kernel asked for 163840 tokens of every row; since there are builds for short rows it would be the faster way from
    // some 8000 tokens on, and with lists from 2000. (us, three sweeps and this kernel, N(0, 2) and rows of raised tokens, top-p 0.9. The lines stand: which way rows of these
    // lengths go is held to the token by a test.)
    //   without lists, 1 row:    of 2051 15.6 / 16.2, 8195 16.5 / 16.4, 16387 17.9 / 16.7, 20011 19.3 / 17.0;  256 rows: of 2051 17.7 / 16.7, 8195 19.0 / 16.8, 16387 22.6 / 17.0, 20011 23.7 / 17.3
    //           masked, 1 row:   of 2051 16.5 / 18.0, 8195 17.7 / 18.1, 12001 18.6 / 18.0, 32003 22.6 / 18.0;  256 rows: of 6001 19.2 / 20.3, 8195 19.8 / 19.2, 32003 29.3 / 21.0
    //   16 and 64 ids, 1 row:    of 2051 19.4 / 17.9, 12001 21.5 / 18.2;  256 rows: of 2051 22.0 / 18.8, 12001 24.3 / 18.6
    //           masked, 1 row:   of 2051 20.1 / 20.0, 20011 24.9 / 20.1;  256 rows: of 4099 22.7 / 22.7, 6001 23.1 / 21.7, 20011 28.6 / 23.3
    //   500 ids, 1 row:          of 2051 21.7 / 17.9, 6001 22.3 / 18.1;  256 rows: of 2051 25.7 / 18.5, 6001 25.9 / 18.5;  masked: 256 rows of 2051 26.4 / 22.4, 20011 30.7 / 23.5
    //   longer rows (with the build of 163840): 1 row of 50257 28.7 / 22.0, with ids 38.7 / 24.5, of 151937 49.1 / 32.1; 256 rows of 50257 37.9 / 25.2, of 151937 67.1 / 40.0, with ids 77.9 / 42.8
    // Rows without a filter are none of its own either: of a batch that has neither top-p nor min-p it would hand back every one (three sweeps and this kernel: 1 row of
    // 50257 40 / 44, 256 rows 51 / 61, 256 of 151937 with 500 ids 117 / 125; the other single-sweep kernel and this one: 256 rows of 50256 52 / 61, of 151936 87 / 109).
    // Rows of 163841 to 262144 tokens, which no other single-sweep kernel takes, have their build of it with the longer bin cache (us, three sweeps and this; top-p 0.9):
    //   1 row of 262144 69 / 47, 64 of 200000 with 500 ids 84 / 53, 32 of 163841 65 / 42, 256 of 262144 with 2000 ids 128 / 93, 200 Zipfian of 262144 with 3000 135 / 93, 100 of
    //   200000 65 / 50; raised tokens: 16 of 256000 114 / 53, 256 of 163848 with 64 ids 83 / 67; masked: 88 of 248576, 17 % allowed, 94 / 58, 281 of 204976, 15 %, 150 / 119
    //   Rows whose cut no list holds are swept in vain, and go on to the exact path from there: 200 flat Zipfian rows of 262144, T up to 1.4, 845 / 675; 64 of 262144 in steps of 0.5 954 / 947.
    const uint32_t lean_least = vec_rows ? 8u : (cap >= (b->allow ? 512u : 128u) ? 8192u : (cap ? (b->allow ? 20480u : 16384u) : (b->allow ? 32768u : 20480u)));
    p.lean = (p.fused || !vec_rows || b->vocab > 163840u) && (b->top_p || b->min_p) && b->dtype == WS_DTYPE_F32 && b->mode == WS_MODE_AUTO && !b->top_k && !b->kept_ids && !b->query_prob && !wants_entropy && !b->race &&
             b->vocab >= lean_least && b->vocab <= 262144u && (!b->bias_ids || b->max_bias <= 2047u) && fused_total + kStaticLean <= kMaxLds;
    if (p.lean) {
        p.lds_ab = 65536u;
        p.lds_cnt = static_cast<uint32_t>(65536u + maps);
        uint64_t lt = fused_total;
        p.lean_tie = 0;
        if (lt + 32768u + kStaticLean <= kMaxLds) {
            p.lean_tie = static_cast<uint32_t>((lt + 15u) & ~uint64_t{15});
            lt = p.lean_tie + 32768u;
        }
        p.lean_total = static_cast<uint32_t>(lt);
        const uint64_t three = 65536u + maps;
        p.lean_fb_tie = three + spare_bytes <= lt ? static_cast<uint32_t>((three + 15u) & ~uint64_t{15}) : 0u;
    }
    // The short-list kernel: its own layout (32 KiB of list, the bitmap with 16-bit prefixes, a word and a 16-bit index
    // per history / bias entry), and under it room for the three-pass layout of the rows it hands back.
    const bool word_k = b->top_k && b->top_k_max >= 1u && b->top_k_max <= 1024u;  // every row with a top-k: at most top_k_max
    const bool word_p = b->min_p && b->min_p_min > 0.0;                            // every row without: a min-p
    p.shortlist = (b->top_k ? (word_k || word_p) : word_p) && (!b->top_k || b->top_k_max <= 1024u) && b->mode == WS_MODE_AUTO && b->vocab >= 8u && !b->race &&
                  (!b->bias_ids || b->max_bias <= 2047u);
    if (p.shortlist) {
        const uint64_t maps_s = uint64_t{nW} * 4u + ((uint64_t{nW} * 2u + 15u) & ~uint64_t{15});
        const uint64_t tabs_s = ((cap * 4u + 15u) & ~uint64_t{15}) + ((cap * 2u + 15u) & ~uint64_t{15});
        const uint64_t own = 32768u + maps_s + tabs_s;
        const uint64_t three = (cap * 8u > 65536u ? ((cap * 8u + 15u) & ~uint64_t{15}) : 65536u) + maps;
        uint64_t st = own > three ? own : three;
        if (st + kStaticShort > kMaxLds) {
            p.shortlist = false;
        } else {
            p.short_ab = 32768u;
            p.short_cnt = static_cast<uint32_t>(32768u + maps_s);
            p.short_fb_tie = 0;
            p.short_fb_ab = static_cast<uint32_t>(three - maps);
            if (three + spare_bytes + kStaticShort <= kMaxLds) {
                p.short_fb_tie = static_cast<uint32_t>((three + 15u) & ~uint64_t{15});
                if (p.short_fb_tie + spare_bytes > st) st = p.short_fb_tie + spare_bytes;
            }
            p.short_total = static_cast<uint32_t>(st);
            twin_plan(nW, cap, p);
        }
    }
    code_plan(b, cap, maps, spare_bytes, p);
    if (p.shortlist) {
        p.lean = false;
        p.split_log2 = 0;
        p.workspace = p.workspace_min = 0;
        if (few) few_plan(b, cap, maps, p);
        if (p.code) code_or_short(b, cap, p);
        if (!p.code && !p.few_parts && (p.split_log2 = short_split_log2(b)) != 0u) p.workspace = p.workspace_min = uint64_t{b->rows} * ws::kShortSplitRowBytes;
        p.twin = !p.code && !p.few_parts && !p.split_log2 && twin_rows(b);
        p.err = WS_OK;
        return p;
    }
    if (p.code) {
        p.split_log2 = 0;
        p.workspace = p.workspace_min = 0;
        p.err = WS_OK;
        return p;
    }
    // Small batches of the single-sweep kernel: with rows to spare on the compute units a row is split over 2, 4, 8 or
    // 16 workgroups (each at least 16384 tokens; 8192 for the step from 8 to 16, which a lone 151936-token row still wins: 29.2 -> 28.0 us), which meet in global memory. All parts of all rows have to be running
    // at the same time - they wait for each other - so rows * parts stays within the compute units of the device.
    p.split_log2 = 0;
    p.workspace = 0;
    if (p.fused && b->max_split != 1u) {
        const uint32_t cus = static_cast<uint32_t>(compute_units());
        const uint32_t most = b->max_split ? b->max_split : 16u;
        uint32_t lg = 0;
        while (lg < 4u && (2u << lg) <= most && b->rows * (2u << lg) <= cus && b->vocab / (2u << lg) >= (lg == 3u ? 8192u : 16384u)) ++lg;
        // Meeting in global memory costs two round trips of several thousand clocks each; measured on batches of
        // 151936-token rows, four parts and more win that back (64 rows: 49.5 against 52.9 us; 16 rows: 40 against 50),
        // two do not. A caller that names a number gets it.
        if (!b->max_split && lg < 2u) lg = 0;
        p.split_log2 = lg;
        // (with a kept-set dump the rows also get a staging area; a caller whose memory holds only the rows' meeting
        // places - the library's own, ws_sample_batch_static - goes without)
        if (lg) p.workspace_min = uint64_t{b->rows} * ws::kSplitRowBytes;
        if (lg) p.workspace = uint64_t{b->rows} * (b->kept_ids ? ws::kSplitRowBytesKept : ws::kSplitRowBytes);
    }
    // The kernels without a bin cache (long vocabularies, unaligned rows) take the touched tokens' raw logits from
    // their first sweep when they have somewhere to put them: 8 bytes per history / bias entry and row.
    if (!p.fused && !p.lean && cap > 0 && b->mode == WS_MODE_AUTO) p.workspace = uint64_t{b->rows} * ws::capture_row_bytes(p.patch_cap);
    p.err = WS_OK;
    return p;
}

// Memory of the library's own for ws_sample_batch_static: the split rows' meeting place (kStaticRows rows of it), in every
// GPU's copy of the code object, zero-filled when the code object is loaded and left zero-filled by every launch.
constexpr uint32_t kStaticRows = 64;
static __device__ __align__(256) unsigned char scratch[kStaticRows * ws::kSplitRowBytes];
std::atomic<unsigned char*> scratch_at[64];  // per device: where its copy of `scratch` lies

// the address of the current device's copy (asked for once per device; no allocation)
int scratch_address(unsigned char** out) {
    int dev = 0;
    if (const hipError_t e = hipGetDevice(&dev); e != hipSuccess) return static_cast<int>(e);
    if (dev < 0 || dev >= 64) return WS_E_UNSUPPORTED;
    unsigned char* at = scratch_at[dev].load(std::memory_order_acquire);
    if (!at) {
        void* sym = nullptr;
        if (const hipError_t e = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)); e != hipSuccess) return static_cast<int>(e);
        at = static_cast<unsigned char*>(sym);
        scratch_at[dev].store(at, std::memory_order_release);
    }
    *out = at;
    return WS_OK;
}

// workgroups a row of a greedy pick: within the compute units, at least 4096 tokens each (and byte offsets of 32 bits)
unsigned argmax_parts(int n, unsigned rows) {
    if (n >= (1 << 30) || rows == 0) return 0u;
    unsigned parts = static_cast<unsigned>(compute_units()) / rows;
    if (parts > 16u) parts = 16u;
    if (parts > static_cast<unsigned>(n) / 4096u) parts = static_cast<unsigned>(n) / 4096u;
    return parts < 2u ? 0u : parts;
}
bool argmax_workspace_ok(const void* w, uint64_t bytes, int n, unsigned rows) {
    return w && bytes >= ws_argmax_workspace(n, rows) && reinterpret_cast<uintptr_t>(w) % 8u == 0;
}
// another one for every launch of the process: the n-th output of the splitmix64 generator (a bijection of n), zero left out
unsigned long long launch_tag() {
    static std::atomic<uint64_t> launches{0};
    for (;;) {
        uint64_t z = (launches.fetch_add(1, std::memory_order_relaxed) + 1u) * 0x9E3779B97F4A7C15ull;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        if (z ^= z >> 31; z != 0) return z;
    }
}

// the kernels launched from this file whose dynamic LDS goes beyond the default limit
int prepare_three_pass() {
    static std::atomic<uint64_t> done{0};
    return ws::raise_lds_limit(done, {reinterpret_cast<const void*>(&ws::sample_batch_kernel<false>)}, kMaxLds - kStaticLds);
}
int prepare_adjust() {
    static std::atomic<uint64_t> done{0};
    return ws::raise_lds_limit(done, {reinterpret_cast<const void*>(&ws::adjust_rows_kernel)}, ws::kAdjustLds);
}
// everything a launch would otherwise set on its first call on this device: ws_probe does it ahead, outside any capture
int prepare_all() {
    if (const int e = prepare_three_pass(); e != 0) return e;
    if (const int e = prepare_adjust(); e != 0) return e;
    if (const int e = ws::prepare_fused(kMaxLds - kStaticLds); e != 0) return e;
    if (const int e = ws::prepare_split(kMaxLds - kStaticLds); e != 0) return e;
    if (const int e = ws::prepare_fused_kept(kMaxLds - kStaticLds); e != 0) return e;
    if (const int e = ws::prepare_split_kept(kMaxLds - kStaticLds); e != 0) return e;
    if (const int e = ws::prepare_lean(kMaxLds - kStaticLean); e != 0) return e;
    if (const int e = ws::prepare_code(kMaxLds - kStaticCode); e != 0) return e;
    if (const int e = ws::prepare_twin(kMaxLds - kStaticTwin); e != 0) return e;
    if (const int e = ws::prepare_few(kMaxLds - kStaticFew); e != 0) return e;
    if (const int e = ws::prepare_top(); e != 0) return e;
    return ws::prepare_short(kMaxLds - kStaticShort);
}

}  // namespace

extern "C" {

int ws_abi_version(void) { return WS_ABI_VERSION; }

const char* ws_error_string(int code) {
    switch (code) {
    case WS_OK: return "ok";
    case WS_E_INVALID: return "invalid argument";
    case WS_E_WORKSPACE: return "workspace missing or too small";
    case WS_E_STATIC_LIMIT: return "the batch would split more rows than the library's own workspace holds (64): use ws_sample_batch with a workspace, or max_split = 1";
    case WS_E_UNSUPPORTED: return "unsupported combination";
    case WS_E_NO_DEVICE: return "no usable HIP device";
    default: return code > 0 ? hipGetErrorString(static_cast<hipError_t>(code)) : "unknown error";
    }
}

int ws_probe(void) {
    static std::atomic<uint64_t> ready{0};  // devices this has succeeded on
    int n = 0, dev = -1;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 && (ready.load(std::memory_order_acquire) >> dev & 1u)) return WS_OK;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        return WS_E_NO_DEVICE;
    }
    hipFuncAttributes fa;
    if (hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(&argmax_rows)) != hipSuccess) {
        (void)hipGetLastError();
        return WS_E_NO_DEVICE;
    }
    unsigned char* at = nullptr;  // the current device's copy of the static workspace: resolved here, outside any capture
    if (const int e = scratch_address(&at); e != WS_OK) return e;
    if (const int e = prepare_all(); e != WS_OK) return e;
    if (dev >= 0 && dev < 64) ready.fetch_or(uint64_t{1} << dev, std::memory_order_release);
    return WS_OK;
}

uint64_t ws_argmax_workspace(int n, unsigned rows) { return n > 0 ? uint64_t{rows} * argmax_parts(n, rows) * 16u : 0ull; }

int ws_argmax(void* stream, const float* x, int n, int* out, int* ids, int* pos, int advance) {
    return ws_argmax_ws(stream, x, n, out, ids, pos, advance, nullptr, 0);
}

int ws_argmax_ws(void* stream, const float* x, int n, int* out, int* ids, int* pos, int advance, void* workspace, uint64_t workspace_bytes) {
    if (!x || !out || !ids || !pos || n <= 0) return WS_E_INVALID;
    if (const unsigned parts = argmax_parts(n, 1u); parts && argmax_workspace_ok(workspace, workspace_bytes, n, 1u))
        return ws::launch_argmax_shared(S(stream), 2, x, n, out, nullptr, ids, pos, advance, 1u, parts, static_cast<unsigned long long*>(workspace), launch_tag());
    hipLaunchKernelGGL(argmax, dim3(1), dim3(WS_BLOCK), 0, S(stream), x, n, out, ids, pos, advance);
    return done();
}

int ws_argmax_rows(void* stream, const float* x, int n, int* out, unsigned rows) { return ws_argmax_rows_ws(stream, x, n, out, rows, nullptr, 0); }

int ws_argmax_rows_ws(void* stream, const float* x, int n, int* out, unsigned rows, void* workspace, uint64_t workspace_bytes) {
    if (!x || !out || n <= 0 || rows == 0) return WS_E_INVALID;
    if (const unsigned parts = argmax_parts(n, rows); parts && argmax_workspace_ok(workspace, workspace_bytes, n, rows))
        return ws::launch_argmax_shared(S(stream), 0, x, n, out, nullptr, nullptr, nullptr, 0, rows, parts, static_cast<unsigned long long*>(workspace), launch_tag());
    hipLaunchKernelGGL(argmax_rows, dim3(rows), dim3(WS_BLOCK), 0, S(stream), x, n, out);
    return done();
}

int ws_argmax_rows_to(void* stream, const float* x, int n, int* out, const ws_row_idx* dst, unsigned rows) {
    return ws_argmax_rows_to_ws(stream, x, n, out, dst, rows, nullptr, 0);
}

int ws_argmax_rows_to_ws(void* stream, const float* x, int n, int* out, const ws_row_idx* dst, unsigned rows, void* workspace, uint64_t workspace_bytes) {
    if (!x || !out || !dst || n <= 0 || rows == 0 || rows > WS_MAX_TABLE_ROWS) return WS_E_INVALID;
    if (const unsigned parts = argmax_parts(n, rows); parts && argmax_workspace_ok(workspace, workspace_bytes, n, rows))
        return ws::launch_argmax_shared(S(stream), 1, x, n, out, dst, nullptr, nullptr, 0, rows, parts, static_cast<unsigned long long*>(workspace), launch_tag());
    RowIdx d;
    std::memcpy(&d, dst, sizeof d);
    hipLaunchKernelGGL(argmax_rows_to, dim3(rows), dim3(WS_BLOCK), 0, S(stream), x, n, out, d);
    return done();
}

int ws_argmax_prob(void* stream, const float* x, int n, int* out_tok, float* out_prob) {
    if (!x || !out_tok || !out_prob || n <= 0) return WS_E_INVALID;
    hipLaunchKernelGGL(argmax_prob, dim3(1), dim3(WS_BLOCK), 0, S(stream), x, n, out_tok, out_prob);
    return done();
}

int ws_argmax_prob_ws(void* stream, const float* x, int n, int* out_tok, float* out_prob, void* workspace, uint64_t workspace_bytes);

int ws_draft_pick(void* stream, const float* x, int n, int* tok, float* prob, int* ctl, int r, int n_min, float p_min,
                  const int* map) {
    if (!x || !tok || !prob || !ctl || n <= 0 || r < 0) return WS_E_INVALID;
    hipLaunchKernelGGL(draft_pick, dim3(1), dim3(WS_BLOCK), 0, S(stream), x, n, tok, prob, ctl, r, n_min, p_min, map);
    return done();
}

int ws_draft_pick_rows(void* stream, const float* x, int n, int* ctl_all, const ws_row_idx* area, int r, int n_min, float p_min,
                       const int* map, unsigned rows) {
    if (!x || !ctl_all || !area || n <= 0 || r < 0 || r >= 16 || rows == 0 || rows > WS_MAX_TABLE_ROWS) return WS_E_INVALID;
    RowIdx a;
    std::memcpy(&a, area, sizeof a);
    hipLaunchKernelGGL(draft_pick_rows, dim3(rows), dim3(WS_BLOCK), 0, S(stream), x, n, ctl_all, a, r, n_min, p_min, map);
    return done();
}

namespace {
// parts per row that pay for the greedy draft picks: the launch within the compute units, at least 16384 tokens a part
unsigned pick_split_log2(int n, unsigned rows) {
    const uint64_t cus = static_cast<uint64_t>(compute_units());
    unsigned lg = 0;
    while (lg < 4u && (static_cast<uint64_t>(rows) << (lg + 1u)) <= cus && (n >> (lg + 1u)) >= 16384) ++lg;
    return lg;
}
bool pick_workspace_ok(const void* w, uint64_t bytes, unsigned rows) {
    return w && bytes >= uint64_t{rows} * ws::kPickSplitRowBytes && reinterpret_cast<uintptr_t>(w) % 4u == 0;
}
}  // namespace

int ws_argmax_prob_ws(void* stream, const float* x, int n, int* out_tok, float* out_prob, void* workspace, uint64_t workspace_bytes) {
    if (!x || !out_tok || !out_prob || n <= 0) return WS_E_INVALID;
    const unsigned lg = pick_split_log2(n, 1u);
    if (!lg || !pick_workspace_ok(workspace, workspace_bytes, 1u)) return ws_argmax_prob(stream, x, n, out_tok, out_prob);
    hipLaunchKernelGGL(argmax_prob_split, dim3(1u << lg), dim3(WS_BLOCK), 0, S(stream), x, n, out_tok, out_prob, lg,
                       static_cast<unsigned*>(workspace));
    return done();
}

uint64_t ws_draft_pick_workspace(int n, unsigned rows) { return pick_split_log2(n, rows) ? uint64_t{rows} * ws::kPickSplitRowBytes : 0ull; }

int ws_draft_pick_ws(void* stream, const float* x, int n, int* tok, float* prob, int* ctl, int r, int n_min, float p_min,
                     const int* map, void* workspace, uint64_t workspace_bytes) {
    if (!x || !tok || !prob || !ctl || n <= 0 || r < 0) return WS_E_INVALID;
    const unsigned lg = pick_split_log2(n, 1u);
    if (!lg || !pick_workspace_ok(workspace, workspace_bytes, 1u)) return ws_draft_pick(stream, x, n, tok, prob, ctl, r, n_min, p_min, map);
    hipLaunchKernelGGL(draft_pick_split, dim3(1u << lg), dim3(WS_BLOCK), 0, S(stream), x, n, tok, prob, ctl, r, n_min, p_min, map, lg,
                       static_cast<unsigned*>(workspace));
    return done();
}

int ws_draft_pick_rows_ws(void* stream, const float* x, int n, int* ctl_all, const ws_row_idx* area, int r, int n_min, float p_min,
                          const int* map, unsigned rows, void* workspace, uint64_t workspace_bytes) {
    if (!x || !ctl_all || !area || n <= 0 || r < 0 || r >= 16 || rows == 0 || rows > WS_MAX_TABLE_ROWS) return WS_E_INVALID;
    const unsigned lg = pick_split_log2(n, rows);
    if (!lg || !pick_workspace_ok(workspace, workspace_bytes, rows))
        return ws_draft_pick_rows(stream, x, n, ctl_all, area, r, n_min, p_min, map, rows);
    RowIdx a;
    std::memcpy(&a, area, sizeof a);
    hipLaunchKernelGGL(draft_pick_rows_split, dim3(rows << lg), dim3(WS_BLOCK), 0, S(stream), x, n, ctl_all, a, r, n_min, p_min, map, lg,
                       static_cast<unsigned*>(workspace));
    return done();
}

int ws_draft_sample_rows(void* stream, const float* x, int n, int* ctl_all, const ws_row_idx* area, int r, const int* map,
                         const ws_dsamp_args* a, int* qbuf, unsigned rows) {
    if (!x || !ctl_all || !area || !a || !qbuf || n <= 0 || r < 0 || r >= 16 || rows == 0 || rows > WS_MAX_TABLE_ROWS)
        return WS_E_INVALID;
    RowIdx ar;
    DSampArgs da;
    static_assert(sizeof(DSampArgs) == sizeof(ws_dsamp_args) && sizeof(DSampArgs) == 1024, "DSampArgs layout");
    std::memcpy(&ar, area, sizeof ar);
    std::memcpy(&da, a, sizeof da);
    hipLaunchKernelGGL(draft_sample_rows, dim3(rows), dim3(WS_BLOCK), 0, S(stream), x, n, ctl_all, ar, r, map, da, qbuf);
    return done();
}

namespace {
unsigned shared_parts(int n, unsigned rows);
unsigned chunk_log2(const void* x, uint64_t row_bytes);
bool top_workspace_ok(const void* w, uint64_t bytes, unsigned rows);
}
// (a draft's row of any length and alignment is shared: with a workgroup a row and draw 7 rows of 24064 took 17 us, and take 9)
uint64_t ws_draft_sample_rows_workspace(int n, unsigned rows) { return shared_parts(n, rows) ? uint64_t{rows} * ws::kFewRowBytes : 0ull; }

int ws_draft_sample_rows_ws(void* stream, const float* x, int n, int* ctl_all, const ws_row_idx* area, int r, const int* map,
                            const ws_dsamp_args* a, int* qbuf, unsigned rows, void* workspace, uint64_t workspace_bytes) {
    if (!x || !ctl_all || !area || !a || !qbuf || n <= 0 || r < 0 || r >= 16 || rows == 0 || rows > WS_MAX_TABLE_ROWS)
        return WS_E_INVALID;
    const unsigned parts = shared_parts(n, rows);
    if (!parts || !top_workspace_ok(workspace, workspace_bytes, rows))
        return ws_draft_sample_rows(stream, x, n, ctl_all, area, r, map, a, qbuf, rows);
    return ws::launch_draft_shared(S(stream), x, n, ctl_all, area, r, map, a, qbuf, rows, parts, chunk_log2(x, uint64_t{4} * static_cast<unsigned>(n)),
                                   parts_together(parts, rows), static_cast<unsigned char*>(workspace));
}

int ws_topk_rows(void* stream, const float* x, int n, int K, float inv_t, int* ids, float* vals, float* stats, unsigned rows) {
    if (!x || !ids || !vals || !stats || n <= 0 || K <= 0 || rows == 0) return WS_E_INVALID;
    hipLaunchKernelGGL(topk_rows, dim3(rows), dim3(WS_BLOCK), 0, S(stream), x, n, K, inv_t, ids, vals, stats);
    return done();
}

namespace {
// workgroups a row of the kernels of ws_top.h (0: rows are not shared): shares that fit the registers of 512 threads and have 2048
// tokens at least, fewer rows than half the compute units
unsigned shared_parts(int n, unsigned rows) {
    if (n <= 0 || rows == 0) return 0u;
    const uint64_t cus = static_cast<uint64_t>(compute_units());
    const unsigned least = (static_cast<unsigned>(n) + ws::kFewShare - 1u) / ws::kFewShare;
    uint64_t parts = cus / rows;
    if (parts > ws::kFewMaxParts) parts = ws::kFewMaxParts;
    if (parts > static_cast<unsigned>(n) / 2048u) parts = static_cast<unsigned>(n) / 2048u;
    if (parts < least) parts = least;
    return parts < 2u || parts > ws::kFewMaxParts || rows * parts > 2u * cus || 2u * rows > cus ? 0u : static_cast<unsigned>(parts);
}
unsigned top_parts(int n, int K, unsigned rows) {
    if (n < 32768 || n % 4 != 0 || K <= 0 || K > 512) return 0u;  // (a short list, and the shapes the workspace functions have always named)
    return shared_parts(n, rows);
}
// chunks of eight lanes, a line of memory; where rows lie off the lines a chunk straddles two, and longer ones straddle fewer
unsigned chunk_log2(const void* x, uint64_t row_bytes) { return reinterpret_cast<uintptr_t>(x) % 16u == 0 && row_bytes % 16u == 0 ? 3u : 5u; }
bool top_workspace_ok(const void* w, uint64_t bytes, unsigned rows) {
    return w && bytes >= uint64_t{rows} * ws::kFewRowBytes && reinterpret_cast<uintptr_t>(w) % 8u == 0;
}
}  // namespace

uint64_t ws_topk_rows_workspace(int n, int K, unsigned rows) { return top_parts(n, K, rows) ? uint64_t{rows} * ws::kFewRowBytes : 0ull; }

int ws_topk_rows_ws(void* stream, const float* x, int n, int K, float inv_t, int* ids, float* vals, float* stats, unsigned rows,
                    void* workspace, uint64_t workspace_bytes) {
    if (!x || !ids || !vals || !stats || n <= 0 || K <= 0 || rows == 0) return WS_E_INVALID;
    const unsigned parts = top_parts(n, K, rows);
    if (!parts || !top_workspace_ok(workspace, workspace_bytes, rows)) return ws_topk_rows(stream, x, n, K, inv_t, ids, vals, stats, rows);
    return ws::launch_topk_shared(S(stream), x, n, K, inv_t, ids, vals, stats, rows, parts, chunk_log2(x, uint64_t{4} * static_cast<unsigned>(n)),
                                  parts_together(parts, rows), static_cast<unsigned char*>(workspace));
}

uint64_t ws_dflash_topk_workspace(int n, int ld, unsigned rows) {
    return ld >= n && ld % 4 == 0 && top_parts(n, 64, rows) ? uint64_t{rows} * ws::kFewRowBytes : 0ull;
}

int ws_dflash_topk_ws(void* stream, const float* x, int n, int ld, int k, int* ids, float* vals, unsigned rows, void* workspace,
                      uint64_t workspace_bytes) {
    if (!x || !ids || !vals || n <= 0 || ld < n || k <= 0 || k > 64 || rows == 0) return WS_E_INVALID;
    const unsigned parts = ld % 4 == 0 ? top_parts(n, k, rows) : 0u;
    if (!parts || !top_workspace_ok(workspace, workspace_bytes, rows)) return ws_dflash_topk(stream, x, n, ld, k, ids, vals, rows);
    return ws::launch_dflash_shared(S(stream), x, n, ld, k, ids, vals, rows, parts, chunk_log2(x, uint64_t{4} * static_cast<unsigned>(ld)),
                                    parts_together(parts, rows), static_cast<unsigned char*>(workspace));
}

int ws_dflash_topk(void* stream, const float* x, int n, int ld, int k, int* ids, float* vals, unsigned rows) {
    if (!x || !ids || !vals || n <= 0 || ld < n || k <= 0 || k > 64 || rows == 0) return WS_E_INVALID;
    hipLaunchKernelGGL(dflash_topk, dim3(rows), dim3(WS_BLOCK), 0, S(stream), x, n, ld, k, ids, vals);
    return done();
}

uint64_t ws_sample_batch_workspace(const ws_batch* b) {
    const BatchPlan p = plan_batch(b);
    return p.err == WS_OK ? p.workspace : 0;
}

int ws_sample_batch_workspace_use(const ws_batch* b) {
    const BatchPlan p = plan_batch(b);
    if (p.err != WS_OK || p.workspace == 0) return WS_WORK_NONE;
    return p.split_log2 || p.few_parts ? WS_WORK_MEETING : WS_WORK_TABLES;
}

namespace {

bool split_fits(const BatchPlan& p, const unsigned char* work, uint64_t work_bytes) {
    return p.workspace_min && work && work_bytes >= p.workspace_min && reinterpret_cast<uintptr_t>(work) % 8u == 0;
}

// the plan for a workspace of this size: rows of ws_few.h need twice the memory of the short-list kernel's own shared rows
BatchPlan plan_for(const ws_batch* b, uint64_t work_bytes) {
    const BatchPlan p = plan_batch(b);
    return p.err == WS_OK && p.few_parts && work_bytes < p.workspace_min ? plan_batch(b, false) : p;
}

// done: a word per row that gets `value` once the row's results are visible to the host, or nullptr (ws_sample_batch_notify)
int sample_batch_on(void* stream, const ws_batch* b, const BatchPlan& p, unsigned char* work, uint64_t work_bytes, uint32_t* done_at = nullptr,
                    uint32_t done_value = 0u, const ws::OwnRow* own = nullptr, bool leave = false) {
    const bool can_split = split_fits(p, work, work_bytes);
    const bool staged = can_split && work_bytes >= p.workspace && p.workspace > p.workspace_min;
    ws::BatchArgs a{};
    a.split_log2 = can_split ? p.split_log2 : 0u;
    a.split_row_bytes = staged ? ws::kSplitRowBytesKept : ws::kSplitRowBytes;
    a.stage_cap = staged ? ws::kSplitStageCap : 0u;
    a.work = (p.fused ? can_split : p.workspace && work && work_bytes >= p.workspace && reinterpret_cast<uintptr_t>(work) % 16u == 0) ? work : nullptr;
    a.split_spins = b->split_spins;
    a.logits = b->logits;
    a.dtype = b->dtype;
    a.rows = b->rows;
    a.vocab = b->vocab;
    a.row_stride = b->row_stride;
    a.inv_t = b->inv_t;
    a.top_k = b->top_k;
    a.top_p = b->top_p;
    a.min_p = b->min_p;
    a.seed = b->seed;
    a.step = b->step;
    a.rng = b->rng;
    a.hist = b->hist;
    a.hist_off = b->hist_off;
    a.rep = b->rep;
    a.pres = b->pres;
    a.freq = b->freq;
    a.bias_ids = b->bias_ids;
    a.bias_vals = b->bias_vals;
    a.bias_off = b->bias_off;
    a.patch_cap = p.patch_cap;
    a.allow = b->allow;
    a.allow_stride = b->allow_stride;
    a.token = b->token;
    a.prob = b->prob;
    a.n_kept = b->n_kept;
    a.flags = b->flags;
    a.stats = b->stats;
    a.margin = b->margin;
    a.kept_ids = b->kept_ids;
    a.kept_logits = b->kept_logits;
    a.kept_cap = b->kept_cap;
    a.tol = b->tol > 1e-6 ? b->tol : 1e-6;  // the histogram masses are good to ~5e-7 relative: no decision closer than that is trusted
    a.lds_ab = p.lds_ab;
    a.lds_cnt = p.lds_cnt;
    a.lds_tie = p.lds_tie;
    a.two_sweep = b->mode == WS_MODE_AUTO ? 1 : 0;
    a.race = b->race;
    a.hist_len = b->hist ? b->hist_len : nullptr;
    a.query = b->query;
    a.query_prob = b->query_prob;
    a.entropy = b->entropy;
    if (p.few_parts && can_split) {
        a.done = done_at;
        a.done_value = done_value;
        a.few_parts = p.few_parts;
        const uint32_t waves = p.few_parts * 8u;  // (512 threads a workgroup)
        a.few_magic = static_cast<uint32_t>(((uint64_t{1} << 32) + waves - 1u) / waves);
        a.few_chunk_log2 = chunk_log2(b->logits, b->row_stride * (b->dtype == WS_DTYPE_F32 ? 4u : 2u));
        a.few_together = parts_together(p.few_parts, b->rows);
        a.work = work;
        a.fb_lds_tie = 0u;
        a.fb_lds_ab = p.short_fb_ab;
        return ws::launch_few(S(stream), a, p.few_total, kMaxLds - kStaticFew, own, leave);
    }
    if (p.code) {
        a.lds_tie = p.code_copies > 1u;
        a.fb_lds_tie = p.code_fb_tie;
        a.fb_lds_ab = p.code_fb_ab;
        a.code_cap = p.code_cap;
        a.code_route = p.shortlist ? WS_FLAG_ROUTE_SHORT : (b->top_k ? 0u : WS_FLAG_ROUTE_LEAN);
        a.code_head = p.code_head;
        a.code_above = p.code_above;
        return ws::launch_code(S(stream), a, b->rows, p.code_total, kMaxLds - kStaticCode);
    }
    if (p.shortlist) {
        a.fb_lds_tie = p.short_fb_tie;
        a.fb_lds_ab = p.short_fb_ab;
        if (p.twin) {
            a.work = nullptr;
            a.lds_ab = p.twin_ab;
            a.lds_cnt = p.twin_tabs;
            if (const int e = ws::launch_twin(S(stream), a, p.twin_total, kMaxLds - kStaticTwin); e != 0) return e;
            return ws::launch_short_rest(S(stream), a, static_cast<uint32_t>(compute_units()), p.short_total, kMaxLds - kStaticShort);
        }
        a.lds_ab = p.short_ab;
        a.lds_cnt = p.short_cnt;
        a.work = a.split_log2 ? work : nullptr;
        return ws::launch_short(S(stream), a, p.short_total, kMaxLds - kStaticShort);
    }
    if (p.fused && a.split_log2)
        return (a.kept_ids ? ws::launch_split_kept : ws::launch_split)(S(stream), a, b->rows << a.split_log2, p.lds_total, kMaxLds - kStaticLds);
    if (p.lean) {
        a.lds_tie = p.lean_tie;
        a.fb_lds_tie = p.lean_fb_tie;
        a.fb_lds_ab = 65536u;
        return ws::launch_lean(S(stream), a, b->rows, p.lean_total, kMaxLds - kStaticLean);
    }
    if (p.fused) return (a.kept_ids ? ws::launch_fused_kept : ws::launch_fused)(S(stream), a, b->rows, p.lds_total, kMaxLds - kStaticLds);
    if (const int e = prepare_three_pass(); e != 0) return e;
    hipLaunchKernelGGL(ws::sample_batch_kernel<false>, dim3(b->rows), dim3(WS_BLOCK), p.lds_total, S(stream), a);
    return done();
}

}  // namespace

int ws_sample_batch(void* stream, const ws_batch* b) {
    const BatchPlan p = plan_for(b, b ? b->workspace_bytes : 0);
    if (p.err != WS_OK) return p.err;
    return sample_batch_on(stream, b, p, static_cast<unsigned char*>(b->workspace), b->workspace_bytes);
}

namespace {
// what load_row_params makes of the first row's parameters, read by the host
void own_row(const ws_batch* b, ws::OwnRow& o) {
    ws::LeanRowParams& P = o.P;
    P.inv_t = b->inv_t[0];
    P.top_k = b->top_k ? b->top_k[0] : 0u;
    P.race = b->race && b->race[0];
    P.top_p = b->top_p ? b->top_p[0] : 1.0;
    P.min_p = b->min_p ? b->min_p[0] : 0.0;
    P.h0 = b->hist ? b->hist_off[0] : 0u;
    P.nh = b->hist ? (b->hist_len ? b->hist_len[0] : b->hist_off[1] - P.h0) : 0u;
    P.b0 = b->bias_ids ? b->bias_off[0] : 0u;
    P.nb = b->bias_ids ? b->bias_off[1] - P.b0 : 0u;
    P.seed = b->seed[0];
    P.step = b->step[0];
    P.rep = b->rep ? b->rep[0] : 1.f;
    P.pres = b->pres ? b->pres[0] : 0.f;
    P.freq = b->freq ? b->freq[0] : 0.f;
    o.n_ids = P.nh <= ws::kOwnIds && P.nh <= b->max_hist ? P.nh : 0u;  // (a row with more than the batch declares: its ids are not read)
    if (o.n_ids) std::memcpy(o.ids, b->hist + P.h0, o.n_ids * sizeof(int32_t));
}

int notify_on(void* stream, const ws_batch* b, uint32_t* done, uint32_t value, bool host_inputs, bool leave = false) {
    if (!done) return WS_E_INVALID;
    const BatchPlan p = plan_for(b, b ? b->workspace_bytes : 0);
    if (p.err != WS_OK) return p.err;
    unsigned char* work = static_cast<unsigned char*>(b->workspace);
    const bool few = p.few_parts && split_fits(p, work, b->workspace_bytes), with_row = host_inputs && few && b->rows == 1u;
    ws::OwnRow own;
    if (with_row) own_row(b, own);
    if (const int e = sample_batch_on(stream, b, p, work, b->workspace_bytes, done, value, with_row ? &own : nullptr, leave); e != WS_OK) return e;
    if (few) return WS_OK;  // (that kernel writes the words itself)
    if (!b->rows) return WS_OK;
    for (uint32_t r = 0; r + 1u < b->rows; ++r) done[r] = value;
    return static_cast<int>(hipStreamWriteValue32(S(stream), done + b->rows - 1u, value, 0));
}
}  // namespace

int ws_sample_batch_notify(void* stream, const ws_batch* b, uint32_t* done, uint32_t value) { return notify_on(stream, b, done, value, false); }

int ws_sample_batch_notify_host(void* stream, const ws_batch* b, uint32_t* done, uint32_t value) { return notify_on(stream, b, done, value, true); }

int ws_sample_batch_try_host(void* stream, const ws_batch* b, uint32_t* done, uint32_t value) { return notify_on(stream, b, done, value, true, true); }

int ws_sample_batch_static(void* stream, const ws_batch* b) {
    const BatchPlan p = plan_for(b, sizeof(scratch));
    if (p.err != WS_OK) return p.err;
    if (p.code || (!p.fused && !p.shortlist)) return sample_batch_on(stream, b, p, nullptr, 0);  // (nothing may be left in the split rows' memory)
    if (p.workspace_min > sizeof(scratch)) {  // more split rows than the library's own memory holds
        if (p.shortlist && b->max_split == 0u) return sample_batch_on(stream, b, p, nullptr, 0);  // (split by the library's own choice: not here)
        return WS_E_STATIC_LIMIT;
    }
    unsigned char* at = nullptr;
    if (const int e = scratch_address(&at); e != WS_OK) return e;
    return sample_batch_on(stream, b, p, at, sizeof(scratch));
}

int ws_adjust_rows(void* stream, const ws_adjust* b) {
    if (!b || !b->logits || !b->out || b->rows == 0 || b->vocab == 0 || b->row_stride < b->vocab || b->out_stride < b->vocab)
        return WS_E_INVALID;
    if (b->dtype != WS_DTYPE_F32 && b->dtype != WS_DTYPE_BF16) return WS_E_INVALID;
    if ((b->hist && !b->hist_off) || (b->bias_ids && (!b->bias_off || !b->bias_vals))) return WS_E_INVALID;
    ws::AdjustArgs a{};
    a.logits = b->logits;
    a.dtype = b->dtype;
    a.vocab = b->vocab;
    a.row_stride = b->row_stride;
    a.hist = b->hist;
    a.hist_off = b->hist_off;
    a.rep = b->rep;
    a.pres = b->pres;
    a.freq = b->freq;
    a.bias_ids = b->bias_ids;
    a.bias_vals = b->bias_vals;
    a.bias_off = b->bias_off;
    a.allow = b->allow;
    a.allow_stride = b->allow_stride;
    a.out = b->out;
    a.out_stride = b->out_stride;
    a.lds_bytes = ws::kAdjustLds;
    if (const int e = prepare_adjust(); e != 0) return e;
    // a small batch shares a row between workgroups (slices of at least 8192 tokens, one workgroup per compute unit)
    uint32_t parts = 1;
    while (parts < 16u && static_cast<uint64_t>(b->rows) * (parts * 2u) <= compute_units() && b->vocab / (parts * 2u) >= 8192u) parts *= 2u;
    a.parts = parts;
    hipLaunchKernelGGL(ws::adjust_rows_kernel, dim3(b->rows * parts), dim3(WS_BLOCK), ws::kAdjustLds, S(stream), a);
    return done();
}

namespace {
ws::HistoryRef history_ref(const ws_history& h) { return ws::HistoryRef{h.tokens, h.len, h.n_gen, h.slot, h.cap}; }
bool history_ok(const ws_history& h) { return !h.tokens || (h.len && h.slot && h.cap >= 2u); }
}  // namespace

namespace {
int accept_sampled_on(void* stream, const ws_accept* b, bool fresh) {
    if (!b || !b->token || !b->flags || !b->row0 || !b->ctl_all || !b->area || !b->n_accepted || !b->chosen || !b->status)
        return WS_E_INVALID;
    if (b->n_seq == 0 || !history_ok(b->hist)) return WS_E_INVALID;
    if (b->typical && (!b->query_prob || !b->entropy)) return WS_E_INVALID;
    ws::AcceptArgs a{};
    a.token = b->token;
    a.flags = b->flags;
    a.row0 = b->row0;
    a.ctl_all = b->ctl_all;
    a.area = b->area;
    a.n_seq = b->n_seq;
    a.host_mask = WS_FLAG_ALL_MASKED | WS_FLAG_OVERFLOW | WS_FLAG_BAD_PARAM;
    a.n_accepted = b->n_accepted;
    a.chosen = b->chosen;
    a.status = b->status;
    a.query_prob = b->query_prob;
    a.entropy = b->entropy;
    a.typical = b->typical;
    a.eps = b->eps;
    a.delta = b->delta;
    a.approx_mask = WS_FLAG_APPROX_ENTROPY;
    a.relaxed = b->relaxed;
    a.hist = history_ref(b->hist);
    hipLaunchKernelGGL(fresh ? ws::accept_sampled_kernel<true> : ws::accept_sampled_kernel<false>, dim3(b->n_seq), dim3(64), 0, S(stream), a);
    return done();
}
}  // namespace

int ws_accept_sampled(void* stream, const ws_accept* b) { return accept_sampled_on(stream, b, false); }

int ws_accept_sampled_fresh(void* stream, const ws_accept* b) { return accept_sampled_on(stream, b, true); }

int ws_accept_greedy(void* stream, const ws_accept_greedy_args* b) {
    if (!b || !b->ctl_all || !b->area || !b->row0 || !b->n_accepted || !b->chosen || !b->status || b->n_seq == 0) return WS_E_INVALID;
    if (!history_ok(b->hist)) return WS_E_INVALID;
    if (b->relax && (!b->relax_ids || !b->relax_vals || !b->relax_stats || b->k == 0 || b->relax_k == 0)) return WS_E_INVALID;
    ws::AcceptGreedyArgs a{};
    a.ctl_all = b->ctl_all;
    a.area = b->area;
    a.row0 = b->row0;
    a.n_seq = b->n_seq;
    a.relax = b->relax;
    a.relax_ids = b->relax_ids;
    a.relax_vals = b->relax_vals;
    a.relax_stats = b->relax_stats;
    a.k = b->k;
    a.relax_k = b->relax_k;
    a.alpha = b->alpha;
    a.n_accepted = b->n_accepted;
    a.chosen = b->chosen;
    a.status = b->status;
    a.relaxed = b->relaxed;
    a.relax_gap = b->relax_gap;
    a.hist = history_ref(b->hist);
    hipLaunchKernelGGL(ws::accept_greedy_kernel, dim3(b->n_seq), dim3(64), 0, S(stream), a);
    return done();
}

int ws_history_stage(void* stream, const ws_history_stage_args* b) {
    if (!b || !b->hist.tokens || !history_ok(b->hist) || !b->ctl_all || !b->area || !b->row0 || !b->hist_off || !b->hist_len || !b->status ||
        b->n_seq == 0)
        return WS_E_INVALID;
    if (b->step && !b->hist.n_gen) return WS_E_INVALID;
    ws::StageArgs a{};
    a.hist = history_ref(b->hist);
    a.ctl_all = b->ctl_all;
    a.area = b->area;
    a.row0 = b->row0;
    a.n_seq = b->n_seq;
    a.hist_off = b->hist_off;
    a.hist_len = b->hist_len;
    a.query = b->query;
    a.step = b->step;
    a.status = b->status;
    hipLaunchKernelGGL(ws::history_stage_kernel, dim3((b->n_seq + ws::kStageSeqs - 1u) / ws::kStageSeqs), dim3(64), 0, S(stream), a);
    return done();
}

uint64_t ws_spec_verify_workspace(const ws_spec_verify* v) { return ws::spec_workspace(v, compute_units()); }

int ws_spec_verify_classic(void* stream, const ws_spec_verify* v) { return ws::spec_launch(S(stream), v, compute_units()); }

}  // extern "C"
