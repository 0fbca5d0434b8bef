// The kernels of ws_top.h, a translation unit of its own: 512 threads per workgroup, shares of up to 20, 40 and 80 tokens a thread.
#define WS_BLOCK 512
#define WS_NO_NAMED_KERNELS
#include "ws_lds_limit.h"
#include "ws_top.h"

namespace ws {

namespace {
constexpr unsigned kTopLds = 65536u;  // the list and its sorted copy

struct Sizes {
    dim3 grid;
    TopSplit sp;
    int size;  // 0: 5 vectors a thread, 1: 10, 2: 20
};
Sizes sizes(int n, unsigned rows, unsigned parts, unsigned chunk_log2, unsigned together, unsigned char* work) {
    const unsigned vectors = (static_cast<unsigned>(n) + 3u) / 4u, load = 64u * WS_WAVES * parts, each = (vectors + load - 1u) / load;
    return {few_grid(parts, rows, together), TopSplit{parts, chunk_log2, rows, together, each, kFewKeys / (parts * WS_WAVES), work}, each <= 5u ? 0 : (each <= 10u ? 1 : 2)};
}
using TopkFn = void (*)(const float*, int, int, float, int*, float*, float*, TopSplit);
using DflashFn = void (*)(const float*, int, int, int, int*, float*, TopSplit);
using DraftFn = void (*)(const float*, int, int*, RowIdx, int, const int*, DSampArgs, int*, TopSplit);
const TopkFn kTopk[3] = {topk_rows_shared<5>, topk_rows_shared<10>, topk_rows_shared<20>};
const DflashFn kDflash[3] = {dflash_topk_shared<5>, dflash_topk_shared<10>, dflash_topk_shared<20>};
const DraftFn kDraft[3] = {draft_sample_rows_shared<5>, draft_sample_rows_shared<10>, draft_sample_rows_shared<20>};
}  // namespace

int prepare_top() {
    static std::atomic<uint64_t> done{0};
    const void* all[9];
    for (int k = 0; k < 3; ++k) {
        all[k] = reinterpret_cast<const void*>(kTopk[k]);
        all[3 + k] = reinterpret_cast<const void*>(kDflash[k]);
        all[6 + k] = reinterpret_cast<const void*>(kDraft[k]);
    }
    return raise_lds_limit_of(done, all, kTopLds);
}

int launch_topk_shared(hipStream_t stream, const float* x, int n, int K, float inv_t, int* ids, float* vals, float* stats, unsigned rows, unsigned parts,
                       unsigned chunk_log2, unsigned together, unsigned char* work) {
    if (const int e = prepare_top(); e != 0) return e;
    const Sizes z = sizes(n, rows, parts, chunk_log2, together, work);
    hipLaunchKernelGGL(kTopk[z.size], z.grid, dim3(WS_BLOCK), kTopLds, stream, x, n, K, inv_t, ids, vals, stats, z.sp);
    return static_cast<int>(hipGetLastError());
}

int launch_dflash_shared(hipStream_t stream, const float* x, int n, int ld, int k, int* ids, float* vals, unsigned rows, unsigned parts, unsigned chunk_log2, unsigned together,
                         unsigned char* work) {
    if (const int e = prepare_top(); e != 0) return e;
    const Sizes z = sizes(n, rows, parts, chunk_log2, together, work);
    hipLaunchKernelGGL(kDflash[z.size], z.grid, dim3(WS_BLOCK), kTopLds, stream, x, n, ld, k, ids, vals, z.sp);
    return static_cast<int>(hipGetLastError());
}

int launch_draft_shared(hipStream_t stream, const float* x, int n, int* ctl_all, const void* area, int r, const int* map, const void* args, int* qbuf,
                        unsigned rows, unsigned parts, unsigned chunk_log2, unsigned together, unsigned char* work) {
    if (const int e = prepare_top(); e != 0) return e;
    const Sizes z = sizes(n, rows, parts, chunk_log2, together, work);
    RowIdx ri;
    DSampArgs da;
    __builtin_memcpy(&ri, area, sizeof ri);
    __builtin_memcpy(&da, args, sizeof da);
    hipLaunchKernelGGL(kDraft[z.size], z.grid, dim3(WS_BLOCK), kTopLds, stream, x, n, ctl_all, ri, r, map, da, qbuf, z.sp);
    return static_cast<int>(hipGetLastError());
}

int launch_argmax_shared(hipStream_t stream, int mode, const float* x, int n, int* out, const void* dst, int* ids, int* pos, int advance, unsigned rows,
                         unsigned parts, unsigned long long* scratch, unsigned long long tag) {
    const PickArgs a{x, out, scratch, tag, static_cast<unsigned>(n), parts, ids, pos, advance};
    const dim3 grid(parts, rows);
    if (mode == 1) {
        PickArgsTo to{a, {}};
        __builtin_memcpy(&to.dst, dst, sizeof to.dst);
        hipLaunchKernelGGL(argmax_shared<1>, grid, dim3(WS_BLOCK), 0, stream, to);
    } else {
        hipLaunchKernelGGL(mode == 0 ? argmax_shared<0> : argmax_shared<2>, grid, dim3(WS_BLOCK), 0, stream, a);
    }
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
