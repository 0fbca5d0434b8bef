// The short-list sampler (ws_short.h), a translation unit of its own: 1024 threads per workgroup; fp32 and bf16 rows,
// with and without an allow mask, a workgroup's own or shared by several; the three-pass code of ws_sample.h as a function for the rows it hands back,
// and the kernel that runs it on those ws_twin.h has left.
#define WS_BLOCK 1024
#include "ws_lds_limit.h"
#include "ws_short.h"

namespace ws {

namespace {
// [dtype][masked][shared]
using ShortKernel = void (*)(BatchArgs);
const ShortKernel kShortKernels[2][2][2] = {{{short_batch_kernel<0, false, false>, short_batch_kernel<0, false, true>},
                                             {short_batch_kernel<0, true, false>, short_batch_kernel<0, true, true>}},
                                            {{short_batch_kernel<1, false, false>, short_batch_kernel<1, false, true>},
                                             {short_batch_kernel<1, true, false>, short_batch_kernel<1, true, true>}}};
// The rows that ws_twin.h has left to the three-pass code: launched behind it, with as many workgroups as compute units at most.
// (The flags of all of a workgroup's rows are read at once: one after the other they took 3 us of 1000 rows that all were done. The rows are a function's of their own: around
// its calls no register keeps the thread's number, and in the kernel that was a trip to scratch memory at its very start, 0.4 us of launches that had nothing to do.)
__device__ __noinline__ __attribute__((not_tail_called)) void short_rest(LeanArgPtr Ap_, const uint32_t n_) {
    LeanArgPtr Ap = wave_args(Ap_);
    const uint32_t n = __builtin_amdgcn_readfirstlane(n_);
    for (uint32_t row = blockIdx.x; row < Ap->rows; row += n) {
        const bool left = Ap->flags[row] == kTwinRest;
        __syncthreads();  // (every wave has read the word before one of them writes the row's flags there; and the row before is done with LDS)
        if (!left) continue;  // uniform
        if (Ap->kept_ids) three_pass_row<true>(Ap, row);
        else three_pass_row<false>(Ap, row);
    }
}
__global__ void __launch_bounds__(WS_BLOCK) short_rest_kernel(BatchArgs A) {
    const uint32_t n = gridDim.x, lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    bool any = false;
    for (uint32_t row = blockIdx.x + lane * n; row < A.rows; row += 64u * n) any |= A.flags[row] == kTwinRest;
    if (!__ballot(any)) return;  // (every wave asks for itself, and all get the same: the first flag is written behind a barrier)
    LeanArgPtr Ap = (LeanArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    short_rest(Ap, n);
}
}  // namespace

int prepare_short(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[9];
    for (int k = 0; k < 8; ++k) all[k] = reinterpret_cast<const void*>(kShortKernels[k / 4][k / 2 % 2][k % 2]);
    all[8] = reinterpret_cast<const void*>(short_rest_kernel);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_short(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_short(lds_limit); e != 0) return e;
    hipLaunchKernelGGL(kShortKernels[a.dtype][a.allow ? 1 : 0][a.split_log2 ? 1 : 0], dim3(a.rows << a.split_log2), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

int launch_short_rest(hipStream_t stream, const BatchArgs& a, unsigned blocks, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_short(lds_limit); e != 0) return e;
    hipLaunchKernelGGL(short_rest_kernel, dim3(blocks), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
