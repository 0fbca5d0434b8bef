// The lean single-sweep sampler (ws_lean.h), a translation unit of its own (with and without an allow mask, for rows of up to 163840 and of up to 262144 tokens): 1024 threads per
// workgroup, 128 registers a thread, and the three-pass code of ws_sample.h as a function for the rows it hands back.
#define WS_BLOCK 1024
#include "ws_lds_limit.h"
#include "ws_lean.h"

namespace ws {

namespace {
// [rows that the longer bin cache takes][masked]
using LeanKernel = void (*)(BatchArgs);
const LeanKernel kLeanKernels[2][2] = {{lean_batch_kernel<false, kLeanRegs>, lean_batch_kernel<true, kLeanRegs>},
                                       {lean_batch_kernel<false, kLeanRegsLong>, lean_batch_kernel<true, kLeanRegsLong>}};
}  // namespace

int prepare_lean(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[4];
    for (int k = 0; k < 4; ++k) all[k] = reinterpret_cast<const void*>(kLeanKernels[k / 2][k % 2]);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_lean(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_lean(lds_limit); e != 0) return e;
    hipLaunchKernelGGL(kLeanKernels[a.vocab > kLeanRegs * 4u * WS_BLOCK ? 1 : 0][a.allow ? 1 : 0], dim3(rows), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
