// The short-list sampler (ws_short.h), a translation unit of its own: 1024 threads per workgroup; fp32 and bf16 rows,
// with and without an allow mask, a workgroup's own or shared by several; the three-pass code of ws_sample.h as a function for the rows it hands back.
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
}  // namespace

int prepare_short(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[8];
    for (int k = 0; k < 8; ++k) all[k] = reinterpret_cast<const void*>(kShortKernels[k / 4][k / 2 % 2][k % 2]);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_short(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_short(lds_limit); e != 0) return e;
    hipLaunchKernelGGL(kShortKernels[a.dtype][a.allow ? 1 : 0][a.split_log2 ? 1 : 0], dim3(a.rows << a.split_log2), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
