// The short-list sampler for rows that are not shared (ws_twin.h), a translation unit of its own: 512 threads per workgroup.
#define WS_BLOCK 512
#include "ws_lds_limit.h"
#include "ws_twin.h"

namespace ws {

namespace {
// [dtype][masked]
using TwinKernel = void (*)(BatchArgs);
const TwinKernel kTwinKernels[2][2] = {{twin_batch_kernel<0, false>, twin_batch_kernel<0, true>}, {twin_batch_kernel<1, false>, twin_batch_kernel<1, true>}};
}  // namespace

int prepare_twin(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[4];
    for (int k = 0; k < 4; ++k) all[k] = reinterpret_cast<const void*>(kTwinKernels[k / 2][k % 2]);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_twin(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_twin(lds_limit); e != 0) return e;
    hipLaunchKernelGGL(kTwinKernels[a.dtype][a.allow ? 1 : 0], dim3(a.rows), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
