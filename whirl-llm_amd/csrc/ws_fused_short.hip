// The fused-sweep instantiation of the batched sampler (ws_fused.hip) for short rows: the sweep is unrolled over the whole bin cache and asks for the vectors past
// a row's end like the others, so these have caches of 16384 to 131072 tokens. (us, the build of 163840 and these, rows with a top-k or without, of which the batch says nothing: 64 rows of 16000 with 200 ids 26.3 / 19.0, 1 of 32768
// 21.4 / 15.8, 5 of 31168 with 3410 ids 30.8 / 24.9, 256 of 50304 with 1000 36.5 / 28.3, 113 masked of 57408 47.9 / 42.7, 200 of 8000 with 300 ids and 100 bias entries 29.4 / 21.9.)
#define WS_BLOCK 512
#include "ws_lds_limit.h"
#include "ws_sample.h"

namespace ws {

namespace {
using Kernel = void (*)(BatchArgs);
constexpr int kBuilds = 5;
constexpr uint32_t kTokens[kBuilds] = {16384u, 32768u, 65536u, 98304u, kFusedShort};
const Kernel kKernels[kBuilds] = {sample_batch_kernel<true, false, false, kTokens[0]>, sample_batch_kernel<true, false, false, kTokens[1]>, sample_batch_kernel<true, false, false, kTokens[2]>,
                                  sample_batch_kernel<true, false, false, kTokens[3]>, sample_batch_kernel<true, false, false, kTokens[4]>};
}  // namespace

int prepare_fused_short(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[kBuilds];
    for (int k = 0; k < kBuilds; ++k) all[k] = reinterpret_cast<const void*>(kKernels[k]);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_fused_short(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_fused_short(lds_limit); e != 0) return e;
    int k = 0;
    while (k + 1 < kBuilds && a.vocab > kTokens[k]) ++k;
    hipLaunchKernelGGL(kKernels[k], dim3(rows), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
