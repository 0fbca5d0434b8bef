// The lean single-sweep sampler (ws_lean.h), a translation unit of its own: with and without an allow mask, for rows of up to 32768, 49152, 65536, 98304,
// 155648, 163840 and 262144 tokens. 1024 threads per workgroup, 128 registers a thread, and the three-pass code of ws_sample.h as a function for the rows it hands back.
#define WS_BLOCK 1024
#include <array>
#include <iterator>
#include <utility>

#include "ws_lds_limit.h"
#include "ws_lean.h"

namespace ws {

namespace {
using LeanKernel = void (*)(BatchArgs);
constexpr int kBuilds = static_cast<int>(std::size(kLeanRegs));
// [registers of the bin cache][masked]
template <int... K>
std::array<std::array<LeanKernel, 2>, sizeof...(K)> lean_kernels(std::integer_sequence<int, K...>) {
    return {{{lean_batch_kernel<false, kLeanRegs[K]>, lean_batch_kernel<true, kLeanRegs[K]>}...}};
}
const auto kLeanKernels = lean_kernels(std::make_integer_sequence<int, kBuilds>{});
}  // namespace

int prepare_lean(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[2 * kBuilds];
    for (int k = 0; k < 2 * kBuilds; ++k) all[k] = reinterpret_cast<const void*>(kLeanKernels[k / 2][k % 2]);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_lean(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_lean(lds_limit); e != 0) return e;
    int k = 0;  // the shortest cache that takes the row
    while (k + 1 < kBuilds && a.vocab > static_cast<uint32_t>(kLeanRegs[k]) * 4u * WS_BLOCK) ++k;
    hipLaunchKernelGGL(kLeanKernels[k][a.allow ? 1 : 0], dim3(rows), dim3(WS_BLOCK), lds_bytes, stream, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
