// The lean kernel's builds of one translation unit (ws_lean.h): by registers of the bin cache, with and without an allow mask.
#pragma once
#include <array>
#include <iterator>
#include <utility>

#include "ws_lds_limit.h"
#include "ws_lean.h"

namespace ws {

using LeanKernel = void (*)(BatchArgs);

template <const int* REGS, int... K>
std::array<std::array<LeanKernel, 2>, sizeof...(K)> lean_table(std::integer_sequence<int, K...>) {
    return {{{lean_batch_kernel<false, REGS[K]>, lean_batch_kernel<true, REGS[K]>}...}};
}

template <const int* REGS, int N>
struct LeanBuilds {
    static inline const auto kernels = lean_table<REGS>(std::make_integer_sequence<int, N>{});
    static int prepare(unsigned lds_limit) {
        static std::atomic<uint64_t> done{0};
        const void* all[2 * N];
        for (int k = 0; k < 2 * N; ++k) all[k] = reinterpret_cast<const void*>(kernels[k / 2][k % 2]);
        return raise_lds_limit_of(done, all, lds_limit);
    }
    static int launch(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) {
        if (const int e = prepare(lds_limit); e != 0) return e;
        int k = 0;  // the shortest cache that takes the row
        while (k + 1 < N && a.vocab > static_cast<uint32_t>(REGS[k]) * 4u * WS_BLOCK) ++k;
        hipLaunchKernelGGL(kernels[k][a.allow ? 1 : 0], dim3(rows), dim3(WS_BLOCK), lds_bytes, stream, a);
        return static_cast<int>(hipGetLastError());
    }
};

}  // namespace ws
