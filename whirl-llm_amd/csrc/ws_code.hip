// The sampler for bf16 rows (ws_code.h), a translation unit of its own: with and without an allow mask, with and without touched
// tokens, for rows of up to 5, 10, 15 and 19 vectors a thread and for longer ones. 1024 threads per workgroup, 128 registers a thread, and the three-pass
// code of ws_sample.h as a function for the rows it hands back.
#define WS_BLOCK 1024
#include <vector>

#include "ws_lds_limit.h"
#include "ws_code.h"

namespace ws {

typedef void (*CodeKernel)(BatchArgs);
// by number: vectors a thread (5, 10, 15, 19), + 4 with touched tokens, + 8 with an allow mask
template <bool MASKED, bool TOUCHED>
static void add_kernels(std::vector<CodeKernel>& k) {
    k.insert(k.end(), {&code_batch_kernel<MASKED, TOUCHED, 5>, &code_batch_kernel<MASKED, TOUCHED, 10>, &code_batch_kernel<MASKED, TOUCHED, 15>, &code_batch_kernel<MASKED, TOUCHED, kCodeHeldVecs>});
}
static const std::vector<CodeKernel>& code_kernels() {
    static const std::vector<CodeKernel> all = [] {
        std::vector<CodeKernel> k;
        add_kernels<false, false>(k);
        add_kernels<false, true>(k);
        add_kernels<true, false>(k);
        add_kernels<true, true>(k);
        return k;
    }();
    return all;
}

int prepare_code(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    std::vector<const void*> kernels;
    for (CodeKernel k : code_kernels()) kernels.push_back(reinterpret_cast<const void*>(k));
    return raise_lds_limit_of(done, kernels, lds_limit);
}

int launch_code(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) {
    if (const int e = prepare_code(lds_limit); e != 0) return e;
    const uint32_t vecs = ((a.vocab + 7u) / 8u + WS_BLOCK - 1u) / WS_BLOCK;
    const uint32_t which = (vecs <= 5u ? 0u : (vecs <= 10u ? 1u : (vecs <= 15u ? 2u : 3u))) + (a.code_cap ? 4u : 0u) + (a.allow ? 8u : 0u);
    code_kernels()[which]<<<dim3(rows), dim3(WS_BLOCK), lds_bytes, stream>>>(a);
    return static_cast<int>(hipGetLastError());
}

uint64_t code_lds_bytes(uint32_t vocab, uint32_t cap, uint32_t copies) { return code_lds(vocab, cap, copies).total; }

}  // namespace ws
