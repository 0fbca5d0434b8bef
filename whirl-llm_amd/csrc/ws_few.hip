// The sampler for few rows (ws_few.h), a translation unit of its own: 512 threads per workgroup (256 registers each); fp32 and bf16 rows, with
// and without an allow mask, shares of up to 20 (bf16: 24), 40, 80 and 112 tokens a thread; the three-pass code of ws_sample.h as a
// function for the rows it hands back.
#define WS_BLOCK 512
#include "ws_lds_limit.h"
#include "ws_few.h"

namespace ws {

namespace {
// [dtype][masked][size]: vectors a thread
using FewKernel = void (*)(BatchArgs);
constexpr uint32_t kFewVectors[2][4] = {{5u, 10u, 20u, 28u}, {3u, 5u, 10u, 14u}};
const FewKernel kFewKernels[2][2][4] = {
    {{few_batch_kernel<0, false, 5>, few_batch_kernel<0, false, 10>, few_batch_kernel<0, false, 20>, few_batch_kernel<0, false, 28>},
     {few_batch_kernel<0, true, 5>, few_batch_kernel<0, true, 10>, few_batch_kernel<0, true, 20>, few_batch_kernel<0, true, 28>}},
    {{few_batch_kernel<1, false, 3>, few_batch_kernel<1, false, 5>, few_batch_kernel<1, false, 10>, few_batch_kernel<1, false, 14>},
     {few_batch_kernel<1, true, 3>, few_batch_kernel<1, true, 5>, few_batch_kernel<1, true, 10>, few_batch_kernel<1, true, 14>}}};
// a lone row of up to 16 parts: fp32, unmasked; rows beyond 327680 tokens go the other way
constexpr int kOwnSizes = 2;
void (*const kOwnKernels[2][kOwnSizes])(BatchArgs, OwnRow) = {{few_own_kernel<0, 5>, few_own_kernel<0, 10>}, {few_try_kernel<0, 5>, few_try_kernel<0, 10>}};
}  // namespace

int prepare_few(unsigned lds_limit) {
    static std::atomic<uint64_t> done{0};
    const void* all[16 + 2 * kOwnSizes];
    for (int k = 0; k < 16; ++k) all[k] = reinterpret_cast<const void*>(kFewKernels[k / 8][k / 4 % 2][k % 4]);
    for (int k = 0; k < 2 * kOwnSizes; ++k) all[16 + k] = reinterpret_cast<const void*>(kOwnKernels[k / kOwnSizes][k % kOwnSizes]);
    return raise_lds_limit_of(done, all, lds_limit);
}

int launch_few(hipStream_t stream, const BatchArgs& a, unsigned lds_bytes, unsigned lds_limit, const OwnRow* own, bool leave) {
    if (const int e = prepare_few(lds_limit); e != 0) return e;
    const uint32_t per = a.dtype == 0 ? 4u : 8u, vectors = (a.vocab + per - 1u) / per, load = 64u * WS_WAVES * a.few_parts;
    const uint32_t each = (vectors + load - 1u) / load;
    BatchArgs b = a;
    b.few_vecs = each;
    b.few_slots = kFewKeys / (WS_WAVES * a.few_parts);
    int size = 0;
    while (size < 3 && each > kFewVectors[a.dtype][size]) ++size;
    if (own && a.rows == 1u && a.dtype == 0 && !a.allow && size < kOwnSizes)
        hipLaunchKernelGGL(kOwnKernels[leave ? 1 : 0][size], few_grid(a.few_parts, 1u, a.few_together), dim3(WS_BLOCK), lds_bytes, stream, b, *own);
    else
        hipLaunchKernelGGL(kFewKernels[a.dtype][a.allow ? 1 : 0][size], few_grid(a.few_parts, a.rows, a.few_together), dim3(WS_BLOCK), lds_bytes, stream, b);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ws
