// The lean single-sweep sampler (ws_lean.h) for rows of more than 131072 tokens, a translation unit of its own: 1024 threads per
// workgroup, 128 registers a thread, and the three-pass code of ws_sample.h as a function for the rows it hands back.
#define WS_BLOCK 1024
#include "ws_lean_table.h"

namespace ws {

typedef LeanBuilds<kLeanRegsLong, std::size(kLeanRegsLong)> Builds;

// ws_lean_short.hip
int prepare_lean_short(unsigned lds_limit);
int launch_lean_short(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit);

int prepare_lean(unsigned lds_limit) {
    if (const int e = prepare_lean_short(lds_limit); e != 0) return e;
    return Builds::prepare(lds_limit);
}

int launch_lean(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) {
    if (a.vocab <= static_cast<uint32_t>(*std::rbegin(kLeanRegsShort)) * 4u * WS_BLOCK) return launch_lean_short(stream, a, rows, lds_bytes, lds_limit);
    return Builds::launch(stream, a, rows, lds_bytes, lds_limit);
}

}  // namespace ws
