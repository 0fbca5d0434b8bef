// The lean single-sweep sampler (ws_lean.h) for rows of up to 131072 tokens: see ws_lean.hip.
#define WS_BLOCK 1024
#include "ws_lean_table.h"

namespace ws {

typedef LeanBuilds<kLeanRegsShort, std::size(kLeanRegsShort)> Builds;

int prepare_lean_short(unsigned lds_limit) { return Builds::prepare(lds_limit); }

int launch_lean_short(hipStream_t stream, const BatchArgs& a, unsigned rows, unsigned lds_bytes, unsigned lds_limit) { return Builds::launch(stream, a, rows, lds_bytes, lds_limit); }

}  // namespace ws
