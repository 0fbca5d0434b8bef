"""CPU: what the host layer's DeviceRows asks of the C ABI, over a stand-in for it and for the runtime: a lone row goes through the quick entry point, one that comes
back undone is asked for again, and while a request's rows are of that kind each takes one launch."""
import os
import subprocess

import wo

PROGRAM = r"""
#include "sampling/device_rows.h"
#include "whirl_sampling_abi.h"
#include <hip/hip_runtime_api.h>
#include <cstdio>
#include <cstdlib>
#include <string>

using namespace whirl::sampling;

static std::string asked;       // t: the quick entry point, f: the full one
static bool hard = false;       // the row is one that the quick kernel leaves
extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
int ws_probe(void) { return 0; }
const char* ws_error_string(int) { return ""; }
uint64_t ws_sample_batch_workspace(const ws_batch*) { return 0; }
int ws_sample_batch_workspace_use(const ws_batch*) { return WS_WORK_NONE; }
int ws_adjust_rows(void*, const ws_adjust*) { return 0; }
int ws_topk_rows(void*, const float*, int, int, float, int*, float*, float*, unsigned) { return 0; }
static int answer(const ws_batch* b, uint32_t* done, uint32_t value, bool quick) {
    asked += quick ? 't' : 'f';
    for (uint32_t r = 0; r < b->rows; ++r) {
        if (quick && b->rows == 1 && hard) {
            b->flags[r] = WS_FLAGS_LEFT;
        } else {
            b->flags[r] = WS_FLAG_ROUTE_SHORT;
            if (hard) b->flags[r] = WS_FLAG_ROUTE_HANDED_BACK;
            b->token[r] = 7;
            b->n_kept[r] = 1;
            b->stats[2 * r] = 1.f;
            b->stats[2 * r + 1] = 1.f;
            b->kept_ids[r * b->kept_cap] = 7;
            b->kept_logits[r * b->kept_cap] = 1.f;
        }
        done[r] = value;
    }
    return 0;
}
int ws_sample_batch_try_host(void*, const ws_batch* b, uint32_t* done, uint32_t value) { return answer(b, done, value, true); }
int ws_sample_batch_notify_host(void*, const ws_batch* b, uint32_t* done, uint32_t value) { return answer(b, done, value, false); }
}

int main() {
    float logits[400] = {};
    std::vector<Cand> scratch(200);
    DeviceRows rows(logits, 2, 200);
    Sampler s;
    s.top_k = 5;
    s.cands = &scratch;
    auto step = [&](bool is_hard) {
        hard = is_hard;
        rows.newCycle();
        s.n = 0;
        rows.prepareRow(s, 0);
        if (s.n != 1 || scratch[0].id != 7 || rows.lastFlags() == WS_FLAGS_LEFT) std::puts("wrong answer");
        asked += ' ';
    };
    step(false), step(false), step(true), step(true), step(true), step(false), step(false);
    rows.prefetchRows(s, 0, 2);  // several rows are never left
    std::puts(asked.c_str());
    return 0;
}
"""


def test_a_row_the_quick_kernel_leaves_is_asked_for_again_once(tmp_path):
    host, include = os.path.join(wo.ROOT, "whirl-llm_amd", "host"), os.path.join(wo.ROOT, "include")
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(PROGRAM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++20", "-O1", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__", "-I", host, "-I", include, "-I", os.path.join(rocm, "include"),
                    "-o", str(exe), str(src), *(os.path.join(host, f) for f in ("device_rows.cpp", "sampler.cpp", "spec_sample.cpp"))], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "t t tf f f f t f", (r.returncode, r.stdout, r.stderr)
