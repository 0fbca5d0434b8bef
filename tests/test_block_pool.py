"""CPU: the pool of memory blocks the host layer's objects hand on to each other (host/block_pool.h), over a stand-in for the
runtime with two devices: a block comes back on the device it was made on, whichever is current when its owner lets go of it."""
import os
import subprocess

import wo

PROGRAM = r"""
#include "block_pool.h"
#include <cstdio>
#include <cstdlib>
#include <map>
#include <thread>

using whirl::sampling::Block;
using whirl::sampling::BlockMemory;
using whirl::sampling::BlockPool;

static int current = 0;
static std::mutex guard;
static std::map<void*, int> made;  // which device every live block was made on
static int device() { return current; }
static void* make(std::size_t bytes) {
    void* p = std::malloc(bytes);
    const std::lock_guard<std::mutex> lock(guard);
    made[p] = current;
    return p;
}
static void drop(void* p) {
    const std::lock_guard<std::mutex> lock(guard);
    if (!made.erase(p)) std::abort();
    std::free(p);
}
#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }

int main() {
    BlockPool pool(BlockMemory{device, make, drop});
    bool fresh = false;
    Block a = pool.take(1000, fresh);  // made on device 0, let go of while device 1 is current
    CHECK(fresh && a.dev == 0 && a.bytes == 1000);
    void* const first = a.at;
    current = 1;
    pool.give(a);
    CHECK(a.at == nullptr && a.bytes == 0);
    Block b = pool.take(1000, fresh);
    CHECK(fresh && b.at != first && b.dev == 1 && made[b.at] == 1);
    current = 0;
    Block c = pool.take(900, fresh);
    CHECK(!fresh && c.at == first && c.bytes == 1000 && made[c.at] == 0);
    pool.give(c);
    Block d = pool.take(200, fresh);  // (less than a quarter of what lies there: not wasted on it)
    CHECK(fresh && d.bytes == 200);
    pool.give(d);
    pool.give(b);
    pool.give(b);  // (empty: nothing)
    // bounded in number and in bytes
    std::vector<Block> many;
    for (int i = 0; i < 40; ++i) many.push_back(pool.take(100000, fresh));
    for (Block& m : many) pool.give(m);
    CHECK(made.size() == BlockPool::kMost);
    Block big = pool.take(BlockPool::kMostBytes + 1, fresh);
    pool.give(big);
    CHECK(made.size() == BlockPool::kMost);
    // several threads: nobody has a block that another one holds
    std::vector<std::thread> threads;
    for (int k = 0; k < 4; ++k)
        threads.emplace_back([&pool, k]() {
            for (int i = 0; i < 2000; ++i) {
                bool f;
                Block m = pool.take(100000, f);
                static_cast<volatile int*>(m.at)[0] = k;
                std::this_thread::yield();
                if (static_cast<volatile int*>(m.at)[0] != k) std::abort();
                pool.give(m);
            }
        });
    for (std::thread& t : threads) t.join();
    CHECK(made.size() <= BlockPool::kMost);
    std::puts("ok");
    return 0;
}
"""


def test_blocks_stay_with_the_device_they_were_made_on(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++20", "-O1", "-Wall", "-Wextra", "-pthread", "-I", os.path.join(wo.ROOT, "whirl-llm_amd", "host"),
                    "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout)
