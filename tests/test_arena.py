"""The device-memory arena of the quantized weights' copies, on the CPU against
a hipMalloc of the host: pieces are disjoint and stay what was written to them,
memory given back is used again, a slab goes with its last piece, and a slab that
finds no room is cut down to the piece."""
import subprocess

import pytest

HIP = """
#pragma once
#include <cstdlib>
#include <cstdint>
#include <map>
enum hipError_t { hipSuccess, hipErrorOutOfMemory };
inline std::map<void*, uint64_t> live;
inline uint64_t in_use = 0, room = ~0ull;
inline hipError_t hipMalloc(void** p, uint64_t n) {
    if (n > room - in_use || !(*p = std::malloc(n))) return hipErrorOutOfMemory;
    live[*p] = n, in_use += n;
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    if (!live.count(p)) std::abort();
    in_use -= live[p], live.erase(p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
"""

MAIN = """
#include "arena.h"
#include <cstdio>
#include <random>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\\n", __LINE__, #x); return 1; } } while (0)
int main() {
    using slhip::Arena;
    std::mt19937_64 r(1);
    Arena a;
    std::map<uint8_t*, std::pair<uint64_t, uint8_t>> held;
    uint64_t sum = 0;
    const auto fill = [](uint8_t* p, uint64_t n, uint8_t v) { p[0] = p[n / 2] = p[n - 1] = v; };
    for (int i = 0; i < 20000; ++i) {
        if (held.size() < 40 && r() % 2) {
            const uint64_t n = 1 + r() % (r() % 4 ? 9000 : 3000000);
            uint8_t* p = static_cast<uint8_t*>(a.take(n));
            CHECK(p && reinterpret_cast<uintptr_t>(p) % 16 == 0);
            const auto next = held.lower_bound(p);
            CHECK(next == held.end() || p + n <= next->first);
            CHECK(next == held.begin() || std::prev(next)->first + std::prev(next)->second.first <= p);
            held[p] = {n, static_cast<uint8_t>(i)};
            fill(p, n, static_cast<uint8_t>(i));
            sum += n;
        } else if (!held.empty()) {
            auto it = std::next(held.begin(), r() % held.size());
            const uint64_t n = it->second.first;
            CHECK(it->first[0] == it->second.second && it->first[n / 2] == it->second.second &&
                  it->first[n - 1] == it->second.second);
            a.give(it->first);
            sum -= n;
            held.erase(it);
        }
        CHECK(held.empty() == a.empty());
        if (held.empty()) CHECK(in_use == 0);
    }
    for (auto& h : held) a.give(h.first);
    CHECK(a.empty() && in_use == 0);
    // the same piece over and over next to one that stays: no growth
    void* stay = a.take(1 << 20);
    a.give(a.take(3 << 20));
    const uint64_t once = in_use;
    for (int i = 0; i < 100; ++i) a.give(a.take((i % 3 + 1) << 20));
    CHECK(in_use <= once + (3ull << 20));
    a.give(stay);
    a.give(nullptr);
    CHECK(in_use == 0);
    // no room for a slab that grows with what is held, room for the piece
    void* big = a.take(80 << 20);
    room = in_use + (20 << 20);
    void* small = a.take(10 << 20);
    CHECK(small && !a.take(11 << 20) && in_use == 90ull << 20);
    a.give(big);
    a.give(small);
    CHECK(in_use == 0);
    {
        Arena b;
        CHECK(b.take(100));
    }
    CHECK(in_use == 0);
    return 0;
}
"""


@pytest.mark.parametrize("flags", [["-O1"], ["-O1", "-g", "-fsanitize=address,undefined"]])
def test_arena(tmp_path, flags):
    from conftest import ROOT

    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-Wall", *flags, f"-I{tmp_path}", f"-I{ROOT}/starlight_amd/csrc",
                    str(tmp_path / "main.cpp"), "-o", exe], check=True)
    done = subprocess.run([exe], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout + done.stderr
