// Device memory cut from slabs, for the private copies of quantized weights.
//
// A decode step reads every weight's tile copy and nothing else of the weights.
// One hipMalloc per copy spread them over the payloads and 6-bit copies made in
// between, and a step's reads over 2.5 times the addresses: 8B INT4 decode 3,046
// us over two steps before there were 6-bit copies, 3,061 with those between the
// tile copies, 3,036 with each kind in slabs of its own (1B: 1,109, 1,111, 1,106;
// single runs differ by 1%).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <map>
#include <vector>

namespace slhip {

class Arena {
  public:
    Arena() = default;
    Arena(const Arena&) = delete;
    Arena& operator=(const Arena&) = delete;
    ~Arena() { clear(); }

    // `bytes` of device memory at a multiple of kUnit, or null. Slabs grow with
    // what is held, so that a small model's are small.
    void* take(uint64_t bytes) {
        bytes = (std::max<uint64_t>(bytes, 1) + kUnit - 1) / kUnit * kUnit;
        for (Slab& s : slabs_)
            for (auto f = s.free.begin(); f != s.free.end(); ++f) {
                if (f->second < bytes) continue;
                const uint64_t at = f->first, left = f->second - bytes;
                s.free.erase(f);
                if (left) s.free[at + bytes] = left;
                return record(s, at, bytes);
            }
        uint64_t held = 0;
        for (const Slab& s : slabs_) held += s.size;
        Slab s;
        for (uint64_t size : {std::max(bytes, std::min(std::max(held, kFirst), kSlab)), bytes}) {
            if (hipMalloc(reinterpret_cast<void**>(&s.base), size) == hipSuccess) {
                s.size = size;
                break;
            }
            (void)hipGetLastError();
        }
        if (s.size == 0) return nullptr;
        if (s.size > bytes) s.free[bytes] = s.size - bytes;
        slabs_.push_back(std::move(s));
        return record(slabs_.back(), 0, bytes);
    }

    // Gives back what take returned (null: nothing), which no enqueued work may
    // still use; a slab's memory goes with its last piece.
    void give(void* p) {
        if (p == nullptr) return;
        uint8_t* const q = static_cast<uint8_t*>(p);
        for (size_t i = 0; i < slabs_.size(); ++i) {
            Slab& s = slabs_[i];
            if (q < s.base || q >= s.base + s.size) continue;
            uint64_t at = static_cast<uint64_t>(q - s.base), bytes = s.used[at];
            s.used.erase(at);
            if (s.used.empty()) {
                (void)hipFree(s.base);
                slabs_.erase(slabs_.begin() + static_cast<std::ptrdiff_t>(i));
                return;
            }
            const auto next = s.free.lower_bound(at);
            if (next != s.free.begin()) {
                const auto before = std::prev(next);
                if (before->first + before->second == at) {
                    at = before->first;
                    bytes += before->second;
                    s.free.erase(before);
                }
            }
            if (next != s.free.end() && at + bytes == next->first) {
                bytes += next->second;
                s.free.erase(next);
            }
            s.free[at] = bytes;
            return;
        }
    }

    bool empty() const { return slabs_.empty(); }
    void clear() {
        for (Slab& s : slabs_) (void)hipFree(s.base);
        slabs_.clear();
    }

  private:
    static constexpr uint64_t kUnit = 4096, kFirst = 64ull << 20, kSlab = 256ull << 20;
    struct Slab {
        uint8_t* base = nullptr;
        uint64_t size = 0;
        std::map<uint64_t, uint64_t> used, free;  // pieces, by offset: bytes
    };
    static void* record(Slab& s, uint64_t at, uint64_t bytes) {
        s.used[at] = bytes;
        return s.base + at;
    }
    std::vector<Slab> slabs_;
};

}  // namespace slhip
