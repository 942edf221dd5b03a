// Device workspaces of a handle that grow on demand (host code only; tests/host_layout_check.cpp
// drives it with a counting allocator).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace llmp {

enum class Alloc { ok, no_memory, failed };

// A buffer that grows to what its largest call needs, at least twofold, so that a cache filled
// call by call grows it a few times only; to exactly `need` where memory is short of that.
//
// The smaller buffer is freed first, behind the work on it, unless a captured graph may refer to
// it: then it goes to the handle's outgrown list, freed with the handle.  (Twofold growth bounds
// that list by the present buffer.)
struct Workspace {
    void* mem = nullptr;
    size_t bytes = 0;
    bool captured = false;          // some captured call uses `mem`
    size_t refused = SIZE_MAX;      // the smallest size try_grow found no memory for

    // Dev: Alloc alloc(size_t bytes, void** mem); void release(void* mem), which waits for the work
    // on it.  `capturing`: this call is being captured, so nothing can be waited for.
    template <class Dev>
    Alloc grow(size_t need, bool capturing, std::vector<void*>& outgrown, Dev& dev) {
        if (need > bytes) {
            const size_t twice = std::max(need, 2 * bytes);
            const bool keep = mem != nullptr && (captured || capturing);
            if (mem != nullptr && !keep) {
                dev.release(mem);
                mem = nullptr;
                bytes = 0;
            }
            void* grown = nullptr;
            size_t size = twice;
            Alloc r = dev.alloc(size, &grown);
            if (r == Alloc::no_memory && size > need) r = dev.alloc(size = need, &grown);
            if (r != Alloc::ok) return r;
            if (keep) outgrown.push_back(mem);
            mem = grown;
            bytes = size;
            captured = false;
        }
        if (capturing && need > 0) captured = true;
        return Alloc::ok;
    }
    // For a buffer that the caller can do without, outside capture: whether it holds `need` bytes
    // now.  A size that was refused is not asked for again.
    template <class Dev>
    bool try_grow(size_t need, std::vector<void*>& outgrown, Dev& dev) {
        if (need <= bytes) return true;
        if (need >= refused) return false;
        if (grow(need, false, outgrown, dev) == Alloc::ok) return true;
        refused = need;
        return false;
    }
};

}  // namespace llmp
