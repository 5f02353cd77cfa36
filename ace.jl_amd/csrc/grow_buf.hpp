// Grow-only buffer of device memory (no HIP here: the CPU test shim gives it
// another Memory).
#pragma once

#include <algorithm>
#include <cstddef>
#include <vector>

namespace acehost {

// ensure(n) makes room for n elements and frees the block it replaces.  A
// captured graph holds the pointers of the call it was captured from, and the
// room that a call needs goes up and down with the batch (its split), so a
// smaller batch may replace a block: the blocks that captured calls used
// (held) are kept until the buffer is destroyed.
template <typename T, typename Memory>
struct GrowBuf {
    T* p = nullptr;
    size_t n = 0;
    bool held = false;     // a captured call uses p
    std::vector<T*> kept;  // earlier blocks that captured calls use
    GrowBuf() = default;
    GrowBuf(const GrowBuf&) = delete;
    GrowBuf& operator=(const GrowBuf&) = delete;
    ~GrowBuf() {
        if (p) Memory::release(p);
        for (T* q : kept) Memory::release(q);
    }
    int ensure(size_t count) {
        if (count <= n) return 0;
        if (p) {
            if (held)
                kept.push_back(p);
            else
                Memory::release(p);
            p = nullptr;
            n = 0;
            held = false;
        }
        void* q = nullptr;
        if (Memory::alloc(&q, std::max<size_t>(count, 1) * sizeof(T))) return -1;
        p = static_cast<T*>(q);
        n = count;
        return 0;
    }
    // room for the calls of a graph if they are being captured
    int ensure(size_t count, bool capturing) {
        if (ensure(count)) return -1;
        held = held || capturing;
        return 0;
    }
    int upload(const T* h, size_t count) {
        if (ensure(count)) return -1;
        return count ? Memory::copy(p, h, count * sizeof(T)) : 0;
    }
};

}  // namespace acehost
