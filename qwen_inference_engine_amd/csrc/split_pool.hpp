// split_pool.hpp — the split-K memory of one stream: slabs of partial tiles and the tiles' tickets (host only, no HIP).
//
// Both grow on demand and never shrink.  A launch recorded in a graph keeps the addresses that it was given, and only the
// graph's owner knows how long: once a capture has seen them they are not freed when something larger replaces them, but
// set aside until the stream itself goes (release).  What is set aside stays below what is in use, because held memory is
// replaced by at least twice its size.
#pragma once

#include <algorithm>
#include <cstddef>
#include <vector>

namespace qie {

struct SplitPool {
    float* slab = nullptr;
    unsigned* cnt = nullptr;       // zero at rest
    size_t slab_bytes = 0, cnt_n = 0;
    bool held = false;             // a capture has seen slab and cnt
    std::vector<void*> aside;      // what earlier captures have seen

    bool fits(size_t bytes, size_t tiles) const { return bytes <= slab_bytes && tiles <= cnt_n; }

    // Makes room (no launch that uses the memory may be running: the caller has waited).  alloc(bytes): nullptr when there is
    // none.  false: no memory, and none held by the pool.
    template <typename Alloc, typename Free>
    bool grow(size_t bytes, size_t tiles, Alloc alloc, Free release_one) {
        size_t sb = std::max(bytes, slab_bytes), cn = std::max(tiles, cnt_n);
        for (void* p : {(void*)slab, (void*)cnt}) {
            if (!p) continue;
            if (held) aside.push_back(p);
            else release_one(p);
        }
        if (held) {
            sb = std::max(sb, 2 * slab_bytes);
            cn = std::max(cn, 2 * cnt_n);
        }
        slab = nullptr;
        cnt = nullptr;
        slab_bytes = cnt_n = 0;
        held = false;
        float* s = (float*)alloc(sb);
        unsigned* c = s ? (unsigned*)alloc(cn * sizeof(unsigned)) : nullptr;
        if (!c) {
            if (s) release_one(s);
            return false;
        }
        slab = s;
        cnt = c;
        slab_bytes = sb;
        cnt_n = cn;
        return true;
    }

    // everything back (the stream has drained and nothing recorded on it is launched any more)
    template <typename Free>
    void release(Free release_one) {
        aside.push_back(slab);
        aside.push_back(cnt);
        for (void* p : aside)
            if (p) release_one(p);
        *this = SplitPool{};
    }
};

}  // namespace qie
