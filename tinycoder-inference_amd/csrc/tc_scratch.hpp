// tc_scratch.hpp -- growth rule of the library's device buffers. Host code
// with no HIP in it: `Mem` has void *alloc(size_t) (null on failure) and
// void release(void *) (after the work that may still use it has finished).
#pragma once

#include <stddef.h>

namespace tc {

// A grow-only buffer. `held`: a call recorded into a graph uses its address,
// which the graph's replays go on using.
struct Scratch {
    void *p = nullptr;
    size_t bytes = 0;
    bool held = false;
};

// Makes s hold `need` bytes for a call; `recording`: the call is being
// recorded into a graph.
//  * A held buffer is never released: it is left to its graphs, and the new one
//    is twice its size where that much is free, so that the buffers left behind
//    add up to less than the one in use.
//  * The new buffer is allocated before the old one is released, so a failure
//    leaves s as it was. Only where the call cannot do without (`must`) and
//    no graph uses the old buffer is that one released first to make room.
template <class Mem>
bool scratch_grow(Scratch &s, size_t need, bool recording, bool must, Mem &&mem) {
    if (s.bytes < need) {
        // (nothing may be released while work is being recorded)
        const bool keep = s.p != nullptr && (s.held || recording);
        size_t size = need;
        void *p = nullptr;
        if (keep && need < 2 * s.bytes) p = mem.alloc(size = 2 * s.bytes);
        if (p == nullptr) p = mem.alloc(size = need);
        if (p == nullptr && must && !keep && s.p != nullptr) {
            mem.release(s.p);
            s = Scratch{};
            p = mem.alloc(need);
        }
        if (p == nullptr) return false;
        if (s.p != nullptr && !keep) mem.release(s.p);
        s = Scratch{p, size, false};
    }
    s.held = s.held || (recording && need != 0);
    return true;
}

}  // namespace tc
