// ut_arena.h -- the bookkeeping of a context's scratch arena: one block of
// device memory that grows on demand.  Host code only; `Mem` supplies
// alloc(bytes) (nullptr: none to be had), wait() (false: error) and
// free(ptr) (false: error).
#pragma once

#include <cstddef>
#include <vector>

namespace ut {

struct Arena {
    void *ptr = nullptr;
    size_t bytes = 0;
    // A call was recorded into a graph while this block was the arena: the
    // graph's nodes name its address, so the block outlives its replacement
    // and is given back with the context.  Every block is over 1.25 times the
    // one before, so all that are kept add up to less than four times the
    // newest.
    bool captured = false;
    std::vector<void *> kept;
};

enum ArenaStatus { ARENA_OK, ARENA_OOM, ARENA_ERROR };

// At least `total` bytes in a.ptr.  optional: for a caller that has another
// way without so much; the old block then stays until the new one is there,
// so that a call that gets none costs no wait and leaves the arena as it was.
template <typename Mem>
ArenaStatus arena_reserve(Arena &a, size_t total, bool capturing, bool optional, Mem &&mem) {
    if (total > a.bytes) {
        const size_t want = total + total / 4 + (1 << 20);
        void *early = optional ? mem.alloc(want) : nullptr;
        if (optional && !early) return ARENA_OOM;
        if (!mem.wait()) {
            if (early) (void)mem.free(early);
            return ARENA_ERROR;
        }
        if (a.ptr) {
            if (a.captured) a.kept.push_back(a.ptr);
            else if (!mem.free(a.ptr)) {
                if (early) (void)mem.free(early);
                return ARENA_ERROR;
            }
        }
        a.bytes = 0;
        a.captured = false;
        a.ptr = early ? early : mem.alloc(want);
        if (!a.ptr) return ARENA_OOM;
        a.bytes = want;
    }
    if (capturing) a.captured = true;
    return ARENA_OK;
}

template <typename Mem> void arena_release(Arena &a, Mem &&mem) {
    for (void *p : a.kept) (void)mem.free(p);
    if (a.ptr) (void)mem.free(a.ptr);
    a = Arena{};
}

}  // namespace ut
