"""The scratch arena's bookkeeping (undertow_amd/csrc/ut_arena.h) on the CPU,
over an allocator that records what it gave and what came back: a block that
a captured call named stays alive when the arena grows, and everything is
given back once."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "undertow_amd" / "csrc"

SRC = r"""
#include "ut_arena.h"
#include <cstdint>
#include <map>
struct Log { std::map<uintptr_t, size_t> live; uintptr_t next = 4096; size_t room = ~size_t(0); int bad = 0, waits = 0; };
struct Mem {
    Log *l;
    void *alloc(size_t n) {
        size_t used = 0;
        for (auto &b : l->live) used += b.second;
        if (used + n > l->room) return nullptr;
        const uintptr_t p = l->next;
        l->next += n + 4096;
        l->live[p] = n;
        return (void *)p;
    }
    bool wait() { l->waits++; return true; }
    bool free(void *p) { if (!l->live.erase((uintptr_t)p)) l->bad++; return true; }
};
struct S { ut::Arena a; Log l; };
extern "C" {
void *make(size_t room) { auto *s = new S; s->l.room = room; return s; }
int reserve(void *v, size_t n, int cap, int opt) { auto *s = (S *)v; return ut::arena_reserve(s->a, n, cap != 0, opt != 0, Mem{&s->l}); }
int waits(void *v) { return ((S *)v)->l.waits; }
void release(void *v) { auto *s = (S *)v; ut::arena_release(s->a, Mem{&s->l}); }
uintptr_t ptr(void *v) { return (uintptr_t)((S *)v)->a.ptr; }
size_t bytes(void *v) { return ((S *)v)->a.bytes; }
int alive(void *v, uintptr_t p) { return ((S *)v)->l.live.count(p); }
int count(void *v) { return (int)((S *)v)->l.live.size(); }
size_t total(void *v) { size_t n = 0; for (auto &b : ((S *)v)->l.live) n += b.second; return n; }
int bad(void *v) { return ((S *)v)->l.bad; }
}
"""


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    d = tmp_path_factory.mktemp("arena")
    (d / "a.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", str(CSRC), "-o",
                    str(d / "a.so"), str(d / "a.cpp")], check=True)
    lib = C.CDLL(str(d / "a.so"))
    lib.make.restype = C.c_void_p
    lib.make.argtypes = [C.c_size_t]
    for f, r, a in (("reserve", C.c_int, [C.c_void_p, C.c_size_t, C.c_int, C.c_int]), ("waits", C.c_int, [C.c_void_p]), ("release", None, [C.c_void_p]),
                    ("ptr", C.c_size_t, [C.c_void_p]), ("bytes", C.c_size_t, [C.c_void_p]),
                    ("alive", C.c_int, [C.c_void_p, C.c_size_t]), ("count", C.c_int, [C.c_void_p]),
                    ("total", C.c_size_t, [C.c_void_p]), ("bad", C.c_int, [C.c_void_p])):
        getattr(lib, f).restype, getattr(lib, f).argtypes = r, a
    return lib


MB = 1 << 20


def test_growth_keeps_what_a_graph_names(L):
    s = L.make(1 << 40)
    assert L.reserve(s, 4 * MB, 0, 0) == 0
    eager = L.ptr(s)
    assert L.reserve(s, 8 * MB, 0, 0) == 0 and not L.alive(s, eager)  # no graph: freed
    graph = L.ptr(s)
    assert L.reserve(s, 1 * MB, 1, 0) == 0 and L.ptr(s) == graph  # recorded by a capture
    assert L.reserve(s, 2 * MB, 0, 0) == 0  # eager calls of the same block change nothing
    for mb in (100, 300):
        assert L.reserve(s, mb * MB, 0, 0) == 0 and L.alive(s, graph)
    assert L.count(s) == 2  # the graph's and the newest: the one between was freed
    L.release(s)
    assert L.count(s) == 0 and L.bad(s) == 0


def test_kept_blocks_are_bounded(L):
    s = L.make(1 << 60)
    n = 1
    for _ in range(60):
        assert L.reserve(s, n, 1, 0) == 0
        n = L.bytes(s) + 1  # the smallest growth there is
    assert L.total(s) < 5 * L.bytes(s)
    L.release(s)
    assert L.count(s) == 0 and L.bad(s) == 0


def test_no_room(L):
    s = L.make(64 * MB)
    assert L.reserve(s, 20 * MB, 0, 0) == 0
    assert L.reserve(s, 200 * MB, 0, 0) == 1  # ARENA_OOM
    assert L.reserve(s, 20 * MB, 0, 0) == 0  # and the next call runs
    L.release(s)
    assert L.count(s) == 0 and L.bad(s) == 0


def test_optional_growth_without_room_changes_nothing(L):
    """The grouped experts have the four-row passes to fall back on: asking
    in vain must not wait, free or move what those passes use."""
    s = L.make(64 * MB)
    assert L.reserve(s, 20 * MB, 0, 0) == 0
    block, waits = L.ptr(s), L.waits(s)
    for _ in range(3):
        assert L.reserve(s, 200 * MB, 0, 1) == 1
        assert L.ptr(s) == block and L.alive(s, block) and L.waits(s) == waits
    assert L.reserve(s, 27 * MB, 0, 1) == 0 and L.ptr(s) != block and not L.alive(s, block)
    L.release(s)
    assert L.count(s) == 0 and L.bad(s) == 0
