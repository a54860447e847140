"""The work pool (polymer_amd/csrc/work_pool.h) over a stand-in for the
device's allocator: two devices of a few megabytes whose allocations fail where
their memory ends, as a device's do.  The header is compiled with g++; no GPU."""
import ctypes
import glob
import os
import re
import subprocess

import pytest

from tests.conftest import ROOT

SHIM = r"""
#include <cstdlib>
#include <map>
#include "work_pool.h"
struct Fake {
    static int current;
    static size_t total_[2], in_use[2];
    static std::map<void*, std::pair<size_t, int>> blocks;
    static int device() { return current; }
    static int alloc(void** p, size_t n) {
        if (in_use[current] + n > total_[current]) return 2;
        *p = std::malloc(16);
        in_use[current] += n;
        blocks[*p] = {n, current};
        return 0;
    }
    static void free(void* p) {
        in_use[blocks[p].second] -= blocks[p].first;
        blocks.erase(p);
        std::free(p);
    }
    static size_t total(int d) { return total_[d]; }
};
int Fake::current = 0;
size_t Fake::total_[2], Fake::in_use[2];
std::map<void*, std::pair<size_t, int>> Fake::blocks;
static polyeri::WorkPool<Fake>* pool;
extern "C" {
void start(size_t t0, size_t t1) {
    Fake::current = 0;
    Fake::total_[0] = t0; Fake::total_[1] = t1;
    Fake::in_use[0] = Fake::in_use[1] = 0;
    Fake::blocks.clear();
    pool = new polyeri::WorkPool<Fake>;
    pool->context(0, 1);
    pool->context(1, 1);
}
void set_device(int d) { Fake::current = d; }
size_t in_use(int d) { return Fake::in_use[d]; }
size_t idle(int d) { return pool->idle_bytes(d); }
void* get(size_t n) { void* p = nullptr; return pool->get(&p, n) ? nullptr : p; }
void put(void* p) { pool->put(p); }
void* raw(size_t n) { void* p = nullptr; return pool->alloc(&p, n) ? nullptr : p; }
size_t size_of(void* p) { return Fake::blocks[p].first; }
size_t release(int d) { return pool->release(d); }
void context(int d, int step) { pool->context(d, step); }
}
"""
MB = 1 << 20


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    src, so = str(d / "shim.cpp"), str(d / "shim.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror",
                           "-I", os.path.join(ROOT, "polymer_amd", "csrc"), src, "-o", so])
    L = ctypes.CDLL(so)
    p, n, i = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int
    for name, res, args in [("start", None, [n, n]), ("set_device", None, [i]), ("in_use", n, [i]), ("idle", n, [i]),
                            ("get", p, [n]), ("put", None, [p]), ("raw", p, [n]), ("size_of", n, [p]),
                            ("context", None, [i, i]), ("release", n, [i])]:
        getattr(L, name).restype, getattr(L, name).argtypes = res, args
    return L


@pytest.mark.parametrize("bytes_", [8, 4096, 300_000, MB, 5 * MB, 40 * MB, 1000 * MB])
def test_block_is_hardly_larger_than_its_request(shim, bytes_):
    """A used block's excess is charged to nobody: at most 1 MB, and for small
    requests 64 KB more than the request again."""
    for other in (bytes_, bytes_ + 7, bytes_ + 65536, bytes_ * 9 // 8, 2 * bytes_, 2 * bytes_ + 65536,
                  2 * bytes_ + 65537, bytes_ + MB, bytes_ + MB + 1):
        shim.start(1 << 40, 1 << 40)
        shim.put(shim.get(other))
        p = shim.get(bytes_)
        assert bytes_ <= shim.size_of(p) <= bytes_ + min(MB, bytes_ + 65536)
        if other == bytes_:
            assert shim.in_use(0) == bytes_        # the kept block itself


def test_calls_of_two_sizes_near_the_memorys_end(shim):
    """A call that needs nearly all of the device right after one of twice the
    block sizes: the oversized blocks may not be what it runs out on."""
    shim.start(1000 * MB, MB)
    first = [shim.get(60 * MB) for _ in range(4)]
    for p in first:
        shim.put(p)
    assert shim.idle(0) == 240 * MB
    held = [shim.get(31 * MB) for _ in range(32)]          # 992 of 1000 MB
    assert all(held) and shim.in_use(0) == 992 * MB


def test_bound_of_the_blocks_own_device(shim):
    """A block of a large device given back while a small one is current, and
    the other way round."""
    shim.start(1000 * MB, 100 * MB)
    p = shim.get(50 * MB)
    shim.set_device(1)
    q = shim.get(50 * MB)
    shim.put(p)
    assert shim.idle(0) == 50 * MB
    shim.set_device(0)
    shim.put(q)
    assert shim.idle(1) == 0 and shim.in_use(1) == 0       # more than its device may keep idle


def test_blocks_stay_on_their_device_and_end_with_its_contexts(shim):
    shim.start(1000 * MB, 1000 * MB)
    p = shim.get(10 * MB)
    shim.put(p)
    shim.set_device(1)
    q = shim.get(10 * MB)
    assert q != p and shim.idle(0) == 10 * MB
    shim.put(q)
    shim.context(0, -1)
    assert shim.in_use(0) == 0 and shim.idle(1) == 10 * MB
    shim.context(1, -1)
    assert shim.in_use(1) == 0


def test_failed_allocation_reclaims_idle_blocks(shim):
    """Of the pool's own requests and of others', and only of that device."""
    for request in (shim.get, shim.raw):
        shim.start(100 * MB, 100 * MB)
        shim.put(shim.get(10 * MB))
        assert shim.idle(0) == 10 * MB
        shim.set_device(1)
        shim.put(shim.get(10 * MB))
        shim.set_device(0)
        assert request(95 * MB)
        assert shim.idle(0) == 0 and shim.idle(1) == 10 * MB
        assert not request(6 * MB)                          # really full


def test_release_gives_back_one_devices_idle_blocks(shim):
    shim.start(100 * MB, 100 * MB)
    p, q = shim.get(5 * MB), shim.get(6 * MB)
    shim.put(p)
    assert shim.release(1) == 0 and shim.release(0) == 5 * MB and shim.release(0) == 0
    assert shim.in_use(0) == 6 * MB                         # the block in use stays
    shim.put(q)
    assert shim.idle(0) == 6 * MB


def test_idle_memory_is_bounded_and_the_newest(shim):
    """Blocks of ever new sizes: what is kept never passes a quarter of the
    device, and it is the blocks given back last."""
    shim.start(400 * MB, 10 * MB)
    shim.set_device(1)
    shim.put(shim.get(MB))                                  # the other device's block is not the one to go
    shim.set_device(0)
    for k in range(12):
        shim.put(shim.get((20 + 2 * k) * MB))
        assert shim.idle(0) <= 100 * MB and shim.idle(0) == shim.in_use(0)
    assert shim.idle(0) == (42 + 40) * MB and shim.idle(1) == MB
    shim.put(shim.get(101 * MB))                            # too large to keep, and no reason to drop the others
    assert shim.idle(0) == (42 + 40) * MB == shim.in_use(0)


def test_every_allocation_of_the_library_reclaims():
    """hipMalloc is called in one place, under the pool; every other device
    allocation goes through the functions that reclaim idle blocks."""
    csrc = os.path.join(ROOT, "polymer_amd", "csrc")
    calls = []
    for path in glob.glob(os.path.join(csrc, "**", "*"), recursive=True):
        if path.endswith((".hip", ".cpp", ".h")) and "_build" not in path:
            for line in open(path):
                if re.search(r"\bhip(Ext)?Malloc\w*\s*\(", line.split("//")[0]) and '"hipMalloc' not in line:
                    calls.append((os.path.basename(path), line.strip()))
    assert calls == [("polyeri.hip", "const hipError_t e = hipMalloc(p, bytes);")]
