"""Allocations that fail at a bound (set from the host: a stand-in for
hipMalloc in a child process counts the live bytes and refuses what passes the
bound; no device memory is exhausted).  Whatever the work pool keeps idle may
not be the reason why a call runs out of memory."""
import os
import subprocess
import sys

import numpy as np
import pytest

import polymer_amd as pa
from polymer_amd import geometry, guess
from polymer_amd._lib import check, lib
from tests.conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <cstddef>
#include <cstdlib>
#include <map>
#include <mutex>
static std::mutex mu;
static std::map<void*, size_t> blocks;
static size_t live = 0, peak = 0, bound = ~size_t(0), refused = 0;
static void* real(const char* name) {
    static void* h = dlopen("libamdhip64.so.7", RTLD_NOW);
    void* f = h ? dlsym(h, name) : nullptr;
    if (!f) abort();
    return f;
}
extern "C" {
int hipMalloc(void** p, size_t n) {
    static auto f = (int (*)(void**, size_t))real("hipMalloc");
    std::lock_guard<std::mutex> lk(mu);
    if (live + n > bound) { ++refused; return 2; }
    const int e = f(p, n);
    if (!e) { blocks[*p] = n; live += n; if (live > peak) peak = live; }
    return e;
}
int hipFree(void* p) {
    static auto f = (int (*)(void*))real("hipFree");
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.find(p);
    if (it != blocks.end()) { live -= it->second; blocks.erase(it); }
    return f(p);
}
size_t shim_live() { return live; }
size_t shim_peak() { size_t q = peak; peak = live; return q; }
size_t shim_refused() { size_t r = refused; refused = 0; return r; }
void shim_bound(size_t b) { bound = b; }
}
"""

CHILD = r"""
import ctypes, sys
S = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in (S.shim_live, S.shim_peak, S.shim_refused):
    f.restype = ctypes.c_size_t
S.shim_bound.argtypes = [ctypes.c_size_t]
NONE = 2 ** 64 - 1
import numpy as np
import polymer_amd as pa
from polymer_amd import geometry, guess, run_polyethylene

def others():
    ctx = pa.Context(pa.read_basis("cc-pVDZ", geometry.water_cluster(4, 1)))
    r = ctx.self_consistent_field(scfconv=1e-9, diis=2, scfcycles=100)
    e2 = ctx.mp2_energy(r["co"], r["eps"], 0, r["iocc"], r["n_indep"])
    assert S.shim_live() > 400 << 20, "the stand-in is not in place"
    again = pa.Context(pa.read_basis("cc-pVDZ", geometry.water_cluster(4, 2)))
    small = pa.Context(pa.read_basis("cc-pVDZ", geometry.water()))
    calls = dict(
        device_alloc=lambda: ctx.device_free(ctx.device_alloc(64 << 20)),
        scf=lambda: again.self_consistent_field(scfconv=1e-8, diis=2, scfcycles=100),
        fast_scf=lambda: small.self_consistent_field(scfconv=1e-8, scfcycles=100, solver=1, diis_mode=1),
        fock=lambda: fock(again),
        network=lambda: guess.mlp_forward(guess.MLP([64, 256, 225], seed=5), ctx, np.zeros((700, 64), np.float32)),
        context=lambda: pa.Context(pa.read_basis("6-31Gss", geometry.water_cluster(3, 1))).close(),
    )
    for name, call in calls.items():
        print("bounded:", name, flush=True)
        S.shim_bound(NONE)
        ctx.mp2_energy(r["co"], r["eps"], 0, r["iocc"], r["n_indep"])     # leaves its blocks idle
        S.shim_refused()
        S.shim_bound(S.shim_live())
        call()
        assert S.shim_refused() > 0, name
    S.shim_bound(NONE)
    e = ctx.mp2_energy(r["co"], r["eps"], 0, r["iocc"], r["n_indep"])
    assert np.max(np.abs(np.array(e) - e2)) < 1e-9

def fock(ctx):
    n2 = ctx.basis.ncgs ** 2 * 8
    d = [ctx.device_alloc(n2) for _ in range(4)]
    ctx.to_device(d[0], np.eye(ctx.basis.ncgs))
    ctx.fock_build_device(*d)
    ctx.sync()
    for x in d:
        ctx.device_free(x)

def kpoint_mp2():
    period = 2.55 / pa.ANG_BOHR
    b = pa.read_basis("STO-3G", run_polyethylene.cell())
    ctx = pa.Context(b, period=period, cel1=1, cel2=2)
    r = ctx.self_consistent_field_periodic(kpoints=3, scfconv=1e-9, diis=5, scfcycles=100)
    args = (3, r["co"], r["eps"], r["nall"], 2, r["iocc"])
    ctx.mp2_energy_periodic(*args)         # what the context allocates once
    ctx.release_work()
    held = S.shim_live()
    S.shim_peak()
    want = np.array(ctx.mp2_energy_periodic(*args))
    need = S.shim_peak()
    ctx.release_work()
    S.shim_peak()
    print("bounded: k-point MP2", held, need, flush=True)
    S.shim_refused()
    S.shim_bound(need - 4096)              # the grouped first quarter does not fit, that of one k-point does
    got = np.array(ctx.mp2_energy_periodic(*args))
    refused, peak = S.shim_refused(), S.shim_peak()
    assert refused > 0 and peak < need, (refused, peak)
    assert np.max(np.abs(got - want)) < 1e-13 * np.max(np.abs(want)) + 1e-15
    ctx.release_work()
    S.shim_bound(held + (need - held) // 64)
    try:
        ctx.mp2_energy_periodic(*args)
        raise SystemExit("no error without memory")
    except pa.PolyeriError as e:
        assert e.code == -4 or "memory" in str(e).lower(), e

dict(others=others, kpoint_mp2=kpoint_mp2)[sys.argv[2]]()
print("bounded calls done", flush=True)
"""


@pytest.mark.parametrize("part", ["others", "kpoint_mp2"])
def test_calls_at_the_end_of_memory(tmp_path, part):
    src, so = str(tmp_path / "shim.cpp"), str(tmp_path / "shim.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", src, "-o", so, "-ldl"])
    print(f"case: allocations refused, {part}", flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD, so, part], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "bounded calls done" in r.stdout, r.stdout + r.stderr


def test_network_after_a_batch_that_did_not_fit():
    """A batch whose activations no device holds is refused before anything is
    launched, and leaves a network that allocates again for the next one."""
    print("case: network batch beyond the device's memory", flush=True)
    ctx = pa.Context(pa.read_basis("STO-3G", geometry.water()))
    net = guess.MLP([8, 4096, 4096, 5], seed=3)
    x = np.random.default_rng(1).standard_normal((40, 8)).astype(np.float32)
    y = guess.mlp_forward(net, ctx, x)
    d = ctx.device_alloc(1 << 20)
    with pytest.raises(pa.PolyeriError):
        check(lib().polyeri_mlp_forward(net.h, d, 2 ** 30, d))
    ctx.device_free(d)
    assert np.array_equal(guess.mlp_forward(net, ctx, x), y)
