"""Work buffers kept between calls: a call in blocks that an earlier call of
other sizes left behind gives the result of a call in fresh ones (E(2) and
CCSD of different molecules in turn, contexts alive and closed), and the last
context's end gives the kept memory back."""
import ctypes
import gc

import numpy as np
import pytest

import polymer_amd as pa
from polymer_amd import geometry
from polymer_amd._lib import check, lib
from tests.molecules import BH_GOLDEN, H2O_GOLDEN

pytestmark = pytest.mark.gpu


def _run(atoms, basis):
    ctx = pa.Context(pa.read_basis(basis, atoms))
    r = ctx.self_consistent_field(scfconv=1e-9, diis=2, scfcycles=100)
    e2 = ctx.mp2_energy(r["co"], r["eps"], 0, r["iocc"], r["n_indep"])
    cc = ctx.ccsd(r["co"], r["eps"], 0, r["iocc"], r["n_indep"], conv=1e-9)
    return ctx, np.array([*e2, cc["e3"], cc["e_corr"]])


def _free_bytes():
    """Free device memory, asked of the HIP runtime that the library uses (a
    second runtime in the process, torch's own, may find no device left)."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    check(lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)))
    return free.value


def test_reused_blocks_give_the_same_results():
    gc.collect()
    jobs = [(BH_GOLDEN, "STO-3G"), (H2O_GOLDEN, "cc-pVDZ"), (geometry.water_cluster(3, 1), "6-31G"),
            (H2O_GOLDEN, "6-31Gss")]
    print("case: work buffers reused between calls", flush=True)
    fresh = []
    for atoms, basis in jobs:                 # one context at a time: each starts with no kept blocks
        ctx, e = _run(atoms, basis)
        ctx.close()
        fresh.append(e)
    keep = []
    for k in (1, 2, 0, 3, 2, 1, 3, 0):        # contexts stay: blocks pass from one to the next
        ctx, e = _run(*jobs[k])
        keep.append(ctx)
        # the SCF's atomics change the last digits of the orbitals, and the energies to first order in them
        assert np.max(np.abs(e - fresh[k])) < 1e-8
    held = _free_bytes()
    big, e = _run(geometry.water_cluster(4, 1), "cc-pVDZ")
    big.close()
    after = _free_bytes()
    assert held - after > 400 << 20            # its blocks (0.8 GB the MO integrals alone) are kept
    for ctx in keep:
        ctx.close()
    gc.collect()
    assert _free_bytes() > held


def test_idle_blocks_are_given_back_on_request():
    gc.collect()
    print("case: idle work buffers released", flush=True)
    ctx, e = _run(geometry.water_cluster(4, 1), "cc-pVDZ")
    kept = _free_bytes()
    n = ctx.release_work()
    assert n > 400 << 20                       # the MO integrals alone are 0.8 GB
    assert _free_bytes() - kept > n // 2
    assert ctx.release_work() == 0
    r = ctx.self_consistent_field(scfconv=1e-9, diis=2, scfcycles=100)
    again = np.array(ctx.mp2_energy(r["co"], r["eps"], 0, r["iocc"], r["n_indep"]))
    # the SCF's atomics change the last digits of the orbitals, and the energies to first order in them
    assert np.max(np.abs(again - e[:2])) < 1e-8
    ctx.close()
