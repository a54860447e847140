"""Work buffers kept between calls: a call in blocks that an earlier call of
other sizes left behind gives the result of a call in fresh ones (E(2) and
CCSD of different molecules in turn, contexts alive and closed; gradients,
periodic SCFs and k-point MP2 in turn), and the last context's end or a
request gives the kept memory back."""
import ctypes
import gc

import numpy as np
import pytest

import polymer_amd as pa
from polymer_amd import geometry, run_polyethylene
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


def _gradient(n, basis):
    b = pa.read_basis(basis, geometry.water_cluster(n, 1))
    ctx = pa.Context(b)
    rng = np.random.default_rng(n)
    p = np.zeros((b.ncgs, b.ncgs))
    a = 0.1 * rng.standard_normal((len(b.real_functions), 5 * n))
    p[np.ix_(b.real_functions, b.real_functions)] = a @ a.T
    return ctx, ctx.eri_gradient(p).ravel()


def _polymer(units, kpoints):
    period = 2.55 / pa.ANG_BOHR
    atoms = [(z, x + u * period, y, w) for u in range(units) for z, x, y, w in run_polyethylene.cell()]
    ctx = pa.Context(pa.read_basis("STO-3G", atoms), period=units * period, cel1=1, cel2=2)
    r = ctx.self_consistent_field_periodic(kpoints=kpoints, scfconv=1e-9, diis=5, scfcycles=100)
    e2 = ctx.mp2_energy_periodic(kpoints, r["co"], r["eps"], r["nall"], 2 * units, r["iocc"])
    return ctx, np.array([r["e_total"], *e2])


def test_blocks_pass_between_gradient_and_polymer_calls():
    gc.collect()
    jobs = [(_gradient, 1, "cc-pVDZ"), (_polymer, 1, 3), (_gradient, 3, "6-31Gss"), (_polymer, 2, 1), (_polymer, 1, 1)]
    print("case: work buffers of gradient, periodic SCF and k-point MP2", flush=True)
    fresh = []
    for f, *args in jobs:
        ctx, e = f(*args)
        ctx.close()
        fresh.append(e)
    keep = []
    for k in (3, 1, 0, 4, 2, 3, 0, 1, 2, 4):
        f, *args = jobs[k]
        ctx, e = f(*args)
        keep.append(ctx)
        assert np.max(np.abs(fresh[k])) > 1e-3
        # the order of the atomics' sums: 10^5 terms of at most 10, 1.1e-10, first order in the orbitals' for E(2)
        assert np.max(np.abs(e - fresh[k])) < (1.1e-10 if f is _gradient else 1e-8)
    for ctx in keep:
        ctx.close()


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
