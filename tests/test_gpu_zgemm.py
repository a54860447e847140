"""Planar complex products of the k-point MP2 (polyeri_zgemm_launch through
E(2)): band counts and group sizes at which the tiles have remainders.  The
first quarter takes several k-points in one product when their band counts
agree, so chains with equal and with different counts are both run; E(2)
against the BF16-split transform of the same bands, whose kernel shares no
tile with the FP64 one, to that transform's 1e-6 relative accuracy."""
import numpy as np
import pytest

import polymer_amd as pa
from polymer_amd import run_polyethylene

pytestmark = pytest.mark.gpu
ANG = 1.0 / pa.ANG_BOHR


@pytest.mark.parametrize("units,kpoints", [(1, 2), (2, 1), (2, 3)])
def test_transform_tiles(units, kpoints):
    period = 2.55 * ANG
    atoms = [(z, x + u * period, y, w) for u in range(units) for z, x, y, w in run_polyethylene.cell()]
    b = pa.read_basis("STO-3G", atoms)
    ctx = pa.Context(b, period=units * period, cel1=1, cel2=2)
    r = ctx.self_consistent_field_periodic(kpoints=kpoints, scfconv=1e-9, diis=5, scfcycles=100)
    print(f"case: complex products, {units} units, {2 * kpoints} k-points", flush=True)
    args = (kpoints, r["co"], r["eps"])
    full = np.array(ctx.mp2_energy_periodic(*args, r["nall"], 2 * units, r["iocc"]))
    split = np.array(ctx.mp2_energy_periodic(*args, r["nall"], 2 * units, r["iocc"], transform="bf16x3"))
    assert np.max(np.abs(full)) > 1e-2
    assert np.max(np.abs(split - full)) < 1e-6 * np.max(np.abs(full))
    # one k-point with fewer bands: the group is cut there, and with every
    # k-point cut to it the products are those of a smaller problem
    fewer = r["nall"].copy()
    fewer[-1] -= 3
    cut = np.array(ctx.mp2_energy_periodic(*args, fewer, 2 * units, r["iocc"]))
    cut_split = np.array(ctx.mp2_energy_periodic(*args, fewer, 2 * units, r["iocc"], transform="bf16x3"))
    assert np.max(np.abs(cut_split - cut)) < 1e-6 * np.max(np.abs(full))
    assert np.max(np.abs(cut - full)) > 1e-6 * np.max(np.abs(full))
