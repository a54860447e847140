"""Planar complex products of the k-point MP2 (polyeri_zgemm_launch): the
products themselves against numpy's, at sizes where the tiles, the row and
column splits and the batches have remainders; and E(2) through them against
the oracle, with equal band counts at the k-points (the first quarter takes
several k-points in one product) and with counts that cut such a group at its
end and in its middle."""
import ctypes

import numpy as np
import pytest

import polymer_amd as pa
from oracle import periodic
from polymer_amd import geometry, run_polyethylene
from polymer_amd._lib import lib

pytestmark = pytest.mark.gpu
ANG = 1.0 / pa.ANG_BOHR
F64 = 1


@pytest.fixture(scope="module")
def ctx():
    return pa.Context(pa.read_basis("STO-3G", geometry.water()))


def _put(ctx, ptrs, x):
    d = ctx.device_alloc(x.nbytes)
    ptrs.append(d)
    ctx.to_device_raw(d, x)
    return d


def _launch(*args):
    """polyeri_zgemm_launch(mode, M, N, K, Ar, Ai, sam, sA, Br, Bi, sbk, sB, Cr, Ci, scm, scn, sC, batch, stream,
    nci, sbo, sco, mci, smo) on the null stream, waited for."""
    f = lib().polyeri_zgemm_launch
    i, g, p = ctypes.c_int, ctypes.c_long, ctypes.c_void_p
    f.argtypes = [i, i, i, i, p, p, g, g, p, p, g, g, p, p, g, g, g, i, p, i, g, g, i, g]
    assert f(*args) == 0
    assert lib().hipDeviceSynchronize() == 0


# one, two, three and four column tiles and the widths on either side of them,
# rows and K slices short of, at and beyond a block's 128 and 8
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (16, 16, 8), (127, 15, 7), (128, 17, 9), (129, 32, 16), (33, 33, 3),
                                   (300, 48, 21), (64, 49, 8), (257, 64, 5), (40, 65, 24), (130, 80, 10),
                                   (131, 97, 17), (20, 130, 12)])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("rowc", [False, True])
def test_products_match_numpy(ctx, M, N, K, cplx, rowc):
    """Three batches, M and N split into runs with a gap between them where
    they divide, C by rows or by columns; what lies between the written
    elements keeps its value.  Tolerance: 2 K products and as many sums, each
    rounded once, (2 K + 2) 2^-53 of the sum of the products' magnitudes."""
    print(f"case: complex product M {M} N {N} K {K} complex {cplx} rows contiguous {rowc}", flush=True)
    rng = np.random.default_rng(M * 1009 + N * 31 + K)
    nb, pad = 3, 5
    mci = next((M // q for q in (3, 2) if M % q == 0), M)
    nci = next((N // q for q in (4, 5, 3, 2) if N % q == 0), N)
    mo, no = M // mci, N // nci
    A = rng.standard_normal((nb, M, K + 1)) + 1j * rng.standard_normal((nb, M, K + 1)) * cplx   # a row is longer than K
    B = rng.standard_normal((nb, no, K, nci + 2)) + 1j * rng.standard_normal((nb, no, K, nci + 2))
    bm = np.concatenate([B[:, o, :, :nci] for o in range(no)], axis=2)
    am = A[:, :, :K]
    want = np.matmul(am, bm)
    size = np.matmul(np.abs(am.real) + np.abs(am.imag), np.abs(bm.real) + np.abs(bm.imag))
    # C: outer row runs, outer column runs, then the inner block by rows or by columns
    inner = mci * nci + pad
    scm, scn = (1, mci) if rowc else (nci, 1)
    sco, smo = inner, inner * no
    sC = smo * mo + pad
    fill = 7.25
    cr, ci = np.full(nb * sC, fill), np.full(nb * sC, fill)
    m, n = np.arange(M)[:, None], np.arange(N)[None, :]
    at = (m // mci) * smo + (m % mci) * scm + (n // nci) * sco + (n % nci) * scn
    ptrs = []
    try:
        put = lambda x: _put(ctx, ptrs, np.ascontiguousarray(x))
        dar, dai, dbr, dbi, dcr, dci = put(A.real), put(A.imag), put(B.real), put(B.imag), put(cr), put(ci)
        _launch(F64, M, N, K, dar, dai if cplx else None, K + 1, M * (K + 1), dbr, dbi, nci + 2, no * K * (nci + 2),
                dcr, dci, scm, scn, sC, nb, None, nci, K * (nci + 2), sco, mci, smo)
        ctx.from_device_raw(dcr, cr)
        ctx.from_device_raw(dci, ci)
    finally:
        for d in ptrs:
            ctx.device_free(d)
    for b in range(nb):
        got = cr[b * sC + at] + 1j * ci[b * sC + at]
        tol = (2 * K + 2) * 2.0 ** -53 * size[b]
        assert np.all(np.abs(got.real - want[b].real) <= tol) and np.all(np.abs(got.imag - want[b].imag) <= tol)
        keep = np.ones(sC, dtype=bool)
        keep[at] = False
        assert np.all(cr[b * sC:(b + 1) * sC][keep] == fill) and np.all(ci[b * sC:(b + 1) * sC][keep] == fill)


@pytest.mark.parametrize("units,kpoints", [(1, 2), (1, 3), (2, 1), (2, 3)])
def test_transform_tiles(units, kpoints):
    """E(2) of polyethylene cells to 1e-10 Eh of the oracle's transform of the
    same lattice integrals and bands, to the BF16-split transform's 1e-6."""
    period = 2.55 * ANG
    atoms = [(z, x + u * period, y, w) for u in range(units) for z, x, y, w in run_polyethylene.cell()]
    b = pa.read_basis("STO-3G", atoms)
    ctx = pa.Context(b, period=units * period, cel1=1, cel2=2)
    r = ctx.self_consistent_field_periodic(kpoints=kpoints, scfconv=1e-9, diis=5, scfcycles=100)
    print(f"case: complex products, {units} units, {2 * kpoints} k-points", flush=True)
    nk, icore, iocc = 2 * kpoints, 2 * units, r["iocc"]
    T = ctx.eri_tensor_cells()          # against the oracle's in test_gpu_periodic.py
    args = (kpoints, r["co"], r["eps"])
    last, middle, few = r["nall"].copy(), r["nall"].copy(), r["nall"].copy()
    last[-1] -= 3                       # a group that ends before the last k-point
    middle[(nk - 1) // 2] -= 3          # a second group starts behind this one
    few[:] = iocc + 4                   # the same with fewer columns
    few[(nk - 1) // 2] -= 2
    full = np.array(ctx.mp2_energy_periodic(*args, r["nall"], icore, iocc))
    split = np.array(ctx.mp2_energy_periodic(*args, r["nall"], icore, iocc, transform="bf16x3"))
    assert np.max(np.abs(full)) > 1e-2
    assert np.max(np.abs(split - full)) < 1e-6 * np.max(np.abs(full))
    # the oracle's transform of all bands at many k-points takes long
    for nall in [few] + ([r["nall"], last, middle] if units * kpoints <= 3 else []):
        e = np.array(ctx.mp2_energy_periodic(*args, nall, icore, iocc))
        ref = np.array(periodic.mp2_kpoints(T, r["co"], r["eps"], ctx.reduced_cel1, 2, kpoints, icore, iocc, list(nall)))
        print("bands", list(nall), "E2", e, "oracle", ref, flush=True)
        assert np.max(np.abs(e - ref)) < 1e-10
    cut = np.array(ctx.mp2_energy_periodic(*args, last, icore, iocc))
    cut_split = np.array(ctx.mp2_energy_periodic(*args, last, icore, iocc, transform="bf16x3"))
    assert np.max(np.abs(cut_split - cut)) < 1e-6 * np.max(np.abs(full))
    assert np.max(np.abs(cut - full)) > 1e-6 * np.max(np.abs(full))
