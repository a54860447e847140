"""Work items shared between the lanes of a wavefront (segment and generally
contracted J/K kernels): the ket primitive pairs of a deeply contracted item
are divided over 2 .. 64 lanes and summed back.  Small molecules share nearly
every item, so the cases below reach every lane count, lists shorter than a
wavefront, ket counts that are not a multiple of the lanes, and one member
(shell pairs) or several (s-shell groups) an item."""
import numpy as np
import pytest

import oracle
import polymer_amd as pa
from polymer_amd import geometry
from tests.conftest import basis_path
from tests.molecules import BH_GOLDEN, H2O_GOLDEN

pytestmark = pytest.mark.gpu

CASES = {
    "ne_ccpvdz": ([(10, 0.1, 0.0, -0.2)], "cc-pVDZ"),
    "h2o_ccpvdz": (H2O_GOLDEN, "cc-pVDZ"),
    "h2o_631g": (H2O_GOLDEN, "6-31G"),
    "h2_631gss": ([(1, 0.0, 0.0, 0.0), (1, 0.0, 0.0, 1.4)], "6-31Gss"),
    "bh_sto3g": (BH_GOLDEN, "STO-3G"),
}


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("grouped", [True, False])
def test_shared_items_match_oracle(case, grouped):
    """J/K at Schwarz 0 against the oracle, and the density-screened form at a
    threshold below every bound, which has to keep every quartet.  Tolerance:
    sums of at most 10^5 terms below 10 in FP64, 10^5 x 10 x 2^-53 = 1e-10."""
    atoms, basis = CASES[case]
    b = pa.read_basis(basis, atoms)
    rng = np.random.default_rng(7)
    real = b.real_functions
    p = np.zeros((b.ncgs, b.ncgs))
    a = 0.1 * rng.standard_normal((len(real), len(real)))
    p[np.ix_(real, real)] = a + a.T
    ctx = pa.Context(b, schwarz_tol=0.0)
    ctx.set_general_contraction(grouped)
    print(f"case: shared items {case} grouped {grouped}", flush=True)
    j, k = ctx.fourindex_eri(p)
    n = ctx.stats()["last_quartets"]
    jr, kr = oracle.Basis(basis_path(basis), atoms).fourindex_eri(p, 0.0)[:2]
    assert np.max(np.abs(jr)) > 0 and np.max(np.abs(kr)) > 0
    assert np.max(np.abs(j - jr)) < 1e-10 and np.max(np.abs(k - kr)) < 1e-10
    js, ks = ctx.fourindex_eri(p, dens_tol=1e-290)
    assert np.max(np.abs(js - jr)) < 1e-10 and np.max(np.abs(ks - kr)) < 1e-10
    assert ctx.stats()["last_quartets"] >= n       # every quartet kept


def test_boys_rows_outside_lds_match_register_kernels():
    """Above about 450 functions the (dd|..) rows leave no LDS for the Boys
    rows and the segment kernel reads them from global memory; both it and
    the LDS form of the other classes against the thread-per-quartet kernels
    on the same quartets.  Tolerance: 10^6 terms of at most 1 a matrix
    element, 10^6 x 2^-53 = 1.2e-10, doubled for the two orders of summation."""
    atoms = geometry.water_cluster(19, 2, radius=5.5)
    print("case: Boys rows from global memory, (H2O)19 cc-pVDZ", flush=True)
    b = pa.read_basis("cc-pVDZ", atoms)
    ctx = pa.Context(b, schwarz_tol=1e-9)
    ctx.set_general_contraction(False)
    rng = np.random.default_rng(3)
    real = b.real_functions
    p = np.zeros((b.ncgs, b.ncgs))
    a = 0.05 * rng.standard_normal((len(real), 12))
    p[np.ix_(real, real)] = a @ a.T
    j, k = ctx.fourindex_eri(p)
    cls = ctx.stats()["classes"]
    kinds = {c["cls"]: c["kernel"] for c in cls if c["quartets"]}
    assert kinds["2200"] == "seg" and kinds["0000"] == "seg", kinds
    cfg = ctx.launch_configs()
    for c, x in zip(cfg, cls):
        if x["kernel"] == "seg":
            c[0], c[1], c[2] = 1, 256, 0
    ctx.set_launch_configs(cfg)
    jr, kr = ctx.fourindex_eri(p)
    assert np.max(np.abs(jr)) > 1
    assert np.max(np.abs(j - jr)) < 2.4e-10 and np.max(np.abs(k - kr)) < 2.4e-10


# p of six and d of two primitives: 36 ket primitive pairs in (pp|, 144 and
# more primitive quartets an item, the most lanes a Rys item can be given
DEEP_BASIS = """****
{el}     0
S    1   1.00
      6.0000000E-01          1.0000000
P    6   1.00
      9.5000000E+00          2.0000000E-02
      4.1000000E+00          9.0000000E-02
      2.0000000E+00          2.2000000E-01
      1.0500000E+00          3.5000000E-01
      5.5000000E-01          3.3000000E-01
      2.9000000E-01          1.5000000E-01
D    2   1.00
      1.7000000E+00          4.0000000E-01
      6.3000000E-01          7.0000000E-01
****
"""


@pytest.mark.parametrize("atoms", [[(10, 0.1, 0.0, -0.2)], [(10, 0.0, 0.1, 0.0), (10, 0.3, -0.2, 2.2)]],
                         ids=["one_centre", "two_centres"])
def test_shared_rys_items_match_oracle(tmp_path, atoms):
    """The Rys classes with 8 (six-lane members) and 16 (three-lane members)
    lane groups an item, against the oracle and with the screen that keeps
    every quartet; and the mixed-precision lists, part and all of the quartets
    in FP32.  Tolerance as above; FP32: an integral sums at most 144 primitive
    quartets of 3 to 5 roots, about 512 terms rounded to 2^-24 with errors of
    either sign, sqrt(512) 2^-24 of the sums that the density's magnitudes
    give (1.4e-6 of them; 2e-8 measured)."""
    path = str(tmp_path / "deep")
    with open(path, "w") as f:
        f.write(DEEP_BASIS.format(el="Ne"))
    b = pa.read_basis(path, atoms)
    rng = np.random.default_rng(5)
    real = b.real_functions
    p = np.zeros((b.ncgs, b.ncgs))
    a = 0.1 * rng.standard_normal((len(real), len(real)))
    p[np.ix_(real, real)] = a + a.T
    ctx = pa.Context(b, schwarz_tol=0.0)
    print(f"case: shared Rys items, {len(atoms)} centres", flush=True)
    j, k = ctx.fourindex_eri(p)
    assert any(c["kernel"] == "rys" and c["quartets"] for c in ctx.stats()["classes"])
    jr, kr = oracle.Basis(path, atoms).fourindex_eri(p, 0.0)[:2]
    assert np.max(np.abs(jr)) > 0 and np.max(np.abs(kr)) > 0
    assert np.max(np.abs(j - jr)) < 1e-10 and np.max(np.abs(k - kr)) < 1e-10
    js, ks = ctx.fourindex_eri(p, dens_tol=1e-290)
    assert np.max(np.abs(js - jr)) < 1e-10 and np.max(np.abs(ks - kr)) < 1e-10
    ja, ka = oracle.Basis(path, atoms).fourindex_eri(np.abs(p), 0.0)[:2]
    for cut in (1.0, 1e30):
        mixed = pa.Context(b, schwarz_tol=0.0, precision=pa.MIXED, mixed_cut=cut)
        jm, km = mixed.fourindex_eri(p)
        assert any(c["prec"] == "fp32" and c["kernel"] == "rys" and c["quartets"] for c in mixed.stats()["classes"])
        f32 = 512 ** 0.5 * 2.0 ** -24
        assert np.max(np.abs(jm - jr)) < f32 * np.max(np.abs(ja))
        assert np.max(np.abs(km - kr)) < f32 * np.max(np.abs(ka))
