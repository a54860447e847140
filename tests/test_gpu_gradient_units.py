"""The two-electron gradient with a quartet's work shared by several lanes:
cases from one lane a quartet (STO-3G) to hundreds (two contracted s pairs of
cc-pVDZ), whole primitive quartets and single roots as units, against the
host run of the same code.  Tolerance: the sums differ in their order only,
10^5 contributions of at most 10 to a coordinate, 10^6 x 2^-53 = 1.1e-10."""
import numpy as np
import pytest

import polymer_amd as pa
from tests.molecules import BH_GOLDEN, FH_GOLDEN, H2O_GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("atoms,basis", [(BH_GOLDEN, "STO-3G"), (H2O_GOLDEN, "6-31G"), (FH_GOLDEN, "cc-pVDZ"),
                                         ([(1, 0.0, 0.0, 0.0), (1, 0.0, 0.0, 1.4)], "6-31Gss")])
@pytest.mark.parametrize("tol", [0.0, 1e-9])
def test_gradient_lanes_match_host(atoms, basis, tol):
    b = pa.read_basis(basis, atoms)
    rng = np.random.default_rng(11)
    p = np.zeros((b.ncgs, b.ncgs))
    real = b.real_functions
    a = 0.2 * rng.standard_normal((len(real), len(real)))
    p[np.ix_(real, real)] = a + a.T
    print(f"case: gradient units {basis} {len(atoms)} atoms tol {tol}", flush=True)
    g = pa.Context(b, schwarz_tol=tol).eri_gradient(p)
    ref = pa.eri_gradient_host(b, p, schwarz_tol=tol)
    assert np.max(np.abs(ref)) > 1e-3
    # at a threshold the two sides' bounds (recursion and quadrature) may differ in the last digit
    assert np.max(np.abs(g - ref)) < (1.1e-10 if tol == 0.0 else 1e-8)
    assert np.max(np.abs(g.sum(0))) < 1.1e-10
