"""A coordinate that is not a number shows in the one-electron integrals: every element of S and T with a
function of that atom is NaN and the others are those of the molecule without it; V, to which the atom's
nucleus adds everywhere, is NaN throughout.

Tolerance: 1e-12 on the finite elements (the bar of the other one-electron tests)."""
import numpy as np
import pytest

import hfscf_amd as H
from conftest import golden
from oracle import basis_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", ["sto-3g", "6-31g**", "cc-pvdz"])
def test_nan_coordinate(basis):
    Z, X = basis_ref.read_xyz(golden("h2o.xyz"))
    bad = np.array(X, dtype=float)
    bad[2, 1] = np.nan
    mol = H.Molecule.from_arrays(Z, bad, basis)
    s = mol.shells()
    off = s["pure_off"] if mol.pure else s["cart_off"]
    fine = np.concatenate([np.arange(o, o + (2 * L + 1 if mol.pure else (L + 1) * (L + 2) // 2))
                           for L, o, a in zip(s["L"], off, s["atom"]) if a != 2])
    S, T, V = H.GpuContext(mol).oneint()
    S0, T0, _ = H.GpuContext(H.Molecule.from_arrays(Z[:2], X[:2], basis)).oneint()
    rest = np.ones((mol.nbf, mol.nbf), dtype=bool)
    rest[np.ix_(fine, fine)] = False
    for M, M0 in ((S, S0), (T, T0)):
        assert np.isnan(M[rest]).all()
        assert np.abs(M[np.ix_(fine, fine)] - M0).max() < 1e-12
    assert np.isnan(V).all()
    # the engine goes on with finite coordinates
    ok = H.Molecule.from_arrays(Z, X, basis)
    assert all(np.isfinite(M).all() for M in H.GpuContext(ok).oneint())
