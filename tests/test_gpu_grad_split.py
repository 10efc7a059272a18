"""The register gradient kernels where their split over the primitives changes, against the oracle: few
quartets (more lanes per shell quartet than a bra pair has primitives), a dimer, and a batch (about one
lane per quartet); minimal, split-valence and generally contracted bases, spherical and Cartesian, so
that a bra pair has 1 to 64 primitives.

Tolerance: 1e-10 on a gradient component (derivative integrals good to a few 1e-14 summed over at most 48^2
densities of about 0.1 and their products)."""
import numpy as np
import pytest

import hfscf_amd as H
import oracle
from conftest import golden
from oracle import basis_ref

pytestmark = pytest.mark.gpu


def _mol(kind, basis):
    Z, X = basis_ref.read_xyz(golden("h2o.xyz"))
    X = X + np.array([[0.1, -0.05, 0.02], [0.0, 0.03, -0.04], [0.02, 0.0, 0.05]])
    if kind == "atom":
        Z, X = Z[:1], X[:1]
    elif kind == "dimer":
        Z, X = np.concatenate([Z, Z]), np.concatenate([X, X @ np.diag([-1.0, 1.0, -1.0]) + np.array([0.7, 5.2, 0.4])])
    return H.Molecule.from_arrays(Z, X, basis)


def _density(n, seed):
    A = np.random.default_rng(seed).standard_normal((n, n))
    return 0.1 * (A + A.T)


@pytest.mark.parametrize("basis", ["sto-3g", "6-31g*", "cc-pvdz"])
@pytest.mark.parametrize("kind", ["atom", "water", "dimer"])
def test_split_gradient_matches_oracle(kind, basis):
    mol = _mol(kind, basis)
    D = _density(mol.nbf, 2)
    ref = oracle.Oracle(mol.shells(), mol.geometry()[1], mol.pure, 1e-14, screen=False).grad2e(D)
    err = float(np.abs(H.GpuContext(mol, schwarz=False).energy_backward(D) - ref).max())
    print(f"{kind} {basis}: |dG| {err:.1e}", flush=True)
    assert err < 1e-10


def test_split_gradient_in_a_batch():
    mol = _mol("dimer", "cc-pvdz")
    D = _density(mol.nbf, 3)
    one = H.GpuContext(mol).energy_backward(D)
    g = H.GpuContext([mol] * 40).energy_backward(np.concatenate([D.ravel()] * 40))
    assert np.abs(np.asarray(g).reshape((40,) + one.shape) - one).max() < 1e-11
