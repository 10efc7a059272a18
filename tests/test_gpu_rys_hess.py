"""The Hessian's Rys kernels against the oracle's second-derivative integrals where their branches
change: one centre (T = 0, every derivative cancels), quartets beyond the tabulated T (a dimer 40
bohr apart), Cartesian d with every class of a dimer, and water / cc-pVDZ, whose 81 x 81 primitive
quartets take many work items of one shell quartet.

Tolerance: 1e-10 Eh/bohr^2 absolute (a hundredth of the entry point's 1e-8 bar: integrals good to a
few 1e-15 times second-derivative factors 4 alpha^2 of the tight primitives, up to 1e4 in weighted
sums that cancel)."""
import numpy as np
import pytest

import hfscf_amd as H
import oracle
from conftest import golden
from oracle import basis_ref

pytestmark = pytest.mark.gpu


def _system(kind):
    Z, X = basis_ref.read_xyz(golden("h2o.xyz"))
    if kind == "atom":
        return Z[:1], X[:1]
    if kind == "water":
        return Z, X + np.array([[0.1, -0.05, 0.02], [0.0, 0.03, -0.04], [0.02, 0.0, 0.05]])
    shift = {"near": np.array([0.7, 5.2, 0.4]), "far": np.array([3.0, 1.0, 40.0])}[kind]
    R = np.array([[0.36, 0.48, -0.8], [-0.8, 0.6, 0.0], [0.48, 0.64, 0.6]])
    return np.concatenate([Z, Z]), np.concatenate([X, X @ R.T + shift])


@pytest.mark.parametrize("kind,basis", [("atom", "6-31g*"), ("atom", "cc-pvdz"), ("water", "cc-pvdz"), ("near", "6-31g*"),
                                        ("far", "sto-3g"), ("far", "6-31g*")])
def test_rys_hessian_matches_oracle(kind, basis):
    Z, X = _system(kind)
    mol = H.Molecule.from_arrays(Z, X, basis)
    A = np.random.default_rng(4).standard_normal((mol.nbf, mol.nbf))
    D = 0.1 * (A + A.T)
    hc, hx = H.GpuContext(mol).hessian_2e(D)
    rc, rx = oracle.Oracle(mol.shells(), mol.geometry()[1], mol.pure, 1e-14, screen=False).hess2e(D)
    ec, ex = float(np.abs(hc - rc).max()), float(np.abs(hx - rx).max())
    print(f"{kind} {basis}: |dHC| {ec:.1e} |dHX| {ex:.1e}", flush=True)
    assert ec < 1e-10 and ex < 1e-10
