"""FP64 gradient classes on the Rys kernel (L >= 4) against the oracle's contracted derivative
integrals, where the kernel's branches change: Cartesian and spherical d, every class (a dimer has
one- and four-primitive p shells beside the d shells), quartets on one centre (T = 0), quartets
beyond the tabulated T (a dimer 40 bohr apart: T = rho R^2 from 72 up for all but the most diffuse
primitives), and a batch whose molecules have different Cartesian offsets.

Tolerance: 1e-11 of the largest component. The kernel sums of the order of 1e5 products per
component, each good to a few 1e-16 of integrals that cancel by less than 1e2."""
import numpy as np
import pytest

import hfscf_amd as H
import oracle
from conftest import golden
from oracle import basis_ref

pytestmark = pytest.mark.gpu


def _density(n, seed):
    A = np.random.default_rng(seed).standard_normal((n, n))
    return 0.1 * (A + A.T)


def _system(kind):
    Z, X = basis_ref.read_xyz(golden("h2o.xyz"))
    if kind == "atom":
        return Z[:1], X[:1]
    if kind == "water":
        return Z, X + np.array([[0.1, -0.05, 0.02], [0.0, 0.03, -0.04], [0.02, 0.0, 0.05]])
    shift = {"near": np.array([0.7, 5.2, 0.4]), "far": np.array([3.0, 1.0, 40.0])}[kind]
    R = np.array([[0.36, 0.48, -0.8], [-0.8, 0.6, 0.0], [0.48, 0.64, 0.6]])
    return np.concatenate([Z, Z]), np.concatenate([X, X @ R.T + shift])


@pytest.mark.parametrize("basis", ["6-31g**", "cc-pvdz"])
@pytest.mark.parametrize("kind", ["atom", "water", "near", "far"])
def test_rys_gradient_matches_oracle(kind, basis):
    Z, X = _system(kind)
    mol = H.Molecule.from_arrays(Z, X, basis)
    D = _density(mol.nbf, 11)
    g = H.GpuContext(mol, schwarz=False).energy_backward(D)
    r = oracle.Oracle(mol.shells(), mol.geometry()[1], mol.pure, 1e-14, screen=False).grad2e(D)
    err, top = float(np.abs(g - r).max()), max(1.0, float(np.abs(r).max()))
    print(f"{kind} {basis}: |dg| {err:.1e}, max |g| {top:.1e}", flush=True)
    assert err < 1e-11 * top


def test_rys_gradient_batch_offsets():
    mols = [H.Molecule.from_arrays(*_system(k), "cc-pvdz") for k in ("water", "near", "atom", "water")]
    Ds = [_density(m.nbf, 20 + k) for k, m in enumerate(mols)]
    g = H.GpuContext(mols, schwarz=False).energy_backward(np.concatenate([d.ravel() for d in Ds]))
    one = np.concatenate([H.GpuContext(m, schwarz=False).energy_backward(d) for m, d in zip(mols, Ds)])
    assert np.abs(g - one).max() < 1e-11 * max(1.0, np.abs(one).max())
