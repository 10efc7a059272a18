"""The one-electron kernels where their work split changes, against the oracle's numpy restatement:
one nucleus (fewer nuclei than slices), three and six nuclei, 1 to 81 primitive pairs per shell
pair, every pair class of Cartesian and spherical d shells, and a dimer so far apart that primitive
pairs vanish (the cut of terms that no double can hold).

Tolerances: matrix elements 1e-12, gradient terms 1e-11 (the bars of the other one-electron tests)."""
import numpy as np
import pytest

import hfscf_amd as H
from conftest import golden
from oracle import basis_ref
from oracle import oneint_ref as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", ["6-31g**", "cc-pvdz"])
@pytest.mark.parametrize("kind", ["atom", "water", "far"])
def test_oneint_and_gradient(kind, basis):
    Z, X = basis_ref.read_xyz(golden("h2o.xyz"))
    if kind == "atom":
        Z, X = Z[:1], X[:1] + np.array([0.3, -0.2, 0.1])
    elif kind == "far":
        Z, X = np.concatenate([Z, Z]), np.concatenate([X, X[:, [1, 2, 0]] + np.array([1.0, 2.0, 25.0])])
    sh, pure, n = basis_ref.shells_for(Z, basis, None)
    mol = H.Molecule.from_arrays(Z, X, basis)
    ctx = H.GpuContext(mol)
    err = max(float(np.abs(a - b).max()) for a, b in zip(ctx.oneint(), O.oneint(sh, pure, Z, X)))
    rng = np.random.default_rng(8)
    D, Q = (0.1 * (A + A.T) for A in rng.standard_normal((2, n, n)))
    g = ctx.oneint_gradient(D, Q)
    eg = float(np.abs(g - O.oneint_gradient(sh, pure, Z, X, D, Q)).max())
    print(f"{kind} {basis}: |dSTV| {err:.1e} |dg| {eg:.1e}", flush=True)
    assert err < 1e-12 and eg < 1e-11
