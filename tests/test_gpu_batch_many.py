"""A batch of more molecules than the 65,536 workgroups of a grid's second dimension: its gradient, whose Cartesian
densities are formed one molecule per grid row, against one molecule's.

Tolerance: 1e-11 on a gradient component (the bar of the other batch gradients)."""
import numpy as np
import pytest

import hfscf_amd as H

pytestmark = pytest.mark.gpu


def test_gradient_of_many_molecules():
    n = 65600
    mol = H.Molecule.from_arrays(np.array([1, 1], dtype=np.int32), np.array([[0.0, 0.0, 0.0], [0.3, 0.2, 1.35]]), "cc-pvdz")
    A = np.random.default_rng(2).standard_normal((mol.nbf, mol.nbf))
    D = 0.1 * (A + A.T)
    one = H.GpuContext(mol).energy_backward(D)
    ctx = H.GpuContext([mol] * n)
    print("set up", flush=True)
    g = np.asarray(ctx.energy_backward(np.tile(D.ravel(), n))).reshape(n, 2, 3)
    assert np.abs(one).max() > 1e-3 and np.abs(g - one).max() < 1e-11
