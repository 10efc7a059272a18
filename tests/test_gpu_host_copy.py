"""The copy of the ERI vector to the host on both sides of the size from which it runs in chunks over
host threads (16 MB; the vectors end inside a chunk), from one thread and from two at once: every
chunk of the vector is checked through its Coulomb contraction against the direct build.

Tolerance: 1e-11 on J (integrals good to a few 1e-15 summed over at most 100^2 densities of about 0.1)."""
import threading

import numpy as np
import pytest

import hfscf_amd as H
from conftest import golden
from oracle import basis_ref

pytestmark = pytest.mark.gpu


def _coulomb_error(nwater, seed):
    Z, X = basis_ref.read_xyz(golden("h2o_8.xyz"))
    mol = H.Molecule.from_arrays(Z[: 3 * nwater], X[: 3 * nwater], "cc-pvdz")
    ctx = H.GpuContext(mol)
    v = ctx.eri_vector()
    n = mol.nbf
    A = np.random.default_rng(seed).standard_normal((n, n))
    D = 0.1 * (A + A.T)
    i, j = np.tril_indices(n)
    P = np.zeros((len(i), len(i)))
    P[np.tril_indices(len(i))] = v
    w = np.where(i == j, 1.0, 2.0) * D[i, j]
    Jv = P @ w + P.T @ w - np.diag(P) * w
    err = float(np.abs(Jv - ctx.build_jk(D)[0][i, j]).max())
    print(f"{nwater} waters, {v.nbytes / 2**20:.2f} MB: |dJ| {err:.1e}", flush=True)
    return err


@pytest.mark.parametrize("nwater", [1, 2, 3, 4])
def test_eri_vector_copy(nwater):
    assert _coulomb_error(nwater, nwater) < 1e-11


def test_eri_vector_copy_from_two_threads():
    errs = {}
    run = lambda n: errs.update({n: _coulomb_error(n, n)})
    ts = [threading.Thread(target=run, args=(n,)) for n in (3, 4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert len(errs) == 2 and max(errs.values()) < 1e-11
