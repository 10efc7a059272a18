"""The FP64 Rys J/K kernels (L >= 6, and L = 4 and 5 with few shell quartets) against the oracle where
their branches change: Cartesian and spherical d, with and without the screen (element screen and
Cartesian diagonal), one centre (T = 0), a dimer 40 bohr apart (T beyond the table), the
density-screened incremental build, and a batch on both sides of the shell-quartet count that moves
L = 4 and 5 between the kernels, and mixed contexts from L = 7. The exported ERI vector has the same integrals.

Tolerance: 1e-11 on J and K (integrals good to a few 1e-15 summed over at most 48^2 densities of
about 0.1) and 1e-12 on single integrals."""
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


def _density(n, seed):
    A = np.random.default_rng(seed).standard_normal((n, n))
    return 0.1 * (A + A.T)


@pytest.mark.parametrize("screen", [True, False])
@pytest.mark.parametrize("basis", ["6-31g**", "cc-pvdz"])
@pytest.mark.parametrize("kind", ["atom", "water", "near", "far"])
def test_rys_jk_matches_oracle(kind, basis, screen):
    Z, X = _system(kind)
    mol = H.Molecule.from_arrays(Z, X, basis)
    D = _density(mol.nbf, 3)
    ctx = H.GpuContext(mol, schwarz=screen)
    orc = oracle.Oracle(mol.shells(), mol.geometry()[1], mol.pure, 1e-14, screen=screen)
    err = max(float(np.abs(a - b).max()) for a, b in zip(ctx.build_jk(D), orc.jk(D)))
    orc.build_eri()
    ev = float(np.abs(ctx.eri_vector() - orc.eri_vector()).max())
    print(f"{kind} {basis} screen {screen}: |dJ|, |dK| {err:.1e}, ERIs {ev:.1e}", flush=True)
    assert err < 1e-11 and ev < 1e-12


def test_rys_jk_incremental_density_screen():
    Z, X = _system("near")
    mol = H.Molecule.from_arrays(Z, X, "cc-pvdz")
    D0, D1 = _density(mol.nbf, 4), _density(mol.nbf, 5)
    D1 = D0 + 1e-3 * D1
    Hc = np.zeros_like(D0)
    ctx = H.GpuContext(mol, density_tol=1e-15)
    ctx.fock(Hc, D0)
    F = ctx.fock(Hc, D1, incremental=True)
    assert np.abs(F - H.GpuContext(mol).fock(Hc, D1)).max() < 1e-11


def test_rys_jk_batch_across_the_quartet_count():
    mols = [H.Molecule.from_arrays(*_system("near"), "cc-pvdz") for _ in range(24)]
    D = _density(mols[0].nbf, 6)
    one = H.GpuContext(mols[0]).build_jk(D)
    J, K = H.GpuContext(mols).build_jk(np.concatenate([D.ravel()] * len(mols)))
    n = mols[0].nbf
    for got, ref in zip((J, K), one):
        assert np.abs(got.reshape(len(mols), n, n) - ref).max() < 1e-11


@pytest.mark.parametrize("basis", ["6-31g**", "cc-pvdz"])
@pytest.mark.parametrize("kind", ["water", "near", "far"])
def test_mixed_runs_fp64_rys_from_l7(kind, basis):
    # a density over the d functions alone: J and K between them come from (dd|dd) only, and so does the
    # gradient's two-electron part; a mixed context has both to FP64
    mol = H.Molecule.from_arrays(*_system(kind), basis)
    s = mol.shells()
    d = np.concatenate([np.arange(o, o + (5 if mol.pure else 6))
                        for L, o in zip(s["L"], s["pure_off"] if mol.pure else s["cart_off"]) if L == 2])
    D = np.zeros((mol.nbf, mol.nbf))
    D[np.ix_(d, d)] = _density(len(d), 7)
    ctx, ref = H.GpuContext(mol, precision=H.MIXED), H.GpuContext(mol)
    for got, want in zip(ctx.build_jk(D), ref.build_jk(D)):
        assert np.abs(got - want)[np.ix_(d, d)].max() < 1e-11
    assert np.abs(ctx.energy_backward(D) - ref.energy_backward(D)).max() < 1e-11
