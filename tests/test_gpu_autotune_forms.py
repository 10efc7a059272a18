"""Autotuning of contexts that ask for the cooperative kernels (coop_min_l 4 to 7): a class is only tried
and left on kernels that its precision has, also when the other precision runs afterwards.

Tolerances: 1e-11 on J and K, 1e-10 on gradients, 1e-12 on single integrals in FP64 (the bars of the FP64 kernels'
tests), 1e-5 on a mixed context's J and K against FP64."""
import numpy as np
import pytest

import hfscf_amd as H
from conftest import golden

pytestmark = pytest.mark.gpu


def _density(n):
    A = np.random.default_rng(11).standard_normal((n, n))
    return 0.1 * (A + A.T)


def _results(ctx, D):
    J, K = ctx.build_jk(D)
    return J, K, ctx.energy_backward(D), ctx.eri_vector()


def _check(got, want, bars=(1e-11, 1e-11, 1e-10, 1e-12)):
    err = [float(np.abs(a - b).max()) for a, b in zip(got, want)]
    print(" ".join(f"{e:.1e}" for e in err), flush=True)
    assert all(e < b for e, b in zip(err, bars))


@pytest.mark.parametrize("basis", ["6-31g**", "cc-pvdz"])
@pytest.mark.parametrize("coop_min_l", [4, 5, 6, 7])
def test_autotune_fp64(basis, coop_min_l):
    mol = H.Molecule.from_xyz(golden("h2o.xyz"), basis)
    D = _density(mol.nbf)
    want = _results(H.GpuContext(mol), D)
    ctx = H.GpuContext(mol, coop_min_l=coop_min_l)
    ctx.build_jk(D)
    ctx.autotune(3)
    _check(_results(ctx, D), want)


@pytest.mark.parametrize("coop_min_l", [0, 4, 5, 6])
def test_autotune_mixed_then_fp64(coop_min_l):
    mol = H.Molecule.from_xyz(golden("h2o.xyz"), "cc-pvdz")
    D = _density(mol.nbf)
    want = _results(H.GpuContext(mol), D)
    ctx = H.GpuContext(mol, precision=H.MIXED, coop_min_l=coop_min_l)
    ctx.build_jk(D)
    ctx.autotune(3)
    _check(ctx.build_jk(D), want[:2], (1e-5, 1e-5))
    ctx.set_precision(H.FP64)
    _check(_results(ctx, D), want)
    ctx.autotune(3)
    _check(_results(ctx, D), want)
    ctx.set_precision(H.MIXED)
    _check(ctx.build_jk(D), want[:2], (1e-5, 1e-5))


def test_launch_shapes_name_the_kernel_form():
    # block -1: the Rys kernels (FP64 J/K from L = 6 and gradient from L = 4 in a small molecule, mixed from
    # L = 7) or the cooperative ones that coop_min_l asks for; the others have a block of their own
    mol = H.Molecule.from_xyz(golden("h2o.xyz"), "cc-pvdz")
    L = lambda s: sum(int(x) for x in s["cls"])  # noqa: E731
    ctx = H.GpuContext(mol)
    for precision, jk_min, grad_min in ((H.FP64, 6, 4), (H.MIXED, 7, 7)):
        ctx.set_precision(precision)
        for s in ctx.launch_shapes():
            if L(s) >= jk_min or L(s) < 4 or precision == H.MIXED:
                assert (s["jk"][1] == -1) == (L(s) >= jk_min), s
            assert (s["grad"][1] == -1) == (L(s) >= grad_min), s
    assert all((s["jk"][1] == -1) == (L(s) >= 5) for s in H.GpuContext(mol, precision=H.MIXED, coop_min_l=5).launch_shapes())
