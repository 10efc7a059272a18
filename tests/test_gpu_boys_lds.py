"""The Boys functions of the LDS table against their series in 60-digit arithmetic, at the table's rows and
midpoints, its end, the temperatures from which e^-T is dropped, and at random.

Tolerance: 1e-15 relative for F_0 and 1e-14 up to F_4 (nine Taylor terms, or four steps of the upward
recursion from T = 36, of a few roundings each)."""
from decimal import Decimal, getcontext

import numpy as np
import pytest

import hfscf_amd as H
from conftest import golden

pytestmark = pytest.mark.gpu


def _boys(m, T):
    getcontext().prec = 60
    T = Decimal(float(T))
    t = s = Decimal(1) / (2 * m + 1)
    k = 0
    while abs(t) > Decimal("1e-45") * s:
        k += 1
        t = t * 2 * T / (2 * m + 2 * k + 1)
        s += t
    return s * (-T).exp()


@pytest.mark.parametrize("m", [0, 1, 2, 3, 4])
def test_boys_lds_table(m):
    ctx = H.GpuContext(H.Molecule.from_xyz(golden("h2o.xyz"), "sto-3g"))
    rng = np.random.default_rng(m)
    edge = [0.0, 1e-14, 1e-8, 0.0625, 0.0624999, 0.125, 35.9374, 35.9376, 35.99999, 36.0, 36.01]
    edge += [39.0 + 3 * k + d for k in range(1, 5) for d in (-1e-9, 0.0, 0.1)]
    T = np.concatenate([edge, rng.uniform(0, 36, 200), rng.uniform(36, 80, 60)])
    F = ctx.boys(m, T, closed_form=2)
    err = np.zeros(m + 1)
    for i, t in enumerate(T):
        for k in range(m + 1):
            ref = _boys(k, t)
            err[k] = max(err[k], float(abs(Decimal(float(F[i, k])) - ref) / ref))
    print(f"F_0..F_{m}: max relative errors {err}", flush=True)
    assert err[0] < 1e-15 and err.max() < 1e-14
