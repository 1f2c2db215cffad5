"""GPU test of the group update (sdc_amd/csrc/rbc_update.hip): inverse B, the implicit operator and
whole steps against the FP64 oracle at vertical resolutions around the kernels' edges (16, 32 and 48
modes, odd L with classes of unequal size, the smallest and the largest L), on a grid whose waves take
one mode each and on one whose waves take up to four.

Tolerance: the 32-mode tests hold inverse B to 1e-14 and the implicit operator to 1e-13 in FP64 (2e-6
in FP32).  The condition of the class matrices grows like the fourth power of the vertical wave number,
by 16 from 32 to 64 modes: 2e-12 and 4e-5 for every L.  Steps: 1e-10 and 1e-4 as the other step tests.
"""
import numpy as np
import pytest

from oracle import oracle as O
from sdc_amd.initial import kept_mask
from tests.helpers import random_state, rel_err

pytestmark = pytest.mark.gpu

LS = [1, 2, 15, 16, 17, 32, 33, 47, 48, 49, 63, 64]


def _check(out, ref, keep, tol):
    for i, (a, b) in enumerate(zip(out, ref)):
        a, b = (x[:, keep] if x.ndim == 3 else x for x in (a, b))
        if np.abs(b).max() == 0:
            assert np.abs(a).max() == 0, i
        else:
            assert rel_err(a, b) < tol, (i, rel_err(a, b))


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("M,N,L", [(32, 16, L) for L in LS] + [(256, 256, 9), (256, 256, 33)])
def test_operators_vs_oracle(prec, M, N, L):
    print(f"case: update operators {prec} {M}x{N}x{L}", flush=True)
    import sdc_amd
    cfg = (M, N, L, 3.3, 4.1, 2e4, 0.7, 2e-4)
    st = random_state(M, N, L, seed=L, amp=1e-2, decay=0.05)
    keep = kept_mask(M, N)
    o = O.Stepper(*cfg, nthreads=8)
    ref = o.inverse_B(*st), o.implicit(*st)
    with sdc_amd.Stepper(*cfg, precision=prec) as G:
        out = G.calculate_inverse(*st), G.calculate_implicit(*st)
    for a, b in zip(out, ref):
        _check(a, b, keep, 2e-12 if prec == "f64" else 4e-5)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("L", LS[1:])  # at L = 1 the products of F and G vanish by symmetry
def test_steps_vs_oracle(prec, L):
    print(f"case: update steps {prec} L={L}", flush=True)
    import sdc_amd
    M, N = 32, 16
    cfg = (M, N, L, 3.3, 4.1, 2e4, 0.7, 1e-4)
    st = random_state(M, N, L, seed=L, amp=1e-2, decay=0.05)
    keep = kept_mask(M, N)
    o = O.Stepper(*cfg, nthreads=8)
    o.set_state(*st)
    o.step(3)
    with sdc_amd.Stepper(*cfg, precision=prec) as G:
        G.set_state(*st)
        G.step_time(3)
        out = G.get_state()
    _check(out, o.get_state(), keep, 1e-10 if prec == "f64" else 1e-4)
    for a in out[:3]:  # make_real: the kx = 0 column is Hermitian bit for bit, (0, 0) real
        assert not a[:, 0, 0].imag.any()
        for r in range(1, N // 2):
            assert np.array_equal(a[:, r, 0], np.conj(a[:, N - r, 0])), r
