"""GPU test of the group transforms (rbc_device.hpp fft_group and the row and column kernels on it)
at every size and precision they take, against the generic LDS Stockham kernels: the nonlinear
term of a random state in every kept mode, oblong grids so that each size runs in x beside another
in y, with ragged last blocks (odd L, levels times rows not a multiple of a block's rows).

Tolerance: both forms round each butterfly once per pass; a 2-D transform pair has at most 20 + 20
radix-2 stages, so the relative difference in the largest entry stays within about 40 eps times the
k^2 weights' cancellation (a few tens): 1e-12 in FP64, 2e-5 in FP32 (the bound the FP32 64..256-point
kernels have been held to).
"""
import os

import numpy as np
import pytest

from sdc_amd.initial import kept_mask, random_theta

pytestmark = pytest.mark.gpu

SIZES = [("f32", m, n) for m, n in ((16, 512), (32, 16), (512, 32), (1024, 16), (16, 1024), (256, 512), (512, 64))] + \
        [("f64", m, n) for m, n in ((16, 512), (32, 16), (64, 32), (128, 64), (256, 128), (512, 256), (512, 512))]


@pytest.mark.parametrize("prec,M,N", SIZES)
def test_group_against_generic(prec, M, N):
    print(f"case: group FFT {prec} {M}x{N}", flush=True)
    import sdc_amd
    L = 3
    st = [random_theta(M, N, L, seed=s, amp=a)[0] for s, a in ((1, 1.0), (2, 1e-2), (3, 1e-1))]
    r = np.random.default_rng(4)
    st += [r.normal(size=L).astype(np.complex128), r.normal(size=L).astype(np.complex128)]
    keep = kept_mask(M, N)
    with sdc_amd.Stepper(M, N, L, 4.0, 2.5, 1e5, 0.7, 1e-4, precision=prec) as G:
        group = G.calculate_nonlinear(*st)
        os.environ["RBC_GENERIC_FFT"] = "1"
        try:
            generic = G.calculate_nonlinear(*st)
        finally:
            del os.environ["RBC_GENERIC_FFT"]
    for a, b in zip(group, generic):
        a, b = (x[:, keep] if x.ndim == 3 else x for x in (a, b))
        assert np.abs(a - b).max() <= (1e-12 if prec == "f64" else 2e-5) * np.abs(b).max()
