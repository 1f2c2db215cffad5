"""GPU test of the ensemble autotuner: it offers, and reports, launch shapes only for grids whose kernels
read them.  Group transforms of FP32 grids of 64 to 256 points: 2, 4 or 8 waves per block, each direction by
its own size; the generic LDS kernels (here the forward y-FFT of a 32-point grid with few columns, and
8-point grids): the column tile and 64 to 256 threads; every other grid keeps the kernels' own choice, 0."""
import pytest

pytestmark = pytest.mark.gpu

TILES, THREADS, GROUP = {1, 2, 4, 8, 16}, {64, 128, 256}, {128, 256, 512}


def _cols(n):
    return {w * 512 // n for w in (2, 4, 8)}


@pytest.mark.parametrize("precision,M,N,cols,threads", [
    ("f64", 64, 64, {0}, {0}), ("f64", 32, 32, TILES, {0}), ("f64", 512, 128, {0}, {0}), ("f64", 8, 8, TILES, THREADS),
    ("f32", 64, 128, _cols(128), GROUP), ("f32", 64, 512, {0}, GROUP), ("f32", 512, 64, _cols(64), {0}),
    ("f32", 128, 32, TILES, GROUP), ("f32", 1024, 64, _cols(64), {0}), ("f32", 512, 512, {0}, {0}),
])
def test_tuned_shapes_are_ones_that_a_kernel_reads(precision, M, N, cols, threads):
    print(f"case: tune {precision} {M}x{N}", flush=True)
    from sdc_amd import Ensemble
    from sdc_amd.initial import random_theta
    L = 3
    with Ensemble([dict(M=M, N=N, L=L, Lx=4.0, Ly=4.0, Ra=1e4, Pr=0.7, dt=1e-6, precision=precision)]) as E:
        E.members[0].set_state(*random_theta(M, N, L, seed=1, amp=1e-3))
        tx, th, ms = E.tune()[0]
    assert tx in cols and (th in threads or th == 0), (tx, th)
    assert ms > 0
