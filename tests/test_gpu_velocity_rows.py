"""GPU test of the velocity grid (sdc_amd/csrc/rbc_velocity.hip k_vel_levels, k_vel_rows_w, k_vel_rows) at
every row length, and of the RK4 tracer on its interleaved grid there, against the FP64 restatement;
height counts that are no multiple of a thread's four.

Tolerance: as the other velocity tests, 2e-6 of the field's maximum; tracer positions 2e-5 after three
steps of a flow of unit speed that moves a particle by a fraction of a cell."""
import numpy as np
import pytest

from oracle import velocity as V
from tests.helpers import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,L,nz", [(8, 8, 3, 1), (16, 8, 5, 2), (32, 16, 8, 5), (64, 32, 4, 3), (128, 16, 8, 4),
                                      (256, 16, 9, 7), (512, 16, 3, 6), (1024, 8, 2, 2)])
def test_velocity_grid_and_rk4(M, N, L, nz):
    print(f"case: velocity rows {M}x{N}x{L} nz={nz}", flush=True)
    from sdc_amd import Stepper, Tracer
    Lx, Ly = 4.0, 3.0
    st = random_state(M, N, L, seed=M + nz, amp=5e-2)
    kx, ky = V.wavenumbers(M, N, Lx, Ly)
    KX, KY = np.meshgrid(kx, ky)
    damp = np.exp(-0.3 * np.sqrt(KX ** 2 + KY ** 2))
    st = [a * damp[None] for a in st[:3]] + list(st[3:])
    z = V.linspace_levels()[:: max(1, 128 // nz)][:nz]
    full = V.velocity_grid(st, M, N, Lx, Ly, V.linspace_levels())
    umax = max(np.abs(c).max() for c in full)
    st = [a / umax for a in st]
    full = [c / umax for c in full]
    n, dt = 500, 1e-3
    with Stepper(M, N, L, Lx, Ly, 2e4, 0.7, 1e-3, precision="f32") as G:
        G.set_state(*st)
        got = G.velocity_grid(z)
        T = Tracer(G, n, buffer_size=8, mode="rk4_trilinear", seed=2)
        T.init_positions("random")
        x, y, zz = (a.astype(np.float64) for a in T.positions())
        for _ in range(3):
            T.step_particles(dt)
        out = T.positions()
        T.close()
    for a, b in zip(got, V.velocity_grid(st, M, N, Lx, Ly, z)):
        assert np.abs(a - b).max() < 2e-6 * np.abs(b).max(), np.abs(a - b).max() / np.abs(b).max()
    for _ in range(3):
        x, y, zz = V.rk4_step(full, Lx, Ly, x, y, zz, dt)
    err = max(np.abs(a - b).max() for a, b in zip(out, (x, y, zz)))
    assert err < 2e-5, err
