"""The per-mode tau solves at the edges of their launch shapes, against the FP64 oracle (dense LU).

The solves give a mode 16, 32 or 64 lanes and each lane one, two or four degrees per parity, so
the sizes run over both sides of every change, the smallest and the largest.  "u" and "psi" are the
two recursions: psi where 1/(c nu (2/Lz)^2) exceeds 16 N^2 (N < 64) or 256 N^2.  RK222 has right-hand
sides in the continuity rows, SBDF2 has none.

Tolerance, set from the oracle: its LU solves of these systems are good to 4e-14 at N = 128
(condition 3e7) and 3e-12 at N = 450 (1e10), so rounding grows like N^4: 1e-12 up to N = 64 (the
bound of the other step tests) and 1e-12 (N / 64)^4 above.  p carries the rounding of u / dt, and a tau
is what an equation row leaves over, whose terms reach (1/dt + nu (2/Lz)^2 N^4) |x|.
"""
import numpy as np
import pytest

from tests.test_gpu_channel import random_state
from tests.test_gpu_channel3d import random_state3

pytestmark = pytest.mark.gpu

FORMS = {"u": (0.1, 5e-2), "psi": (3e-3, 2e-6)}  # kappa = nu, dt


def check(s, ref, fields, p, ntau, N, nu, dt):
    tol = 1e-12 * max(1.0, N / 64.0) ** 4
    size = max(np.abs(ref.get(v)).max() for v in fields)
    for v in fields:
        assert np.abs(s.get(v) - ref.get(v)).max() <= tol * max(np.abs(ref.get(v)).max(), 1e-3 * size), v
    pmax = np.abs(ref.get(p)).max()
    assert np.abs(s.get(p) - ref.get(p)).max() <= tol * max(pmax, size / dt), "p"
    rows = (1.0 / dt + 4.0 * nu * N ** 4) * size + 2.0 * N ** 2 * pmax
    for t in range(ntau):
        assert np.abs(s.tau(t) - ref.tau(t)).max() <= tol * rows, ("tau", t)


@pytest.mark.parametrize("ts", ["SBDF2", "RK222"])
@pytest.mark.parametrize("form", ["u", "psi"])
@pytest.mark.parametrize("N", [4, 5, 6, 31, 33, 63, 64, 65, 128, 129, 256, 257, 512])
def test_tau_solve_2d(gpu, oracle, N, form, ts):
    print(f"tau solve 2-D N={N} {form} {ts}", flush=True)
    nx, Lx, Lz = (16 if N <= 257 else 8), 4.0, 1.0
    nu, dt = FORMS[form]
    st = random_state(oracle, nx, N, Lx, Lz, seed=N)
    ref = oracle.RBC2D(nx, N, Lx, Lz, nu, nu, dt, ts)
    s = gpu.chan(nx, N, Lx, Lz, nu, nu, dt, stepper={"RK222": 0, "SBDF2": 2}[ts])
    for v, c in st.items():
        ref.set(v, c)
        s.set(v, c)
    ref.step(1)
    s.step(1)
    check(s, ref, (oracle.RBC_B, oracle.RBC_UX, oracle.RBC_UZ), oracle.RBC_P, 7, N, nu, dt)
    s.close()


@pytest.mark.parametrize("N,form,ts", [(N, form, ts) for N in (4, 5, 31, 32, 33, 64, 65, 128, 129)
                                       for form in ("u", "psi") for ts in ("SBDF2", "RK222")] + [(256, "u", "SBDF2")])
def test_tau_solve_3d(gpu, oracle, N, form, ts):
    print(f"tau solve 3-D N={N} {form} {ts}", flush=True)
    nx, ny, Lx, Ly, Lz = 8, 8, 4.0, 3.0, 1.0
    nu, dt = FORMS[form]
    st, _ = random_state3(oracle, nx, ny, N, Lx, Ly, Lz, seed=N)
    ref = oracle.RBC3D(nx, ny, N, Lx, Ly, Lz, nu, nu, dt, ts)
    s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, nu, nu, dt, stepper={"RK222": 0, "SBDF2": 2}[ts])
    for v, c in st.items():
        ref.set(v, c)
        s.set(v, c)
    ref.step(1)
    s.step(1)
    fields = (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ)
    check(s, ref, fields, oracle.RBC3_P, 9, N, nu, dt)
    s.close()
