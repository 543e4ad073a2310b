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

from tarang_amd import _lib
from tarang_amd._lib import CHAN3_B, CHAN3_P, CHAN3_UX, CHAN3_UY, CHAN3_UZ, CHAN_B, CHAN_P, CHAN_UX, CHAN_UZ
from tests.conftest import relerr
from tests.tau_reference import Mode
from tests.test_gpu_channel import random_state
from tests.test_gpu_channel3d import random_state3
from tests.test_gpu_channel_group import make_group

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


SCALE = 2.0 ** -600  # products of two state values underflow to zero: a step is its linear solve alone


def spectrum(rng, shape, N):
    """Random complex coefficients, falling off as a resolved field's do."""
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * np.exp(-np.arange(N) * 30.0 / N)


def parts(c):
    return np.stack([c.real, c.imag], axis=-1)


def check_precision(err, lu, what):
    """Geometric means over the modes: within four times a dense FP64 elimination of the same systems (the
    means of the two differ by up to 3.5 over the sizes here) plus a floor of 8 eps for small N."""
    for f in err:
        a, b = (float(np.exp(np.mean(np.log(np.maximum(v[f], 1e-18))))) for v in (err, lu))
        print(f"  {what} {f}: {a:.1e}, dense FP64 {b:.1e}", flush=True)
        assert a <= 4.0 * b + 8 * 2.3e-16, (what, f, a, b)


@pytest.mark.parametrize("Lx", [40.0, 1.0])  # kh from 0.08 to 0.6 s, from 3 to 22 s: uz from E1, and both sides of the change
@pytest.mark.parametrize("mr", [0.05, 1.0, 30.0, 1000.0])  # alpha/beta of the velocity lines over N^2
@pytest.mark.parametrize("N", [16, 33, 97, 128])
def test_tau_solve_precision_2d(gpu, N, mr, Lx):
    """A linear FP64 step against long double: no further off than a dense FP64 elimination."""
    print(f"tau solve precision 2-D N={N} m/N2={mr} Lx={Lx}", flush=True)
    nx, Lz, dt = 16, 1.0, 2.0 ** -10  # a power of two: the right-hand side is the state itself
    nu = 1.0 / (mr * N * N * dt * 4.0)
    rng = np.random.default_rng(N)
    st = {v: spectrum(rng, (nx // 2 + 1, N), N) for v in (CHAN_B, CHAN_UX, CHAN_UZ)}
    for c in st.values():
        c[[0, -1]] = c[[0, -1]].real
    s = gpu.chan(nx, N, Lx, Lz, nu, nu, dt, stepper=4, b_bottom=0.0, b_top=0.0)
    for v, c in st.items():
        s.set(v, c * SCALE)
    s.step(1)
    got = {f: s.get(v) / SCALE for f, v in (("b", CHAN_B), ("u", CHAN_UX), ("uz", CHAN_UZ), ("p", CHAN_P))}
    s.close()
    err, lu = ({f: [] for f in got} for _ in range(2))
    for m in range(nx // 2):
        rhs = [parts(st[CHAN_B][m]), parts(-1j * st[CHAN_UX][m]), parts(st[CHAN_UZ][m])]
        args = (N, 2 * np.pi * m / Lx, dt, nu, nu, 2.0 / Lz)
        ref, dense = Mode(*args)(*rhs), Mode(*args, dtype=np.float64)(*rhs)
        for f in got:
            size = np.linalg.norm(ref[f].astype(float))
            if m == 0 and f == "uz":
                assert np.abs(got[f][0]).max() == 0.0  # E1 at kh = 0
                continue
            g = parts(-1j * got[f][m] if f == "u" else got[f][m])
            err[f].append(float(np.linalg.norm((g - ref[f]).astype(float)) / size))
            lu[f].append(float(np.linalg.norm((dense[f] - ref[f]).astype(float)) / size))
    check_precision(err, lu, "2-D")


@pytest.mark.parametrize("N,mr", [(33, 1000.0), (64, 30.0), (97, 1.0), (128, 30.0)])
def test_tau_solve_precision_3d(gpu, N, mr):
    print(f"tau solve precision 3-D N={N} m/N2={mr}", flush=True)
    nx, ny, Lx, Ly, Lz, dt = 8, 8, 40.0, 1.5, 1.0, 2.0 ** -10
    nu = 1.0 / (mr * N * N * dt * 4.0)
    rng = np.random.default_rng(N)
    fields = (CHAN3_B, CHAN3_UX, CHAN3_UY, CHAN3_UZ)
    st = {v: spectrum(rng, (nx // 2 + 1, ny, N), N) for v in fields}
    s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, nu, nu, dt, stepper=4, b_bottom=0.0, b_top=0.0)
    for v, c in st.items():
        s.set(v, c * SCALE)
    s.step(1)
    o = {v: s.get(v) / SCALE for v in fields + (CHAN3_P,)}
    s.close()
    err, lu = ({f: [] for f in ("b", "u", "v", "uz", "p")} for _ in range(2))
    for m in range(1, nx // 2):  # the kx = 0 and kx = Nx/2 lines are projected onto real fields
        for n in list(range(ny // 2)) + list(range(ny // 2 + 1, ny)):
            kx, ky = 2 * np.pi * m / Lx, 2 * np.pi * (n if n < ny // 2 else n - ny) / Ly
            kh = np.hypot(kx, ky)
            turn = lambda x, y: (parts(-1j * (kx * x + ky * y) / kh), parts(-1j * (-ky * x + kx * y) / kh))  # noqa: E731
            rx, ry = turn(st[CHAN3_UX][m, n], st[CHAN3_UY][m, n])
            rhs = [parts(st[CHAN3_B][m, n]), rx, parts(st[CHAN3_UZ][m, n]), ry]
            args = (N, kh, dt, nu, nu, 2.0 / Lz)
            if len(err["b"]) and n % 2:  # every other mode: the reference is slow
                continue
            ref, dense = Mode(*args)(*rhs), Mode(*args, dtype=np.float64)(*rhs)
            u, v = turn(o[CHAN3_UX][m, n], o[CHAN3_UY][m, n])
            got = {"b": parts(o[CHAN3_B][m, n]), "u": u, "v": v, "uz": parts(o[CHAN3_UZ][m, n]), "p": parts(o[CHAN3_P][m, n])}
            for f in got:
                size = np.linalg.norm(ref[f].astype(float))
                err[f].append(float(np.linalg.norm((got[f] - ref[f]).astype(float)) / size))
                lu[f].append(float(np.linalg.norm((dense[f] - ref[f]).astype(float)) / size))
    check_precision(err, lu, "3-D")


def zero_pivot(N, g):
    """A negative m at which elimination from the top degree down without pivoting meets a zero pivot."""
    def smallest(m):  # the pivots' running product changes sign where one of them does
        top = (N - 1) % 2 == g
        an, out = 0.0, []
        for j in range((N + 1 - g) // 2 - (2 if top else 1), 0, -1):
            k = 2 * j + g
            lo = (2.0 if k == 2 else 1.0) / (4.0 * k * (k - 1))
            if k == N - 2:
                den = 1.0 + m * lo * (0.5 if k == 2 else 1.0)
            else:
                den = 1.0 + m / (2.0 * (k * k - 1.0)) - (0.0 if k == N - 3 else m / (4.0 * k * (k + 1)) * an)
            an = m * lo / den
            out.append(den)
        return min(out)

    a = -1.0
    while smallest(2 * a) > 0:
        a *= 2
    b = 2 * a
    for _ in range(200):
        c = 0.5 * (a + b)
        a, b = (c, b) if smallest(c) > 0 else (a, c)
    return a


ANY_SIGN = [("zero", "zero"), (-1e-2, -3e-3), (-1e-2, 1e-3), (1e-3, -1e-3)]  # kappa, nu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kappa,nu", ANY_SIGN)
@pytest.mark.parametrize("N", [9, 33, 64, 128])
def test_tau_solve_any_sign_2d(gpu, N, kappa, nu, dtype):
    """Negative diffusivities, "zero" among them: a value that brings a pivot of the unpivoted recursion to
    zero in the mean mode.  Against long double: 1e-10 (a line is good to 1e-13, and uz is what up to a
    hundredth of the pressure gradient's size leaves), 1e-6 for the rounding of an FP32 result."""
    print(f"tau solve any sign 2-D N={N} kappa={kappa} nu={nu} {dtype.__name__}", flush=True)
    nx, Lx, Lz, dt = 8, 4.0, 1.0, 2.0 ** -10
    if kappa == "zero":
        kappa = nu = 1.0 / (zero_pivot(N, N % 2) * dt * 4.0)
    scale, tol = (SCALE, 1e-10) if dtype == np.float64 else (2.0 ** -75, 1e-6)
    rng = np.random.default_rng(N)
    st = {v: spectrum(rng, (nx // 2 + 1, N), N).astype(np.complex64 if dtype == np.float32 else complex)
          for v in (CHAN_B, CHAN_UX, CHAN_UZ)}
    for c in st.values():
        c[[0, -1]] = c[[0, -1]].real
    s = gpu.chan(nx, N, Lx, Lz, kappa, nu, dt, stepper=4, dtype=dtype, b_bottom=0.0, b_top=0.0)
    for v, c in st.items():
        s.set(v, c * c.real.dtype.type(scale))
    s.step(1)
    got = {f: s.get(v).astype(complex) / scale for f, v in (("b", CHAN_B), ("u", CHAN_UX), ("uz", CHAN_UZ), ("p", CHAN_P))}
    s.close()
    for m in range(nx // 2):
        st64 = {v: c[m].astype(complex) for v, c in st.items()}
        ref = Mode(N, 2 * np.pi * m / Lx, dt, kappa, nu, 2.0 / Lz)(
            parts(st64[CHAN_B]), parts(-1j * st64[CHAN_UX]), parts(st64[CHAN_UZ]))
        for f in got:
            g = parts(-1j * got[f][m] if f == "u" else got[f][m])
            size = max(float(np.linalg.norm(ref[f].astype(float))), 1e-3 * float(np.linalg.norm(ref["u"].astype(float))))
            e = float(np.linalg.norm((g - ref[f]).astype(float))) / size
            assert e <= tol, (m, f, e)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ts", ["SBDF2", "RK222"])
@pytest.mark.parametrize("N", [6, 33, 256])
def test_tau_solve_any_sign_steps(gpu, oracle, N, ts, dtype):
    """Steps with negative diffusivities against the oracle's dense LU, in 2-D, 3-D and as a group member.  The
    oracle multiplies a relative change of the state by up to 40 here (400 in one FP64 case): 40 times the 1e-5
    of other FP32 steps, and 1e-9 for their 1e-12."""
    print(f"tau solve any sign steps N={N} {ts} {dtype.__name__}", flush=True)
    tol = 1e-9 if dtype == np.float64 else 4e-4
    kappa, nu, dt, code = -1e-3, -2e-3, 1e-3, {"RK222": 0, "SBDF2": 2}[ts]
    st = random_state(oracle, 16, N, 4.0, 1.0, seed=N)
    pair = [oracle.RBC2D(16, N, 4.0, 1.0, kappa, nu, dt, ts)]
    pair += [gpu.chan(16, N, 4.0, 1.0, kappa, nu, dt, stepper=code, dtype=dtype) for _ in range(2)]
    other = [gpu.chan(16, 33, 4.0, 1.0, 1e-3, 1e-3, dt, stepper=code, dtype=dtype) for _ in range(2)]
    for s in pair:
        for v, c in st.items():
            s.set(v, c)
    for s in other:
        for v, c in random_state(oracle, 16, 33, 4.0, 1.0, seed=1).items():
            s.set(v, c)
    ref, s, member = pair
    ref.step(2)
    s.step(2)
    g = make_group([member, other[0]])
    _lib.call("tarang_chan_group_step", g, 2)
    gpu.sync()
    other[1].step(2)
    for v in (oracle.RBC_B, oracle.RBC_UX, oracle.RBC_UZ):
        assert relerr(s.get(v), ref.get(v)) < tol, v
        assert np.array_equal(member.get(v), s.get(v)) and np.array_equal(other[0].get(v), other[1].get(v))
    _lib.call("tarang_chan_group_destroy", g)
    for x in pair[1:] + other:
        x.close()
    if N > 64:
        return
    st, _ = random_state3(oracle, 8, 8, N, 4.0, 3.0, 1.0, seed=N)
    ref = oracle.RBC3D(8, 8, N, 4.0, 3.0, 1.0, kappa, nu, dt, ts)
    s = gpu.chan3(8, 8, N, 4.0, 3.0, 1.0, kappa, nu, dt, stepper=code, dtype=dtype)
    for v, c in st.items():
        ref.set(v, c)
        s.set(v, c)
    ref.step(2)
    s.step(2)
    for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ):
        assert relerr(s.get(v), ref.get(v)) < tol, v
    s.close()


def test_tau_solve_without_diffusion_is_singular(gpu):
    """Zero, and a diffusivity that FP64 cannot divide by."""
    for kappa, nu in ((0.0, 1e-3), (1e-3, 0.0), (1e-320, 1e-3), (1e-3, -1e-320)):
        for make in (lambda: gpu.chan(16, 9, 4.0, 1.0, kappa, nu, 1e-3), lambda: gpu.chan3(8, 8, 9, 4.0, 4.0, 1.0, kappa, nu, 1e-3)):
            with pytest.raises(_lib.TarangError) as e:
                make()
            assert e.value.code == _lib.ERR_SINGULAR and "singular" in str(e.value)
