"""The per-mode tau solves at the edges of their launch shapes and of their recursions' ranges.

A step whose state products underflow is its linear solve alone; it is compared with long-double
elimination of the same systems (tests/tau_reference.py), field by field and tau by tau.

The solves give a mode 16, 32 or 64 lanes and each lane one, two or four degrees per parity, so the
sizes run over both sides of every change, the smallest and the largest.  m = alpha/beta of the lines
chooses the recursion (u-form, and psi-form above N^2/8; FP32 above 16 N^2, from 64 degrees on 256 N^2),
kh the source of uz (E1 up to min(16, N/4) * 2/Lz, E3z above): both sides of each, and beyond.
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

EPS = 2.3e-16
DT = 2.0 ** -10  # a power of two: the right-hand side of an SBDF1 step is the state itself
SBDF1, RK222 = 4, 0
TAUS2 = ("tau_p", "tau_b1", "tau_b2", "tau_u1", "tau_u1z", "tau_u2", "tau_u2z")
TAUS3 = ("tau_p", "tau_b1", "tau_b2", "tau_u1", None, "tau_u1z", "tau_u2", None, "tau_u2z")  # None: the y components

SCALE = 2.0 ** -600  # products of two state values underflow to zero: a step is its linear solve alone


def spectrum(rng, shape, N, decay=lambda k, N: np.exp(-k * 30.0 / N)):
    """Random complex coefficients, falling off as a resolved field's do."""
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * decay(np.arange(N), N)


def square(k, N):
    """A slow fall-off, under which every tau is well above rounding."""
    return 1.0 / (1.0 + k) ** 2


def parts(c):
    return np.stack([c.real, c.imag], axis=-1)


def check_precision(err, lu, what, factor=4.0, floor=8):
    """Geometric means over the modes: within four times a dense FP64 elimination of the same systems (the
    means of the two differ by up to 3.5 over the sizes here) plus a floor of 8 eps for small N."""
    for f in err:
        a, b = (float(np.exp(np.mean(np.log(np.maximum(v[f], 1e-18))))) for v in (err, lu))
        print(f"  {what} {f}: {a:.1e}, dense FP64 {b:.1e}", flush=True)
        assert a <= factor * b + floor * EPS, (what, f, a, b)


def norm(v):
    return float(np.linalg.norm(np.asarray(v, float)))


def tau_scales(N, kh, c, kappa, nu, s, rhs, ref):
    """What one rounding of the largest term of a tau's own equation row amounts to in that tau, over eps: a
    T_{N-1} lift takes row N - 1 over c, a D T_{N-1} lift row N - 2 over c diff s 2 (N - 1)."""
    b = (1 + abs(c * kappa * kh * kh)) * norm(ref["b"]) + norm(rhs[0])
    u = ((1 + abs(c * nu * kh * kh)) * max(norm(ref["u"]), norm(ref["uz"])) + max(norm(rhs[1]), norm(rhs[2])) +
         c * max(kh, s) * norm(ref["p"]) + c * norm(ref["b"]))
    d = lambda diff: c * abs(diff) * s * 2 * (N - 1)  # noqa: E731
    return {"tau_b1": b / d(kappa), "tau_b2": b / c, "tau_u1": u / d(nu), "tau_u2": u / c, "tau_u1z": u / d(nu),
            "tau_u2z": u / c}


def check_taus(got, ref, scales):
    """Within 64 roundings of the tau's own row (a dense FP64 elimination: up to 10); True per tau that stands
    a hundred times above that."""
    live = {}
    for t, s in scales.items():
        e, size = norm(got[t] - ref[t]), norm(ref[t])
        assert e <= 64 * EPS * s, (t, e / s, size / s)
        live[t] = size > 6400 * EPS * s
    return live


def step_2d(gpu, N, kappa, nu, Lx, st, stepper=SBDF1, dtype=np.float64, scale=None):
    """Fields and taus per mode after one linear step from st (B, UX, UZ); u and its taus over i."""
    scale = scale or (SCALE if dtype == np.float64 else 2.0 ** -75)
    s = gpu.chan(2 * (st[CHAN_B].shape[0] - 1), N, Lx, 1.0, kappa, nu, DT, stepper=stepper, dtype=dtype, b_bottom=0.0,
                 b_top=0.0)
    for v, c in st.items():
        s.set(v, c * c.real.dtype.type(scale))
    s.step(1)
    o = {f: s.get(v).astype(complex) / scale for f, v in (("b", CHAN_B), ("u", CHAN_UX), ("uz", CHAN_UZ), ("p", CHAN_P))}
    o.update({t: s.tau(i).astype(complex) / scale for i, t in enumerate(TAUS2)})
    s.close()
    return [{f: parts(-1j * v[m] if f in ("u", "tau_u1", "tau_u2") else v[m]) for f, v in o.items()}
            for m in range(len(o["b"]))]


def state_2d(N, nx, decay, dtype=complex):
    rng = np.random.default_rng(N)
    st = {v: spectrum(rng, (nx // 2 + 1, N), N, decay).astype(dtype) for v in (CHAN_B, CHAN_UX, CHAN_UZ)}
    for c in st.values():
        c[[0, -1]] = c[[0, -1]].real
    return st


def rhs_2d(st, m):
    return [parts(st[CHAN_B][m].astype(complex)), parts(-1j * st[CHAN_UX][m].astype(complex)),
            parts(st[CHAN_UZ][m].astype(complex))]


# alpha/beta over N^2 of the buoyancy and the velocity lines: both sides of the psi-form's start, one on each
# side of it, production convection, and a thin diffusion layer that the grid does not resolve
LINES = [(0.12, 0.12), (0.13, 0.13), (0.1, 10.0), (30.0, 0.1), (30.0, 30.0), (1e4, 1e4)]


def diffusivity(mr, N):
    return 1.0 / (mr * N * N * DT * 4.0)


# short boxes: the pressure lines' psi-form ((kh/s)^2 > N^2/8)
BOXES = [(N, 4.0) for N in (4, 5, 6, 31, 32, 33, 63, 64, 65, 128, 129, 256, 257)] + [(33, 0.05), (128, 0.03)]


@pytest.mark.parametrize("N,Lx,mb,mu", [b + m for b in BOXES for m in LINES] + [(512, 4.0) + m for m in LINES[:2]])
def test_tau_solve_2d(gpu, N, Lx, mb, mu):
    print(f"tau solve 2-D N={N} Lx={Lx} m/N2={mb},{mu}", flush=True)
    nx, kappa, nu = 8, diffusivity(mb, N), diffusivity(mu, N)
    st = state_2d(N, nx, square)
    got = step_2d(gpu, N, kappa, nu, Lx, st)
    err, lu = ({f: [] for f in ("b", "u", "uz", "p")} for _ in range(2))
    live = {}
    for m in ([0, 1, 2, 3] if N < 256 else [1, 3] if N < 512 else [1]):
        args, rhs = (N, 2 * np.pi * m / Lx, DT, kappa, nu, 2.0), rhs_2d(st, m)
        ref, dense = Mode(*args)(*rhs), Mode(*args, dtype=np.float64)(*rhs)
        for f in err:
            if m == 0 and f == "uz":
                assert not got[m][f].any()  # E1 at kh = 0
                continue
            err[f].append(norm(got[m][f] - ref[f]) / norm(ref[f]))
            lu[f].append(norm(dense[f] - ref[f]) / norm(ref[f]))
        scales = tau_scales(*args, rhs, ref)
        if m == 0:
            scales.pop("tau_u1z")  # zero, as E1's right-hand side
        for t, on in check_taus(got[m], ref, scales).items():
            live[t] = live.get(t, False) or on
    check_precision(err, lu, "2-D", factor=8.0, floor=16)
    assert all(live.values()), live


@pytest.mark.parametrize("N", [4, 5, 33, 64, 129, 256])
@pytest.mark.parametrize("mr", [0.12, 0.13, 30.0])
def test_tau_solve_rk_2d(gpu, N, mr):
    """A linear RK222 step ends on its second stage's solution x2 = (M + c L)^-1 (x0 - dt (1 - g) L x1), in exact
    arithmetic; the device forms it from L x2, taus and p among it, so a wrong tau shows in the state's top
    degrees.  1e-12: L x rounds at c nu s^2 sum k^3 |x_k| eps = N^2/(2 m) eps here, the solves at 1e-14."""
    print(f"tau solve 2-D RK222 N={N} m/N2={mr}", flush=True)
    g = 1 - 2 ** -0.5
    nx, Lx, nu = 8, 4.0, diffusivity(mr, N) / g
    st = state_2d(N, nx, square)
    got = step_2d(gpu, N, nu, nu, Lx, st, stepper=RK222)
    for m in (1, 3):
        rhs = rhs_2d(st, m)
        solve = Mode(N, 2 * np.pi * m / Lx, g * DT, nu, nu, 2.0)
        x1 = solve(*rhs)
        x2 = solve(*[r - (1 - g) / g * (r - x1[f]) for r, f in zip(rhs, ("b", "u", "uz"))])
        for f in ("b", "u", "uz"):
            e = norm(got[m][f] - x2[f]) / norm(x2[f])
            assert e < 1e-12, (m, f, e)
            assert g * DT * norm(x2["tau_b2" if f == "b" else "tau_u2"]) > 1e-9 * norm(x2[f])


@pytest.mark.parametrize("N", [4, 5, 31, 33, 64, 65, 128, 129, 256, 257])
@pytest.mark.parametrize("side", [0.9, 1.1])
def test_tau_solve_fp32_2d(gpu, N, side):
    """FP32 states, on both sides of their psi-form's start: 1e-6 for a rounded result."""
    print(f"tau solve 2-D FP32 N={N} side={side}", flush=True)
    nx, Lx, nu = 8, 4.0, diffusivity(side * (16 if N < 64 else 256), N)
    st = state_2d(N, nx, square, np.complex64)
    got = step_2d(gpu, N, nu, nu, Lx, st, dtype=np.float32)
    for m in (1, 3):
        ref = Mode(N, 2 * np.pi * m / Lx, DT, nu, nu, 2.0)(*rhs_2d(st, m))
        for f in ("b", "u", "uz", "p"):
            assert norm(got[m][f] - ref[f]) <= 1e-6 * norm(ref[f]), (m, f)


@pytest.mark.parametrize("Lx", [40.0, 1.0])  # kh from 0.08 to 0.6 s; from 3 to 22 s, both sides of E1's range
@pytest.mark.parametrize("mr", [0.05, 1.0, 30.0, 1000.0])  # alpha/beta of the lines over N^2
@pytest.mark.parametrize("N", [16, 33, 97, 128])
def test_tau_solve_precision_2d(gpu, N, mr, Lx):
    """A linear FP64 step against long double: no further off than a dense FP64 elimination."""
    print(f"tau solve precision 2-D N={N} m/N2={mr} Lx={Lx}", flush=True)
    nx, nu = 16, diffusivity(mr, N)
    st = state_2d(N, nx, lambda k, N: np.exp(-k * 30.0 / N))
    got = step_2d(gpu, N, nu, nu, Lx, st)
    err, lu = ({f: [] for f in ("b", "u", "uz", "p")} for _ in range(2))
    for m in range(1, nx // 2):
        args, rhs = (N, 2 * np.pi * m / Lx, DT, nu, nu, 2.0), rhs_2d(st, m)
        ref, dense = Mode(*args)(*rhs), Mode(*args, dtype=np.float64)(*rhs)
        for f in err:
            err[f].append(norm(got[m][f] - ref[f]) / norm(ref[f]))
            lu[f].append(norm(dense[f] - ref[f]) / norm(ref[f]))
    check_precision(err, lu, "2-D")


@pytest.mark.parametrize("N,mr,stepper", [(N, mr, SBDF1) for N in (4, 5, 31, 32, 33, 64, 65, 128, 129)
                                          for mr in (0.12, 0.13, 30.0, 1000.0)] +
                         [(256, 30.0, SBDF1)] + [(N, 30.0, RK222) for N in (5, 33, 64, 128, 129)])
def test_tau_solve_3d(gpu, N, mr, stepper):
    """kh from 0.08 to 6 s: uz from E1 (up to 16 s, and N/4 s of the smallest sizes) and from E3z."""
    print(f"tau solve 3-D N={N} m/N2={mr} stepper={stepper}", flush=True)
    nx, ny, Lx, Ly = 8, 8, 40.0, 1.5
    fields = (CHAN3_B, CHAN3_UX, CHAN3_UY, CHAN3_UZ)
    rk = stepper == RK222
    g = 1 - 2 ** -0.5
    nu = diffusivity(mr, N) / (g if rk else 1.0)
    c = DT * (g if rk else 1.0)
    rng = np.random.default_rng(N)
    st = {v: spectrum(rng, (nx // 2 + 1, ny, N), N, square) for v in fields}
    s = gpu.chan3(nx, ny, N, Lx, Ly, 1.0, nu, nu, DT, stepper=stepper, b_bottom=0.0, b_top=0.0)
    for v, x in st.items():
        s.set(v, x * SCALE)
    s.step(1)
    o = {v: s.get(v) / SCALE for v in fields + (CHAN3_P,)}
    taus = [s.tau(i) / SCALE for i in range(9)]
    s.close()
    err, lu = ({f: [] for f in ("b", "u", "v", "uz") + (() if rk else ("p",))} for _ in range(2))
    live = {}
    for m, n in ((1, 0), (2, 3), (3, 6)) if N < 128 else ((1, 0), (2, 3)):
        kx, ky = 2 * np.pi * m / Lx, 2 * np.pi * (n if n < ny // 2 else n - ny) / Ly
        kh = np.hypot(kx, ky)
        turn = lambda x, y: (parts(-1j * (kx * x + ky * y) / kh), parts(-1j * (-ky * x + kx * y) / kh))  # noqa: E731
        rx, ry = turn(st[CHAN3_UX][m, n], st[CHAN3_UY][m, n])
        rhs = [parts(st[CHAN3_B][m, n]), rx, parts(st[CHAN3_UZ][m, n]), ry]
        args = (N, kh, c, nu, nu, 2.0)
        exact, dense = Mode(*args), Mode(*args, dtype=np.float64)
        if rk:  # the second stage (test_tau_solve_rk_2d)
            x1 = exact(*rhs)
            rhs = [r - (1 - g) / g * (r - x1[f]) for r, f in zip(rhs, ("b", "u", "uz", "v"))]
        ref, dense = exact(*rhs), dense(*rhs)
        u, v = turn(o[CHAN3_UX][m, n], o[CHAN3_UY][m, n])
        got = {"b": parts(o[CHAN3_B][m, n]), "u": u, "v": v, "uz": parts(o[CHAN3_UZ][m, n]), "p": parts(o[CHAN3_P][m, n])}
        for f in err:
            err[f].append(norm(got[f] - ref[f]) / norm(ref[f]))
            lu[f].append(norm(dense[f] - ref[f]) / norm(ref[f]))
        if rk:
            continue
        got.update({t: parts(x[m, n]) for t, x in zip(TAUS3, taus) if t})
        got["tau_u1"], got["tau_v1"] = turn(taus[3][m, n], taus[4][m, n])
        got["tau_u2"], got["tau_v2"] = turn(taus[6][m, n], taus[7][m, n])
        scales = tau_scales(*args, rhs[:3], ref)
        row = (1 + c * nu * kh * kh) * norm(ref["v"]) + norm(rhs[3])
        scales.update(tau_v1=row / (c * nu * 4 * (N - 1)), tau_v2=row / c)
        for t, on in check_taus(got, ref, scales).items():
            live[t] = live.get(t, False) or on
    if rk:
        assert max(max(v) for v in err.values()) < 1e-12, err
        return
    check_precision(err, lu, "3-D", factor=8.0, floor=16)
    assert all(live.values()), live


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
    nx, Lx, tol = 8, 4.0, 1e-10 if dtype == np.float64 else 1e-6
    if kappa == "zero":
        kappa = nu = 1.0 / (zero_pivot(N, N % 2) * DT * 4.0)
    st = state_2d(N, nx, lambda k, N: np.exp(-k * 30.0 / N), np.complex64 if dtype == np.float32 else complex)
    got = step_2d(gpu, N, kappa, nu, Lx, st, dtype=dtype)
    for m in range(nx // 2):
        ref = Mode(N, 2 * np.pi * m / Lx, DT, kappa, nu, 2.0)(*rhs_2d(st, m))
        for f in ("b", "u", "uz", "p"):
            e = norm(got[m][f] - ref[f]) / max(norm(ref[f]), 1e-3 * norm(ref["u"]))
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
        for three in (False, True):
            with pytest.raises(_lib.TarangError) as e:
                if three:
                    gpu.chan3(8, 8, 9, 4.0, 4.0, 1.0, kappa, nu, 1e-3)
                else:
                    gpu.chan(16, 9, 4.0, 1.0, kappa, nu, 1e-3)
            assert e.value.code == _lib.ERR_SINGULAR and "singular" in str(e.value)
