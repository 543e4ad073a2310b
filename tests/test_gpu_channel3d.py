"""3-D Rayleigh-Benard channel on the GPU (tarang_chan3_*) vs the FP64 oracle.

Tolerances: FP64 1e-12 relative (max-norm against the largest oracle entry) for the
right-hand side and steps, FP32 1e-5.  At the
256 x 256 x 128 workload the check is mode-wise against a small oracle grid on a
small-amplitude state confined to modes kx, ky in {0, 1}, whose products are alias-free
on both grids.
"""
import ctypes

import numpy as np
import pytest

from tarang_amd import _lib
from tests.conftest import relerr

pytestmark = pytest.mark.gpu

TOL = {np.float64: 1e-12, np.float32: 1e-5}


def zgrid(N, Lz):
    return Lz * (1 - np.cos(np.pi * np.arange(N) / (N - 1))) / 2


def random_state3(O, nx, ny, N, Lx, Ly, Lz, seed=2, raw=1e-3):
    rng = np.random.default_rng(seed)
    d = O.domain([O.REALFOURIER, O.REALFOURIER, O.CHEBYSHEVT], [nx, ny, N],
                 bounds=[(0.0, Lx), (0.0, Ly), (0.0, Lz)])
    z = zgrid(N, Lz)
    w = (z * (Lz - z))[None, None, :]
    out = {}
    for v in (O.RBC3_B, O.RBC3_UX, O.RBC3_UY, O.RBC3_UZ):
        g = 0.05 * rng.standard_normal((nx, ny, N)) * w + ((Lz - z)[None, None, :] if v == O.RBC3_B else 0.0)
        c = np.asarray(O.forward_transform(d, g))
        if raw:
            c = c + raw * (rng.standard_normal(c.shape) + 1j * rng.standard_normal(c.shape))
        out[v] = c
    return out, d


def kp():
    return 1e5 ** -0.5, 1e5 ** -0.5


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nx,ny,N", [(16, 8, 12), (32, 16, 17)])
def test_channel3d_rhs_parity(gpu, oracle, dtype, nx, ny, N):
    print(f"channel3d rhs {nx}x{ny}x{N} {dtype.__name__}", flush=True)
    Lx, Ly, Lz = 4.0, 3.0, 1.0
    kappa, nu = kp()
    st, d = random_state3(oracle, nx, ny, N, Lx, Ly, Lz)
    ref = oracle.RBC3D(nx, ny, N, Lx, Ly, Lz, kappa, nu, 5e-3, "SBDF2")
    for v, c in st.items():  # the oracle's rhs takes the grid-round-tripped state
        ref.set(v, oracle.forward_transform(d, oracle.backward_transform(d, c)))
    Fr = ref.rhs()
    s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, kappa, nu, 5e-3, dtype=dtype)
    for v, c in st.items():
        s.set(v, c)
    Fg = s.rhs()
    errs = [relerr(a, b) for a, b in zip(Fg, Fr)]
    print(f"  rel errs {errs}", flush=True)
    assert max(errs) < TOL[dtype]
    s.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ts", ["SBDF2", "SBDF1", "RK222", "RK443"])
def test_channel3d_steps_parity(gpu, oracle, ts, dtype):
    nx, ny, N, Lx, Ly, Lz = 16, 8, 12, 4.0, 3.0, 1.0
    print(f"channel3d steps {ts} {dtype.__name__}", flush=True)
    kappa, nu = kp()
    st, d = random_state3(oracle, nx, ny, N, Lx, Ly, Lz, seed=5)
    ref = oracle.RBC3D(nx, ny, N, Lx, Ly, Lz, kappa, nu, 5e-3, ts)
    s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, kappa, nu, 5e-3, stepper={"SBDF2": 2, "SBDF1": 4, "RK222": 0, "RK443": 1}[ts],
                  dtype=dtype)
    for v, c in st.items():
        ref.set(v, c)
        s.set(v, c)
    for nsteps, dt in ((1, 5e-3), (2, 5e-3), (2, 2.5e-3)):
        ref.set_dt(dt)
        s.set_dt(dt)
        ref.step(nsteps)
        s.step(nsteps)
        errs = [relerr(s.get(v), ref.get(v)) for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ)]
        print(f"  after {nsteps} at dt {dt}: rel errs {errs}", flush=True)
        assert max(errs) < TOL[dtype], (nsteps, dt, errs)
        assert relerr(s.get(oracle.RBC3_P), ref.get(oracle.RBC3_P)) < TOL[dtype] * 100
        scale = max(np.abs(ref.tau(t)).max() for t in range(9))  # tau_p is roundoff around 0
        for t in range(9):
            assert np.abs(s.tau(t) - ref.tau(t)).max() <= TOL[dtype] * 100 * scale, t
    s.close()


def test_channel3d_graph_and_keys(gpu, oracle):
    nx, ny, N, L = 16, 16, 9, 2 * np.pi
    kappa, nu = kp()
    st, _ = random_state3(oracle, nx, ny, N, L, L, 1.0, seed=9)
    out = []
    for graph in (False, True):
        s = gpu.chan3(nx, ny, N, L, L, 1.0, kappa, nu, 5e-3)
        # Lx == Ly: modes share factors by m^2 + k^2
        n_sq = {m * m + k * k for m in range(nx // 2 + 1) for k in range(-ny // 2, ny // 2)}
        assert s.nkeys() == len(n_sq)
        s.set_graph(graph)
        for v, c in st.items():
            s.set(v, c)
        s.step(3)
        out.append([s.get(v) for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ)])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nx,ny,N", [(32, 32, 24), (16, 8, 49), (16, 8, 128), (16, 8, 129)])
def test_channel3d_tuning_variants_same_bits(gpu, oracle, nx, ny, N, dtype):
    """Every kernel variant the autotuner can pick (k3_tau_solve with one or two pairs of waves per workgroup,
    k3_zbwd with 32- or 16-mode tiles) gives the same bits over 3 SBDF2 steps, for each shape of the solve (16
    lanes and one, two or four degrees, 32 lanes)."""
    L = 4.0
    kappa, nu = kp()
    st, _ = random_state3(oracle, nx, ny, N, L, L, 1.0, seed=11)
    variants = [(0, 0), (1, 0)] + ([(0, 1), (1, 1)] if dtype == np.float32 else [])
    out = []
    for v in variants:
        print(f"channel3d tuning variant {v} {dtype.__name__}", flush=True)
        s = gpu.chan3(nx, ny, N, L, L, 1.0, kappa, nu, 5e-3, dtype=dtype)
        t = (ctypes.c_int * 2)(*v)
        _lib.call("tarang_chan3_set_tuning", s.h, t)
        got = (ctypes.c_int * 2)()
        _lib.call("tarang_chan3_get_tuning", s.h, got)
        assert tuple(got) == v
        for var, c in st.items():
            s.set(var, c)
        s.step(3)
        out.append([s.get(var) for var in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ)])
        s.close()
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
    s = gpu.chan3(nx, ny, N, L, L, 1.0, kappa, nu, 5e-3, dtype=np.float64)
    with pytest.raises(_lib.TarangError):  # the 16-mode z tile is an FP32 variant
        _lib.call("tarang_chan3_set_tuning", s.h, (ctypes.c_int * 2)(0, 1))
    with pytest.raises(_lib.TarangError):
        _lib.call("tarang_chan3_set_tuning", s.h, (ctypes.c_int * 2)(2, 0))
    s.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_channel3d_multichunk_keys(gpu, oracle, dtype):
    """64 x 64 x 9 with Lx == Ly: |k_h|^2 keys of up to 12 modes, so one key's modes span several
    workgroups of the solve; every field against the oracle after SBDF1 + SBDF2 steps."""
    nx = ny = 64
    N, L = 9, 2 * np.pi
    print(f"channel3d multichunk {dtype.__name__}", flush=True)
    counts = {}
    for m in range(nx // 2 + 1):
        for k in range(-ny // 2, ny // 2):
            counts[m * m + k * k] = counts.get(m * m + k * k, 0) + 1
    assert max(counts.values()) > 8
    kappa, nu = kp()
    st, _ = random_state3(oracle, nx, ny, N, L, L, 1.0, seed=13)
    ref = oracle.RBC3D(nx, ny, N, L, L, 1.0, kappa, nu, 5e-3, "SBDF2")
    s = gpu.chan3(nx, ny, N, L, L, 1.0, kappa, nu, 5e-3, stepper=2, dtype=dtype)
    assert s.nkeys() == len(counts)
    for v, c in st.items():
        ref.set(v, c)
        s.set(v, c)
    ref.step(2)
    s.step(2)
    for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ):
        assert relerr(s.get(v), ref.get(v)) < TOL[dtype], v
    assert relerr(s.get(oracle.RBC3_P), ref.get(oracle.RBC3_P)) < TOL[dtype] * 100
    scale = max(np.abs(ref.tau(t)).max() for t in range(9))
    for t in range(9):
        assert np.abs(s.tau(t) - ref.tau(t)).max() <= TOL[dtype] * 100 * scale, t
    s.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_channel3d_full_size_modewise(gpu, oracle, dtype):
    """256 x 256 x 128 (the 3-D workload) vs a 16 x 16 x 128 oracle on modes kx, ky in {0, 1}.
    Errors are relative to each mode's own size or the perturbation amplitude (~3e-5 of the
    O(1) conduction profile), whichever is larger: FP64 1e-11 there, since the profile's own
    rounding (1e-16 absolute) is already 3e-12 of the perturbation; FP32 1e-5."""
    nx = ny = 256
    N, Lx, Ly, Lz, dt = 128, 4.0, 4.0, 1.0, 2e-3
    print(f"channel3d full size {dtype.__name__}", flush=True)
    Ra, Pr = 1e7, 0.7
    kappa, nu = (Ra * Pr) ** -0.5, (Ra / Pr) ** -0.5
    small = 16
    rng = np.random.default_rng(4)
    ds = oracle.domain([oracle.REALFOURIER, oracle.REALFOURIER, oracle.CHEBYSHEVT], [small, small, N],
                       bounds=[(0.0, Lx), (0.0, Ly), (0.0, Lz)])
    z = zgrid(N, Lz)
    wall = z * (Lz - z)
    st = {}
    for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ):
        c = np.zeros((small // 2 + 1, small, N), complex)
        if v == oracle.RBC3_B:
            c = np.asarray(oracle.forward_transform(ds, np.tile((Lz - z)[None, None, :], (small, small, 1))))
        for (m, n) in ((1, 0), (0, 1), (1, 1), (1, small - 1)):
            prof = np.polynomial.chebyshev.chebfit(2 * z / Lz - 1, wall * np.sin(2 * np.pi * z / Lz), 30)
            c[m, n, :31] += 1e-6 * small * small * prof * np.exp(1j * rng.uniform(0, 2 * np.pi))
        if v != oracle.RBC3_B:
            c[0, 1] = 0.0   # keep the kx = 0 line Hermitian: (0, 1) and (0, -1) together
        st[v] = c
    for v in st:
        st[v][0, small - 1] = np.conj(st[v][0, 1])
    ref = oracle.RBC3D(small, small, N, Lx, Ly, Lz, kappa, nu, dt, "SBDF2")
    for v, c in st.items():
        ref.set(v, c)
    s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, kappa, nu, dt, stepper=2, dtype=dtype)
    scale = (nx / small) * (ny / small)
    for v, c in st.items():
        big = np.zeros((nx // 2 + 1, ny, N), complex)
        big[:small // 2, :small // 2] = c[:small // 2, :small // 2] * scale
        big[:small // 2, ny - small // 2 + 1:] = c[:small // 2, small // 2 + 1:] * scale
        s.set(v, big)
    ref.step(3)
    s.step(3)
    tol = {np.float64: 1e-11, np.float32: 1e-5}[dtype]
    worst = 0.0
    for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ):
        g = s.get(v) / scale
        r = ref.get(v)
        pert = max(np.abs(r[1, 1]).max(), np.abs(r[1, 0]).max())
        for (m, n, ns) in ((0, 0, 0), (1, 0, 0), (1, 1, 1), (1, ny - 1, small - 1)):
            den = max(np.abs(r[m, ns]).max(), pert)
            err = np.abs(g[m, n] - r[m, ns]).max() / den
            worst = max(worst, err)
            assert err < tol, (v, m, n, err)
    print(f"  worst mode-wise rel err {worst:.3e}", flush=True)
    s.close()


def test_channel3d_rejects_unsupported(gpu):
    kappa, nu = kp()
    with pytest.raises(_lib.TarangError) as e:
        gpu.chan3(24, 16, 9, 4.0, 4.0, 1.0, kappa, nu, 1e-2)
    assert e.value.code == _lib.ERR_INVALID
    with pytest.raises(_lib.TarangError):
        gpu.chan3(16, 16, 300, 4.0, 4.0, 1.0, kappa, nu, 1e-2)
    with pytest.raises(_lib.TarangError):
        gpu.chan3(16, 16, 9, 4.0, 4.0, 1.0, kappa, nu, 1e-2, stepper=3)
    with pytest.raises(_lib.TarangError) as e:  # split_inverse = 1 belongs to the FP32 state
        gpu.chan3(16, 16, 9, 4.0, 4.0, 1.0, kappa, nu, 1e-2, dtype=np.float64, split=1)
    assert e.value.code == _lib.ERR_INVALID and "split_inverse" in str(e.value)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_channel3d_refinement_sweeps(gpu, oracle, dtype):
    """refine_sweeps and split_inverse change nothing: every setting gives the same bits, within 1e-12 (FP64) and
    1e-5 (FP32) of the oracle after SBDF2 steps.  Nz = 65 keeps the tau systems as ill-conditioned as the 3-D
    workload's (condition numbers ~1e7)."""
    nx, ny, N, Lx, Ly, Lz = 16, 16, 65, 4.0, 4.0, 1.0
    kappa, nu = (1e7 * 0.7) ** -0.5, (1e7 / 0.7) ** -0.5
    st, d = random_state3(oracle, nx, ny, N, Lx, Ly, Lz, seed=7)
    ref = oracle.RBC3D(nx, ny, N, Lx, Ly, Lz, kappa, nu, 2e-3, "SBDF2")
    for v, c in st.items():
        ref.set(v, c)
    ref.step(3)
    want = {v: ref.get(v) for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ)}
    out = {}
    forms = [(0, 0), (1, 0), (2, 0)] + ([(0, 1), (1, 1)] if dtype == np.float32 else [])
    for sweeps, split in forms:
        print(f"channel3d refinement sweeps={sweeps} split={split} {dtype.__name__}", flush=True)
        s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, kappa, nu, 2e-3, dtype=dtype, refine=sweeps, split=split)
        for v, c in st.items():
            s.set(v, c)
        s.step(3)
        out[(sweeps, split)] = [s.get(v) for v in want]
        s.close()
    err = max(relerr(a, w) for a, w in zip(out[(0, 0)], want.values()))
    print(f"  max rel err {err}", flush=True)
    assert err < (1e-12 if dtype == np.float64 else 1e-5)
    for f in forms[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(out[f], out[(0, 0)])), f


def test_channel3d_fp32_forms_long_run(gpu):
    """FP32 states against the FP64 one (itself pinned to the oracle at 1e-12) over 300 SBDF2 steps of the 3-D
    workload's physics (Ra = 1e7, Pr = 0.7, dt = 2e-3, Nz = 128, conduction plus noise) on a 16 x 16 grid: every
    setting of split_inverse and refine_sweeps gives the same bits, and b stays within 1e-6 of FP64 (the FP64
    solves leave only the rounding of the state)."""
    nx = ny = 16
    N, Lx, Ly, Lz, dt, steps = 128, 4.0, 4.0, 1.0, 2e-3, 300
    kappa, nu = (1e7 * 0.7) ** -0.5, (1e7 / 0.7) ** -0.5
    z = zgrid(N, Lz)
    rng = np.random.default_rng(42)
    bg = (Lz - z)[None, None, :] + 1e-3 * rng.standard_normal((nx, ny, N)) * (z * (Lz - z))[None, None, :]
    k = np.arange(N)
    T = np.cos(np.outer(np.pi * np.arange(N) / (N - 1), k)) * ((-1.0) ** k)[None, :]
    Bc = np.einsum("kz,mnz->mnk", np.linalg.inv(T), np.fft.fft(np.fft.rfft(bg, axis=0), axis=1))
    out = {}
    for name, dtype, sweeps, split in (("f64", np.float64, 0, 0), ("plain", np.float32, 0, 0),
                                       ("split", np.float32, 0, 1), ("sweeps1", np.float32, 1, 0)):
        print(f"channel3d long run {name}", flush=True)
        s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, kappa, nu, dt, stepper=2, dtype=dtype, refine=sweeps, split=split)
        s.set(_lib.CHAN3_B, Bc)
        for v in (_lib.CHAN3_P, _lib.CHAN3_UX, _lib.CHAN3_UY, _lib.CHAN3_UZ):
            s.set(v, np.zeros_like(Bc))
        s.step(steps)
        out[name] = s.get(_lib.CHAN3_B)
        s.close()
    err = relerr(out["plain"], out["f64"])
    print(f"  b rel err vs FP64 after {steps} steps: {err}", flush=True)
    assert err < 1e-6
    assert np.array_equal(out["split"], out["plain"]) and np.array_equal(out["sweeps1"], out["plain"])


def test_channel3d_rhs_full_size(gpu, oracle):
    """The right-hand side at the 3-D workload's size (256 x 256 x 128, Lx = Ly = 4) on a
    full-spectrum random state, against the oracle's right-hand side (no per-mode matrices):
    every mode, the Nyquist lines and the 384-point padded products included.  FP64 1e-12,
    FP32 1e-5 (relative to the largest oracle entry)."""
    nx = ny = 256
    N, Lx, Ly, Lz = 128, 4.0, 4.0, 1.0
    print("channel3d rhs full size: oracle right-hand side (about half a minute)", flush=True)
    rng = np.random.default_rng(21)
    ref = oracle.RBC3D(nx, ny, N, Lx, Ly, Lz, 0.0, 0.0, 0.0, rhs_only=True)
    st = {}
    for v in (oracle.RBC3_B, oracle.RBC3_UX, oracle.RBC3_UY, oracle.RBC3_UZ):
        c = 1e-3 * (rng.standard_normal(ref.shape) + 1j * rng.standard_normal(ref.shape))
        st[v] = c
        # the oracle's right-hand side takes the grid-round-tripped state, as the solver's does
        ref.set(v, oracle.forward_transform(ref.d, oracle.backward_transform(ref.d, c)))
    Fr = ref.rhs()
    for dtype, tol in ((np.float64, 1e-12), (np.float32, 1e-5)):
        print(f"channel3d rhs full size {dtype.__name__}", flush=True)
        s = gpu.chan3(nx, ny, N, Lx, Ly, Lz, 1e-3, 1e-3, 2e-3, dtype=dtype)
        for v, c in st.items():
            s.set(v, c)
        errs = [relerr(a, b) for a, b in zip(s.rhs(), Fr)]
        print(f"  rel errs {errs}", flush=True)
        assert max(errs) < tol, errs
        s.close()
