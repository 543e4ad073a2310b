"""The per-mode tau systems in long double, from the equations (first-order tau form), by dense elimination.

One mode (|k_h| = kh, implicit coefficient c, s = 2/Lz), with ux = i u~ along k_h; every row times c:
  E2 : (1 + c kappa kh^2) b - c kappa D^2 b - c kappa D(T_{N-1}) tau_b1 + c T_{N-1} tau_b2 = r,  b = 0 on the walls
  E3x: the same with nu and + c kh p;   perp: the same with nu
  E1 : -c kh u~ + c D uz + c T_{N-1} tau_u1z (+ c tau_p at kh = 0) = 0
  E3z: the same with nu and + c D p - c b, lifts tau_u1z and tau_u2z
"""
import numpy as np

LD = np.longdouble


def solve(A, B, dtype=LD):
    """Gaussian elimination with partial pivoting in `dtype`; B is (n, m)."""
    A, B = A.astype(dtype).copy(), B.astype(dtype).copy()
    n = len(A)
    for k in range(n):
        p = k + int(np.argmax(np.abs(A[k:, k])))
        if p != k:
            A[[k, p]], B[[k, p]] = A[[p, k]], B[[p, k]]
        rows = k + 1 + np.flatnonzero(A[k + 1:, k])
        if len(rows):
            f = A[rows, k] / A[k, k]
            A[rows, k:] -= np.outer(f, A[k, k:])
            B[rows] -= np.outer(f, B[k])
    for k in range(n - 1, -1, -1):
        B[k] = (B[k] - A[k, k + 1:] @ B[k + 1:]) / A[k, k]
    return B


def solve_by_parity(A, B, rows, cols, dtype):
    """The two decoupled halves of A X = B: rows and cols label every equation and unknown 0 or 1."""
    X = np.zeros((len(cols), B.shape[1]), dtype)
    for q in (0, 1):
        r, c = np.flatnonzero(rows == q), np.flatnonzero(cols == q)
        assert not A[np.ix_(r, np.flatnonzero(cols != q))].any()
        X[c] = solve(A[np.ix_(r, c)], B[r], dtype)
    return X


def deriv(N, s):
    """d/dz of Chebyshev coefficients."""
    k, j = np.arange(N)[:, None], np.arange(N)[None, :]
    D = np.where((j > k) & ((j - k) % 2 == 1), 2 * j, 0).astype(LD)
    D[0] /= 2
    return D * LD(s)


class Mode:
    """Fields and taus of one mode for right-hand sides r_b, r_x, r_z, r_y (perp), each (N, m), real."""

    def __init__(self, N, kh, c, kappa, nu, s, dtype=LD):
        self.N, self.kh, self.dtype = N, LD(kh), dtype
        self.c = c = LD(c)
        kh = self.kh
        D = deriv(N, s)
        D2, I = D @ D, np.eye(N, dtype=LD)
        self.last, self.dlast = I[:, N - 1], D[:, N - 1]
        k = np.arange(N)
        self.walls = np.stack([k % 2 == 0, k % 2 == 1]).astype(LD)  # half the sum and difference of the wall values
        top = np.array([(N - 2) % 2, (N - 1) % 2])  # degrees of D T_{N-1} and T_{N-1}
        self.rb = np.concatenate([k % 2, [0, 1]])
        self.cb = np.concatenate([k % 2, top])

        def helm(diff):
            return (1 + c * LD(diff) * kh * kh) * I - c * LD(diff) * D2

        def scalar(diff):
            A = np.zeros((N + 2, N + 2), LD)
            A[:N, :N] = helm(diff)
            A[:N, N], A[:N, N + 1] = -c * LD(diff) * self.dlast, c * self.last
            A[N:, :N] = self.walls
            return A

        self.Ab, self.Ay = scalar(kappa), scalar(nu)
        mean = bool(kh == 0)
        n = 3 * N + 4 + (1 if mean else 0)
        A = np.zeros((n, n), LD)
        X, P, Z, t = slice(0, N), slice(N, 2 * N), slice(2 * N, 3 * N), 3 * N
        A[X, X] = A[Z, Z] = helm(nu)
        A[X, P], A[Z, P] = c * kh * I, c * D
        A[P, X], A[P, Z] = -c * kh * I, c * D
        A[X, t], A[X, t + 1] = -c * LD(nu) * self.dlast, c * self.last
        A[Z, t + 2], A[Z, t + 3] = -c * LD(nu) * self.dlast, c * self.last
        A[P, t + 2] = c * self.last
        A[t:t + 2, X] = self.walls
        A[t + 2:t + 4, Z] = self.walls
        # halves by the parity of u~ and p; uz and E3z have the other one
        self.ru = np.concatenate([k % 2, k % 2, 1 - k % 2, [0, 1, 1, 0], [0] * mean])
        self.cu = np.concatenate([k % 2, k % 2, 1 - k % 2, top, 1 - top, [0] * mean])
        if mean:  # tau_p in the constant row of E1, integ(p) = 0
            A[N, t + 4] = c
            A[t + 4, P] = np.where(k % 2 == 0, LD(1) / (1 - k.astype(LD) ** 2 + (k == 1)), 0)
        self.A = A

    def __call__(self, rb, rx, rz, ry=None):
        """dict of b, u, p, uz, v (perp) and the taus, each with the columns of the right-hand sides."""
        N, d = self.N, self.dtype
        m = rb.shape[1]
        z2 = np.zeros((2, m), LD)
        ob = solve_by_parity(self.Ab, np.concatenate([rb, z2]), self.rb, self.cb, d)
        rhs = np.zeros((len(self.A), m), LD)
        rhs[:N] = rx
        rhs[2 * N:3 * N] = rz + self.c * ob[:N]
        o = solve_by_parity(self.A, rhs, self.ru, self.cu, d)
        out = {"b": ob[:N], "tau_b1": ob[N], "tau_b2": ob[N + 1], "u": o[:N], "p": o[N:2 * N], "uz": o[2 * N:3 * N],
               "tau_u1": o[3 * N], "tau_u2": o[3 * N + 1], "tau_u1z": o[3 * N + 2], "tau_u2z": o[3 * N + 3]}
        if ry is not None:
            ov = solve_by_parity(self.Ay, np.concatenate([ry, z2]), self.rb, self.cb, d)
            out.update({"v": ov[:N], "tau_v1": ov[N], "tau_v2": ov[N + 1]})
        return out
