"""The batched complex LU at the edges of its launch shapes, against the oracle (LAPACK's zgetf2 order).

A panel holds one row per thread of 128, 256 or 512, two of 512, or stays in memory (n > 1024);
panels are 16 columns and trailing tiles 16 x 16.  Pivots have to agree exactly.  Tolerance: 1e-12 as
in the parity test up to n = 512, and growing with n above (rounding of a random matrix's factors).
"""
import numpy as np
import pytest

from tests.conftest import relerr
from tests.test_gpu_dense import lu_on_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nm", [(15, 3), (16, 3), (33, 2), (127, 2), (128, 2), (129, 2), (256, 2), (257, 2), (272, 1),
                                  (512, 1), (513, 1), (1024, 1), (1025, 1)])
def test_batched_lu_shape_edges(gpu, oracle, n, nm):
    from tarang_amd.matsolvers import batched_factor_
    print(f"batched LU edges n={n} nmodes={nm}", flush=True)
    r = np.random.default_rng(n)
    A = r.standard_normal((n, n, nm)) + 1j * r.standard_normal((n, n, nm))
    LU_ref, ipiv_ref, _ = oracle.batched_lu_factor(A)
    s = lu_on_device(gpu, A)
    batched_factor_(s)
    assert np.array_equal(s.pivots.cpu().numpy(), ipiv_ref)
    assert relerr(s.A.cpu().numpy(), LU_ref) < 1e-12 * max(1.0, n / 512)


def test_batched_lu_ties(gpu, oracle):
    """A Hadamard matrix: every value stays a power of two, so all arithmetic is exact, and every pivot is one of
    many equal candidates, of which the first row counts."""
    from tarang_amd.matsolvers import batched_factor_
    print("batched LU ties", flush=True)
    H = np.array([[1.0]])
    while len(H) < 128:
        H = np.block([[H, H], [H, -H]])
    i = np.arange(128)
    rev = np.array([int(format(k, "07b")[::-1], 2) for k in i])
    H = H[rev] * np.where(i < 64, 0.5, 1.0)[:, None]  # 111 of the 128 pivots interchange rows
    A = np.stack([H, 1.0j * H], axis=2).astype(complex)
    LU_ref, ipiv_ref, _ = oracle.batched_lu_factor(A)
    s = lu_on_device(gpu, A)
    batched_factor_(s)
    assert np.array_equal(s.pivots.cpu().numpy(), ipiv_ref)
    assert np.array_equal(s.A.cpu().numpy(), LU_ref)


@pytest.mark.parametrize("n", [60, 129, 263, 400])
def test_batched_lu_backward_error(gpu, oracle, n):
    """P A - L U in long double, over |A|: no larger than the oracle's, which updates the trailing matrix term by
    term (mean of four matrices)."""
    from tarang_amd.matsolvers import batched_factor_
    print(f"batched LU backward error n={n}", flush=True)
    r = np.random.default_rng(n)
    A = (r.standard_normal((n, n, 4)) + 1j * r.standard_normal((n, n, 4))) / np.sqrt(n) + 0.5 * np.eye(n)[:, :, None]
    ref, piv, _ = oracle.batched_lu_factor(A)
    s = lu_on_device(gpu, A)
    batched_factor_(s)
    assert np.array_equal(s.pivots.cpu().numpy(), piv)
    got = s.A.cpu().numpy()

    def backward(LU, m):
        P = np.arange(n)
        for k, p in enumerate(piv[:, m]):
            P[[k, p - 1]] = P[[p - 1, k]]
        LU = LU[:, :, m].astype(np.clongdouble)
        R = A[P, :, m] - (np.tril(LU, -1) + np.eye(n)) @ np.triu(LU)
        return np.linalg.norm(R.astype(complex)) / np.linalg.norm(A[:, :, m])

    a, b = (np.mean([backward(x, m) for m in range(4)]) for x in (got, ref))
    print(f"  backward error {a:.2e}, oracle {b:.2e}", flush=True)
    assert a <= b
