"""Largest real part of the eigenvalues (get_eig_or_tr_chi) against LAPACK at
the edges of the wavefront kernel: one and two rows, sizes around 16, 32 and
64 (the largest held in LDS), one size above, and matrices whose Hessenberg
reduction meets zeros.  Random complex matrices have eigenvalue condition
numbers of about n, so both solvers are within n^2 ulp of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nk", [(1, 5), (2, 3), (3, 65), (9, 200), (16, 33), (17, 7), (25, 40), (33, 4), (64, 3),
                                  (65, 2)])
def test_max_real_eigenvalue(n, nk):
    import pyrpa_amd.flibs as F
    rng = np.random.default_rng(n)
    a = rng.standard_normal((nk, n, n)) + 1j * rng.standard_normal((nk, n, n))
    a[0] = np.diag(np.arange(n) - 0.5 * n)              # nothing to reduce
    if nk > 1:
        a[1] = np.triu(a[1])                            # already triangular
    if nk > 2:
        a[2] = np.roll(np.eye(n), 1, axis=0)            # a cycle: every pivot but one is zero
    if nk > 3:
        a[3] = 0.0
    chi = np.ascontiguousarray(a.transpose(2, 1, 0))    # Python [m, l, k]
    invk = np.ones((nk, 3), dtype=np.int64)
    invk[:, 0] = np.arange(nk) + 1
    got = F.get_eig_or_tr_chi(chi, invk, True)
    ref = np.linalg.eigvals(a).real.max(axis=1)
    scale = np.maximum(np.abs(a).sum(axis=2).max(axis=1), 1.0)
    assert np.all(got.imag == 0)
    assert np.all(np.abs(got.real - ref) <= 1e-14 * n * n * scale)
