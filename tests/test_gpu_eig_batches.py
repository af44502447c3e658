"""Largest real part of the eigenvalues on both sides of the batch size where
the lane kernel takes over from the wavefront kernel, and its workspace: against
LAPACK, and the allocation-free entry point bit for bit.  Tolerance as in
test_gpu_eig.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 9])
@pytest.mark.parametrize("over", [0, 1])
def test_both_sides_of_the_line(n, over):
    import pyrpa_amd.flibs as F
    nk = (50000 if n == 1 else 7500 + 30 * n * n) + over
    rng = np.random.default_rng(n)
    a = rng.standard_normal((nk, n, n)) + 1j * rng.standard_normal((nk, n, n))
    a[7] = 0.0
    chi = np.ascontiguousarray(a.transpose(2, 1, 0))
    invk = np.ones((nk, 3), dtype=np.int64)
    invk[:, 0] = np.arange(nk) + 1
    got = F.get_eig_or_tr_chi(chi, invk, True)
    ref = np.linalg.eigvals(a).real.max(axis=1)
    scale = np.maximum(np.abs(a).sum(axis=2).max(axis=1), 1.0)
    assert np.all(np.abs(got.real - ref) <= 1e-14 * n * n * scale) and np.all(got.imag == 0)
    d_chi, d_inv = F.DeviceArray.from_host(chi.ravel()), F.DeviceArray.from_host(invk.ravel())
    out = F.DeviceArray(nk, np.complex128)
    assert F._L().gmod_eig_or_tr_chi_noalloc(out.ptr, d_chi.ptr, d_inv.ptr, nk, nk, n, 1) == 0
    assert np.array_equal(out.download(), got)
