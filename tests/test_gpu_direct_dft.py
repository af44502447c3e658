"""The direct DFT of the per-axis passes (axes with a prime factor above 7)
against numpy, forward and backward: lengths around multiples of the four
outputs and two lines a thread forms, fewer lines than a work-group takes, a
single line, the longest direct pass, lengths past 256 (split in two passes)
and strided and contiguous stores.

Tolerance: a sum of n terms in turn has an error of about eps sqrt(n / 2) of
the RMS of its result (partial sums grow like sqrt(j)); the axes' errors add in
squares and the largest of up to a few 1e5 elements is within six standard
deviations: 8 eps sqrt(sum n), eps = 2^-52 or 2^-23 (the products round as
well)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(11, 1, 1, 1), (13, 3, 1, 2), (1, 17, 1, 5), (29, 29, 1, 9), (9, 10, 1, 22), (4, 1, 1, 26), (8, 8, 1, 131),
          (1, 1, 1, 253), (2, 3, 1, 1632), (44, 4, 1, 162), (1, 2, 1, 251), (5, 1, 1, 254)]


@pytest.mark.parametrize("dims", SHAPES)
@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_against_numpy(dims, dtype):
    import pyrpa_amd.flibs as F
    nx, ny, nz, m = dims
    rng = np.random.default_rng(nx + 7 * m)
    a = (rng.standard_normal((m, nz, ny, nx)) + 1j * rng.standard_normal((m, nz, ny, nx))).astype(dtype)
    tol = 8 * float(np.finfo(dtype).eps) * np.sqrt(nx + ny + nz + m)
    for sign in (-1, 1):
        buf, tmp = F.DeviceArray.from_host(a.ravel()), F.DeviceArray(a.size, dtype)
        F.fft_device(buf, tmp, dims, sign=sign)
        got = buf.download().reshape(a.shape)
        x = a.astype(np.complex128)
        ref = np.fft.fftn(x) if sign < 0 else np.fft.ifftn(x)
        err = np.abs(got - ref).max() / np.sqrt(np.mean(np.abs(ref) ** 2))
        assert err < tol, (dims, sign, err, tol)
