"""Copies between the caller's arrays and the device around the size where the
staged parallel copy takes over (8 MB) and for lengths that are no multiple of
its pieces: the one-orbital Dyson inverse and G0, element by element, where a
wrong piece or a race shows as a wrong element.  One complex division each
side: 1e-14 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,nk", [(1, 524287), (1, 524288), (1, 524289), (7, 100003), (16, 262147)])
def test_large_arrays(nw, nk):
    import pyrpa_amd.flibs as F
    rng = np.random.default_rng(nk)
    sig = rng.standard_normal((1, 1, nw, nk)) - 1j * rng.uniform(0.1, 1.0, (1, 1, nw, nk))
    ham = rng.standard_normal((nk, 1, 1)).astype(complex)
    temp, mu = 0.05, 0.2
    w = (2 * np.arange(nw) + 1) * np.pi * temp
    for _ in range(2):  # the second call reuses the buffers
        G = F.gen_green(sig, ham, mu, temp)
        ref = 1.0 / (1j * w[:, None] + mu - ham[None, :, 0, 0] - sig[0, 0])
        assert np.all(np.abs(G[0, 0] - ref) <= 1e-14 * np.abs(ref))
    F.release_memory()
    G0 = F.gen_Green0(ham[:, :, 0].real.copy(), np.ones((nk, 1, 1), complex), mu, temp, nw)
    ref = 1.0 / (1j * w[:, None] + mu - ham[None, :, 0, 0].real)
    assert np.all(np.abs(G0[0, 0] - ref) <= 1e-14 * np.abs(ref))
