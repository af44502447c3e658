"""FLEX on meshes whose axes the box passes do not cover and whose grids are too
large for a whole batch of them (batches and their scratch grids are cut),
against the oracle: without hopping Sigma does not depend on k, so every mesh has
the Sigma of the four points that the oracle solves, at every k.

The device memory that a solve of larger grids leaves in the pool is compared
with the arrays it needs, in grids of N points (16 N bytes): transformed G and mirror 2 x 4,
work and scratch 2, accumulator 1, the four sources of an output (as many as
fit in 4 GB), G and three Sigma 4 x 1 (Nk Nw 4 = N), chi0 4, polynomials 1/2."""
import ctypes

import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu

NX, NW, TEMP, MU, FILL = 4, 407, 0.05, 0.1, 0.8  # 814 = 2 11 37
RVEC = np.zeros((1, 3))
HAM = np.array([[[0.1, 0.15], [0.15, -0.2]]], dtype=np.complex128)


def solve(L, ny):
    klist, kmap, invk = L.gen_irr_k_TRS(NX, ny, 1)
    hamk = L.gen_ham(klist, HAM, RVEC)
    eig, uni = L.get_eig(hamk)
    olist, site = O.get_chi_orb_list(2, [2])
    S, C = O.get_scmat(olist, site, 0.1, 0.02)  # below the Stoner instability of free levels
    sig, mu = L.mkself(S, C, kmap, invk, olist, hamk, eig, uni, MU, FILL, TEMP, NW, NX, ny, 1, False, False, eps=0.0,
                       pp=0.5, m_diis=1, scf_loop=2, sw_tail=False)
    return sig, mu


def free_bytes(F):
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert F._L().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


# grids of 26 MB (several a launch), 101 MB and 1.2 GB (an output's sources in two parts)
@pytest.mark.parametrize("ny,sources", [(506, None), (1936, 4), (23184, 3)])
def test_flex_on_a_rough_mesh(ny, sources):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    ref, mu1 = solve(O, 1)
    solve(F, 1)  # what the first solve of a process loads
    F.release_memory()
    f0 = free_bytes(F)
    sig, mu = solve(F, ny)
    used = f0 - free_bytes(F)
    F.release_memory()
    assert abs(mu - mu1) < 1e-10
    assert np.abs(sig - ref[..., :1]).max() <= 1e-10 * np.abs(ref).max()
    grid = 16.0 * NX * ny * 2 * NW
    assert not sources or used <= (8 + 2 + 1 + sources + 4 + 4 + 0.5 + 0.5) * grid, used / grid


@pytest.mark.parametrize("ny", [506, 1936])
def test_increments_on_a_rough_mesh(ny):
    """FP32 grids of 13 and 50 MB: the reference's transforms and the increments in several launches.  Tolerance of
    the direct DFT's tests for its FP32 sums: 8 eps sqrt(nx + ny + m)."""
    import pyrpa_amd.flibs as F
    ref, mu1 = solve(O, 1)
    try:
        F.set_precision(1)
        sig, mu = solve(F, ny)
    finally:
        F.set_precision(0)
        F.release_memory()
    tol = 8 * float(np.finfo(np.float32).eps) * np.sqrt(NX + ny + 2 * NW)
    assert abs(mu - mu1) < tol and np.abs(sig - ref[..., :1]).max() <= tol * np.abs(ref).max()
