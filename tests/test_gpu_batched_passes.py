"""Batched transform passes against the oracle where their launches differ:
grids of a single box, few boxes (quarter-size boxes, tiled and not), boxes
whose element count is no multiple of the work-group (the untiled kernel),
lengths the box passes do not cover (a prime above 7: the direct DFT of
the per-axis passes), one item and many, a mesh with odd lengths, and the
spinful functors.  FP64: 1e-11 of the largest element (the transforms' rounding
is a few log2 N ulp); FP32 transforms: 2^-24 log2 N times a small factor."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 2, 1, 1), (2, 4, 4, 1, 4), (1, 32, 32, 1, 32), (2, 16, 16, 4, 16), (3, 9, 9, 3, 10), (2, 6, 10, 2, 15),
          (2, 11, 11, 1, 9), (2, 8, 8, 1, 13), (4, 8, 8, 2, 8)]


@pytest.mark.parametrize("norb,nx,ny,nz,nw", SHAPES)
@pytest.mark.parametrize("prec", [0, 1])
def test_chi0_and_tail(norb, nx, ny, nz, nw, prec):
    import pyrpa_amd.flibs as F
    st = MD.random_model(norb, nx, ny, nz, nw, 0.08, 0.1, 0.5, 0.1, seed=7 + norb)
    args = (st['Smat'], st['Cmat'], st['Gk'])
    mesh = (st['olist'], st['kmap'], st['invk'])
    try:
        F.set_precision(prec)
        a, _ = F.get_chi0(*args, *mesh, st['temp'], nx, ny, nz)
        b, _ = F.get_chi0_tail(*args, st['eig'], st['uni'], *mesh, st['mu'], st['temp'], nx, ny, nz)
    finally:
        F.set_precision(0)
    ra, _ = O.get_chi0(*args, *mesh, st['temp'], nx, ny, nz)
    rb, _ = O.get_chi0_tail(*args, st['eig'], st['uni'], *mesh, st['mu'], st['temp'], nx, ny, nz)
    tol = 1e-11 if prec == 0 else 4e-6
    assert np.abs(a - ra).max() <= tol * np.abs(ra).max()
    # the FP32 tail differs from the oracle by the rounding of conv[G], which
    # the subtraction of conv[G0] leaves in place
    assert np.abs(b - rb).max() <= tol * max(np.abs(rb).max(), np.abs(ra).max())


@pytest.mark.parametrize("norb,nx,ny,nz,nw", [SHAPES[1], SHAPES[3], SHAPES[4], SHAPES[6], SHAPES[7]])
@pytest.mark.parametrize("tail", [False, True])
def test_flex_iterations(norb, nx, ny, nz, nw, tail):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    st = MD.random_model(norb, nx, ny, nz, nw, 0.1, 0.1, 0.5, 0.1, seed=3, real=True)
    args = (st['Smat'], st['Cmat'], st['kmap'], st['invk'], st['olist'], st['hamk'], st['eig'], st['uni'], 0.1,
            0.4 * norb, st['temp'], nw, nx, ny, nz, False, False)
    kw = dict(eps=0.0, pp=0.5, m_diis=1, scf_loop=2, sw_tail=tail)
    a, mu = F.mkself(*args, **kw)
    b, mub = O.mkself(*args, **kw)
    assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max() and abs(mu - mub) < 1e-10


@pytest.mark.parametrize("nx,nw", [(4, 6), (9, 5), (16, 16)])
def test_spinful_chi0(nx, nw):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    st = MD.spinful(MD.two_orbital(Nx=nx, Ny=nx, Nw=nw, temp=0.1, mu=0.1), lam=0.1, alpha=0.1, U=0.5, J=0.1)
    args = (st['Vmat'], st['Gk'], st['olist'], st['slist'], st['kmap'], st['invk'], st['invs'], st['temp'], nx, nx, 1)
    a, r = F.get_chi0_soc(*args)[0], O.get_chi0_soc(*args)[0]
    assert np.abs(a - r).max() <= 1e-11 * np.abs(r).max()
