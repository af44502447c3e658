"""The split t axis (GMOD_FFT_TSPLIT=1: two strided-slot passes with a scratch
grid between them) under every batch of transforms, against the oracle: a
spinless and a spinful chi0, the tail's products, the Sigma heads, the gap's
anomalous functions, and one orbital (no batch).  A 16x2 mesh with 1024
frequencies is split in both precisions and used nowhere else, so its plans are
made with the switch set.  Tolerances as for the unsplit passes
(test_gpu_batched_passes.py)."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu

MESH, NW, TEMP = (16, 2, 1), 1024, 0.05


@pytest.fixture
def F(monkeypatch):
    import pyrpa_amd.flibs as F
    monkeypatch.setenv("GMOD_FFT_TSPLIT", "1")
    yield F
    F.set_precision(0)


@pytest.mark.parametrize("norb", [1, 2])
@pytest.mark.parametrize("prec", [0, 1])
def test_chi0(F, norb, prec):
    st = MD.random_model(norb, *MESH, NW, TEMP, 0.1, 0.5, 0.1, seed=norb)
    args, mesh = (st['Smat'], st['Cmat'], st['Gk']), (st['olist'], st['kmap'], st['invk'])
    F.set_precision(prec)
    a = F.get_chi0(*args, *mesh, TEMP, *MESH)[0]
    b = F.get_chi0_tail(*args, st['eig'], st['uni'], *mesh, st['mu'], TEMP, *MESH)[0]
    ra = O.get_chi0(*args, *mesh, TEMP, *MESH)[0]
    rb = O.get_chi0_tail(*args, st['eig'], st['uni'], *mesh, st['mu'], TEMP, *MESH)[0]
    tol = 1e-11 if prec == 0 else 4e-6
    assert np.abs(a - ra).max() <= tol * np.abs(ra).max()
    assert np.abs(b - rb).max() <= tol * max(np.abs(rb).max(), np.abs(ra).max())


@pytest.mark.parametrize("prec", [0, 1])
def test_flex(F, prec):
    """FP32: the second iteration runs the increments (1e-5: their rounding through the vertex)"""
    st = MD.random_model(2, *MESH, NW, TEMP, 0.1, 0.5, 0.1, seed=3, real=True)
    args = (st['Smat'], st['Cmat'], st['kmap'], st['invk'], st['olist'], st['hamk'], st['eig'], st['uni'], 0.1, 0.8,
            TEMP, NW, *MESH, False, False)
    kw = dict(eps=0.0, pp=0.5, m_diis=1, scf_loop=2, sw_tail=True)
    F.set_precision(prec)
    a, mu = F.mkself(*args, **kw)
    b, mub = O.mkself(*args, **kw)
    tol = 1e-10 if prec == 0 else 1e-5
    assert np.abs(a - b).max() <= tol * np.abs(b).max() and abs(mu - mub) < tol


def test_gap(F):
    st = MD.two_orbital(*MESH, Nw=NW, temp=TEMP, mu=0.1, U=0.6, J=0.1)
    chi = O.get_chi0_conv(st['Gk'], st['kmap'], st['invk'], st['olist'], TEMP, *MESH)
    init = np.cos(2 * np.pi * st['klist'][:, 0])[None] * np.ones((2, 1)) + 0.3
    args = (st['Gk'], st['uni'], init, st['Smat'], st['Cmat'], st['olist'], st['plist'], st['kmap'], st['invk'], *MESH,
            TEMP, 0)
    d, lam = F.linearized_eliashberg(chi.copy(), *args, eps=1e-3, itemax=3, arnoldi_m=0)
    r, lref = O.linearized_eliashberg(chi.copy(), *args, eps=1e-3, itemax=3, arnoldi_m=0)
    assert abs(lam - lref) <= 1e-9 * max(1.0, abs(lref))
    assert np.abs(d - r).max() <= 1e-9 * max(np.abs(r).max(), 1e-3)


def test_spinful_chi0(F):
    st = MD.spinful(MD.two_orbital(*MESH, Nw=NW, temp=TEMP, mu=0.1), lam=0.1, alpha=0.1, U=0.5, J=0.1)
    args = (st['Vmat'], st['Gk'], st['olist'], st['slist'], st['kmap'], st['invk'], st['invs'], TEMP, *MESH)
    a, r = F.get_chi0_soc(*args)[0], O.get_chi0_soc(*args)[0]
    assert np.abs(a - r).max() <= 1e-11 * np.abs(r).max()
