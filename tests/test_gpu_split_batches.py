"""Batches of transforms that take several launches (more grids than a launch
holds): chi0 of three orbitals against the oracle, 45 pairs where a launch takes
32; and the whole FLEX loop and the gap equation on meshes so large that a
launch takes two or three of the four outputs.  For those the model has no
hopping: nothing depends on k, and every k has what the oracle solves on four
points.  FP64: 1e-11 of the largest element for a transform, 1e-10 after a
loop; FP32 transforms 4e-6, and 1e-5 after a loop (the increments' rounding)."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu

TEMP, MU = 0.05, 0.1
HAM = np.array([[[0.1, 0.15], [0.15, -0.2]]], dtype=np.complex128)


@pytest.fixture
def F():
    import pyrpa_amd.flibs as F
    yield F
    F.set_precision(0)
    F.release_memory()


@pytest.mark.parametrize("prec", [0, 1])
def test_chi0(F, prec):
    dims, nw = (16, 16, 4), 128
    st = MD.random_model(3, *dims, nw, TEMP, MU, 0.5, 0.1, seed=2)
    args, mesh = (st['Smat'], st['Cmat'], st['Gk']), (st['olist'], st['kmap'], st['invk'])
    F.set_precision(prec)
    a = F.get_chi0(*args, *mesh, TEMP, *dims)[0]
    b = F.get_chi0_tail(*args, st['eig'], st['uni'], *mesh, st['mu'], TEMP, *dims)[0]
    ra = O.get_chi0(*args, *mesh, TEMP, *dims)[0]
    rb = O.get_chi0_tail(*args, st['eig'], st['uni'], *mesh, st['mu'], TEMP, *dims)[0]
    tol = 1e-11 if prec == 0 else 4e-6
    assert np.abs(a - ra).max() <= tol * np.abs(ra).max()
    assert np.abs(b - rb).max() <= tol * max(np.abs(rb).max(), np.abs(ra).max())


def local(L, dims, nw):
    klist, kmap, invk = L.gen_irr_k_TRS(*dims)
    hamk = L.gen_ham(klist, HAM, np.zeros((1, 3)))
    eig, uni = L.get_eig(hamk)
    olist, site = O.get_chi_orb_list(2, [2])
    S, C = O.get_scmat(olist, site, 0.1, 0.02)  # below the Stoner instability of free levels
    return dict(kmap=kmap, invk=invk, hamk=hamk, eig=eig, uni=uni, olist=olist, S=S, C=C, dims=dims, nw=nw)


def flex(L, m, **kw):
    return L.mkself(m['S'], m['C'], m['kmap'], m['invk'], m['olist'], m['hamk'], m['eig'], m['uni'], MU, 0.8, TEMP,
                    m['nw'], *m['dims'], False, False, eps=0.0, pp=0.5, m_diis=1, scf_loop=3, **kw)


@pytest.mark.parametrize("dims,nw", [((32, 32, 8), 256), ((30, 30, 6), 270)])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("tail", [False, True])
def test_flex(F, dims, nw, prec, tail):
    ref, mu1 = flex(O, local(O, (4, 1, 1), nw), sw_tail=tail)
    F.set_precision(prec)
    sig, mu = flex(F, local(F, dims, nw), sw_tail=tail)
    tol = 1e-10 if prec == 0 else 1e-5
    assert np.abs(sig - ref[..., :1]).max() <= tol * np.abs(ref).max() and abs(mu - mu1) < tol


@pytest.mark.parametrize("dims,nw", [((32, 32, 8), 256), ((30, 30, 6), 270)])
def test_gap(F, dims, nw):
    """chi and the vertex it leaves as (> 8 MB, copied out beside the solver) are the same at every k too; the
    gap's norm is 1 over the zone."""
    out = []
    for L, d in ((O, (4, 1, 1)), (F, dims)):
        m = local(L, d, nw)
        nk = len(m['hamk'])
        g = O.gen_Green0(m['eig'][:1], m['uni'][:1], MU, TEMP, nw)
        G = np.ascontiguousarray(np.repeat(g, nk, axis=3))
        one = local(O, (1, 1, 1), nw)
        c = O.get_chi0_conv(g, one['kmap'], one['invk'], one['olist'], TEMP, 1, 1, 1)
        chi = np.ascontiguousarray(np.repeat(c, nk, axis=3))
        D, lam = L.linearized_eliashberg(chi, G, m['uni'], np.ones((2, nk)), m['S'], m['C'], m['olist'], np.ones(2),
                                         m['kmap'], m['invk'], *d, TEMP, 0, eps=1e-12, itemax=3, arnoldi_m=0)
        out.append((D * np.sqrt(np.prod(d)), lam, O.get_V_delta(c, m['S'], m['C']), chi))
    (D0, lam0, V, _), (D, lam, _, chi) = out
    assert abs(lam - lam0) <= 1e-9 * abs(lam0)
    assert np.abs(D - D0[..., :1]).max() <= 1e-9 * np.abs(D0).max()
    assert np.abs(chi - V).max() <= 1e-11 * np.abs(V).max()
