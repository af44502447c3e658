"""Sums of the Eliashberg solvers (power step, Gram-Schmidt chain) and of the
DIIS mixing where their launches differ: fewer elements than one work-group,
between one group and the 1024 of the fixed summation order, and more than
those hold at once (1024 x 256 elements).  The oracle sums in another order;
both Eliashberg settings are stopped after a few steps, before rounding is
amplified, so 1e-9 of the eigenvalue holds with a wide margin."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nw,arnoldi", [(2, 2, 0), (4, 8, 0), (4, 8, 3), (8, 9, 5), (32, 520, 0), (32, 520, 2)])
def test_eliashberg_sums(nx, nw, arnoldi):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    st = MD.one_orbital(Nx=nx, Ny=nx, Nw=nw, temp=0.1, mu=-0.3, tx=1.0, ty=1.0, U=1.0)
    chi = F.get_chi0_conv(st['Gk'], st['kmap'], st['invk'], st['olist'], st['temp'], nx, nx, 1)
    init = np.cos(2 * np.pi * st['klist'][:, 0])[None] + 0.3
    args = (st['Gk'], st['uni'], init, st['Smat'], st['Cmat'], st['olist'], st['plist'], st['kmap'], st['invk'], nx,
            nx, 1, st['temp'], 0 if arnoldi == 0 else 1)
    d, lam = F.linearized_eliashberg(chi.copy(), *args, eps=1e-3, itemax=5, arnoldi_m=arnoldi)
    r, lref = O.linearized_eliashberg(chi.copy(), *args, eps=1e-3, itemax=5, arnoldi_m=arnoldi)
    assert abs(lam - lref) <= 1e-9 * max(1.0, abs(lref))
    assert np.abs(d - r).max() <= 1e-9 * max(np.abs(r).max(), 1e-3)


@pytest.mark.parametrize("m_diis", [2, 3, 9])
def test_diis_history(m_diis):
    """More iterations than history entries (the Gram matrix's rows are
    replaced in turn) and more entries than one combination launch takes."""
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    st = MD.two_orbital(Nx=4, Ny=4, Nw=8, temp=0.1, mu=0.0, U=0.8, J=0.1)
    args = (st['Smat'], st['Cmat'], st['kmap'], st['invk'], st['olist'], st['hamk'], st['eig'], st['uni'], 0.0, 0.9,
            st['temp'], 8, 4, 4, 1, False, False)
    kw = dict(eps=0.0, pp=0.3, m_diis=m_diis, scf_loop=11 if m_diis > 5 else 6)
    a, mu = F.mkself(*args, **kw)
    b, mub = O.mkself(*args, **kw)
    assert np.abs(a - b).max() <= 1e-8 * np.abs(b).max() and abs(mu - mub) < 1e-8
