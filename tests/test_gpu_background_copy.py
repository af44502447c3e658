"""The vertex that leaves by the in/out chi while the Eliashberg solver runs:
arrays above 8 MB (below, the copy is complete before the solver starts) that
are no multiple of the 2 MB pieces, every element, with the power and the
Arnoldi solver and with a solver that raises.  Spinless against the oracle's
vertex (1e-11: the solves of a 4 x 4 system of condition number below 100),
spinful bit for bit against the vertex by its own entry point."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu

TEMP = 0.1


@pytest.mark.parametrize("solver", ["power", "arnoldi", "raises"])
@pytest.mark.parametrize("gap_sym", [0, -1])
def test_spinless(solver, gap_sym):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    st = MD.two_orbital(Nx=16, Ny=16, Nw=301, temp=TEMP, mu=0.1, U=0.8, J=0.1)
    chi0 = F.get_chi0_conv(st['Gk'], st['kmap'], st['invk'], st['olist'], TEMP, 16, 16, 1)
    assert chi0.nbytes > (8 << 20) and chi0.nbytes % (2 << 20)
    G = np.zeros_like(st['Gk']) if solver == "raises" else st['Gk']  # no pair amplitude: the norm is 0
    init = np.cos(2 * np.pi * st['klist'][:, 0])[None] * np.ones((2, 1)) + 0.3
    args = (G, st['uni'], init, st['Smat'], st['Cmat'], st['olist'], st['plist'], st['kmap'], st['invk'], 16, 16, 1,
            TEMP, gap_sym)
    want = O.get_V_delta(chi0, st['Smat'], st['Cmat'], gap_sym >= 0)
    for _ in range(2):
        chi = chi0.copy()
        if solver == "raises":
            with pytest.raises(RuntimeError):
                F.linearized_eliashberg(chi, *args, eps=1e-6, itemax=3, arnoldi_m=0)
        else:
            F.linearized_eliashberg(chi, *args, eps=1e-6, itemax=3, arnoldi_m=3 if solver == "arnoldi" else 0)
        assert np.abs(chi - want).max() <= 1e-11 * np.abs(want).max()


@pytest.mark.parametrize("solver", ["power", "arnoldi", "raises"])
def test_spinful(solver):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    nx, nw = 8, 75
    st = MD.spinful(MD.two_orbital(Nx=nx, Ny=nx, Nw=nw, temp=TEMP, mu=0.1), lam=0.1, alpha=0.1, U=0.8, J=0.1)
    chi0, sg, sg2, isc = F.get_chi0_soc(st['Vmat'], st['Gk'], st['olist'], st['slist'], st['kmap'], st['invk'],
                                        st['invs'], TEMP, nx, nx, 1)
    assert chi0.nbytes > (8 << 20) and chi0.nbytes % (2 << 20)
    want = F.get_V_soc_flex(chi0.copy(), st['Vmat'])
    G = np.zeros_like(st['Gk']) if solver == "raises" else st['Gk']
    args = (G, st['uni'], O.gap_symms(st['klist'], 4, 1), st['Vmat'], sg, sg2, np.ones(4), st['slist'], st['olist'],
            st['kmap'], st['invk'], st['invs'], isc, nx, nx, 1, TEMP, 1)
    for _ in range(2):
        chi = chi0.copy()
        if solver == "raises":
            with pytest.raises(RuntimeError):
                F.linearized_eliashberg_soc(chi, *args, eps=1e-6, itemax=3, arnoldi_m=0)
        else:
            F.linearized_eliashberg_soc(chi, *args, eps=1e-6, itemax=3, arnoldi_m=3 if solver == "arnoldi" else 0)
        assert np.array_equal(chi, want)
