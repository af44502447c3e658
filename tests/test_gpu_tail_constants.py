"""The tail constants of chi0 formed on the device (rhobar, J, the sawtooth
table) through get_chi0_tail against the oracle, where they are most of the
result: very few frequencies (the sawtooth's power series covers pi j / M <
1/4, its cotangent the rest), meshes below and above one work-group of
points, one and several orbitals, levels far from mu.  Both sides work in
FP64; 1e-12 of the largest element covers the transforms' rounding (a few
log2 N ulp) with a margin of about 100."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O
from tests import models as MD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norb,nx,nz,nw,mu,temp", [
    (1, 4, 1, 1, 0.0, 0.1), (1, 20, 1, 3, -0.3, 0.02), (2, 5, 3, 2, 0.1, 0.05), (3, 4, 2, 40, 3.0, 0.004),
    (4, 6, 1, 9, -4.0, 0.01)])
def test_tail_chi0_at_few_frequencies(norb, nx, nz, nw, mu, temp):
    import pyrpa_amd.flibs as F
    F.set_precision(0)
    st = MD.random_model(norb, nx, nx, nz, nw, temp, mu, 0.6, 0.1, seed=norb)
    args = (st['Smat'], st['Cmat'], st['Gk'], st['eig'], st['uni'], st['olist'], st['kmap'], st['invk'], mu, temp,
            nx, nx, nz)
    chi, _ = F.get_chi0_tail(*args)
    ref, _ = O.get_chi0_tail(*args)
    assert np.abs(chi - ref).max() <= 1e-12 * max(np.abs(ref).max(), 1.0)
