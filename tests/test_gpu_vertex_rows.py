"""The FLEX vertex of 9 x 9 matrices and the spinful vertex of 16 x 16 ones by
rows, against numpy's solves: batches around a work-group's matrices (8 and 16)
and more than one round of work-groups, matrices whose pivots lie off the
diagonal, sparse interactions and dense ones (the LU kernels), and a singular
matrix.  Tolerance: n^2 cond(M) ulp of the largest element of V, cond the
largest of the batch (n = 9, 16: the inverse and three sparse products)."""
import numpy as np
import pytest

import oracle.pyrpa_oracle as O

pytestmark = pytest.mark.gpu


def chi_of(n, nk, nw, scale, swap, V):
    """random chi0 [n, n, nw, nk] (Python order); `swap`: I + chi0 V has a zero diagonal at one matrix"""
    rng = np.random.default_rng(n + 10 * nk + nw)
    a = scale * (rng.standard_normal((nk, nw, n, n)) + 1j * rng.standard_normal((nk, nw, n, n)))
    if swap:
        a[-1, -1] = (np.roll(np.eye(n), 1, axis=0) - np.eye(n)) @ np.linalg.inv(V)
    return a


def interactions(kind):
    if kind == "sparse":
        olist, site = O.get_chi_orb_list(3, [3])
        return O.get_scmat(olist, site, 0.9, 0.15)
    rng = np.random.default_rng(2)
    a = rng.standard_normal((2, 9, 9)) * 0.2
    return a[0] + a[0].T, a[1] + a[1].T


@pytest.mark.parametrize("kind", ["sparse", "dense"])
@pytest.mark.parametrize("nk,nw,swap", [(1, 1, True), (7, 1, False), (4, 2, True), (3, 3, True), (17, 5, False),
                                        (300, 240, True)])
def test_flex_vertex_9(kind, nk, nw, swap):
    import pyrpa_amd.flibs as F
    S, C = (np.ascontiguousarray(x, dtype=np.float64) for x in interactions(kind))
    a = chi_of(9, nk, nw, 0.1, swap, C)
    I = np.eye(9)
    Ms, Mc = I - a @ S, I + a @ C
    W = S + C
    ref = 1.5 * S - 0.5 * C - 0.25 * (W @ a @ W) + 1.5 * S @ np.linalg.solve(Ms, a @ S) \
        + 0.5 * C @ np.linalg.solve(Mc, a @ C)
    cond = max(np.linalg.cond(Ms).max(), np.linalg.cond(Mc).max())
    got = F.get_Vsigma_nosoc_flex(np.ascontiguousarray(a.transpose(3, 2, 1, 0)), S, C).transpose(3, 2, 1, 0)
    tol = 81 * cond * np.finfo(float).eps
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("kind", ["sparse", "dense"])
@pytest.mark.parametrize("nk,nw,swap", [(1, 1, True), (15, 1, False), (4, 4, True), (17, 1, True), (300, 450, False)])
def test_spinful_vertex_16(kind, nk, nw, swap):
    import pyrpa_amd.flibs as F
    if kind == "sparse":
        slist, invs = O.soc_spin_lists(4)
        olist, site = O.get_chi_orb_list(4, [4])
        V = np.asarray(O.get_vmat_soc(olist, slist, site, invs, 0.9, 0.15)).T
    else:
        rng = np.random.default_rng(3)
        V = rng.standard_normal((16, 16)) * 0.2
        V = V + V.T
    V = np.ascontiguousarray(V)
    swap = swap and np.linalg.cond(V) < 1e6
    a = chi_of(16, nk, nw, 0.05, swap, V)
    M = np.eye(16) + a @ V
    ref = -V + V @ np.linalg.solve(M, a @ V)
    got = F.get_V_soc_flex(np.ascontiguousarray(a.transpose(3, 2, 1, 0)), V.T).transpose(3, 2, 1, 0)
    tol = 256 * np.linalg.cond(M).max() * np.finfo(float).eps
    assert np.abs(got - ref).max() <= tol * max(np.abs(ref).max(), np.abs(V).max())


def test_singular_matrix_is_an_error():
    import pyrpa_amd.flibs as F
    S, C = np.diag(np.ones(9)), np.diag(np.ones(9))
    chi = np.zeros((9, 9, 2, 3), dtype=np.complex128)
    chi[:, :, 1, 1] = np.eye(9)
    with pytest.raises(RuntimeError):
        F.get_Vsigma_nosoc_flex(chi, S, C)
