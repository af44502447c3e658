"""The work that users of this package have it do, as timed cases.

Every case is a call (or the usual sequence of calls) of `pyrpa_amd.flibs` and
`pyrpa_amd.lattice` on numpy arrays, as a script that drives the library makes
them: a FLEX self-energy solve (`mkself`, spinless or spinful), an RPA
susceptibility (`get_chi0` / `get_chi0_tail` with the Stoner factor, then the
static chi_s and chi_c), or a linearized Eliashberg solve.  Sizes follow the
repository's workloads (`lattice.config`), its tests and the default mesh of
the drivers (32x32x4 with 256 frequencies); the lattices are its synthetic
ones, with hoppings drawn from the seed.

A case is a dict: `kind` (flex, soc, rpa, eliash), `norb`, the k-mesh `nx`,
`ny`, `nz`, the number of fermionic Matsubara frequencies `nw`, the transform
precision `prec` (`flibs.set_precision`: 0 FP64, 1 FP32 transforms), `tail`
(the Matsubara tail correction of chi0), `temp`, `U`, `J`, and the loop's
settings: `m_diis` and `eps` (flex, soc), `arnoldi` (eliash: Krylov dimension,
0 the power method)."""
import math

import numpy as np
import torch

from pyrpa_amd import flibs as F
from pyrpa_amd import lattice as L


def _case(kind, norb, nx, ny, nz, nw, prec=0, tail=True, m_diis=1, eps=1e-8, arnoldi=10):
    one = norb == 1
    temp = 0.02 if one and nw >= 512 else 0.05 if one else 0.04
    U = {"flex": 2.0 if one else 0.8, "soc": 0.8, "rpa": 0.8, "eliash": 1.6 if one else 0.8}[kind]
    J = 0.0 if one and kind != "soc" else 0.1
    c = dict(kind=kind, norb=norb, nx=nx, ny=ny, nz=nz, nw=nw, prec=prec, tail=tail, temp=temp, U=U, J=J)
    if kind in ("flex", "soc"):
        c.update(m_diis=m_diis, eps=eps)
    if kind == "eliash":
        c.update(arnoldi=arnoldi)
    return c


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # a quick look at a model: the smallest mesh that tests and first runs
        # use, default mixing; all of it is latency
        named("flex_2orb_8x8_w32", "flex", 2, 8, 8, 1, 32, tail=False, m_diis=5, eps=1e-4),
        # one training solve of the learned warm start (thousands of them are run)
        named("flex_1orb_32x32_w256", "flex", 1, 32, 32, 1, 256),
        # one-orbital FLEX to a tight tolerance (the 64x64 x 1024 workload)
        named("flex_1orb_64x64_w1024", "flex", 1, 64, 64, 1, 1024),
        # two orbitals on the drivers' default mesh, default mixing (DIIS)
        named("flex_2orb_32x32x4_w256", "flex", 2, 32, 32, 4, 256, m_diis=5, eps=1e-4),
        # odd and ragged sizes: a mesh commensurate with a three-fold cell
        named("flex_3orb_27x27x5_w90", "flex", 3, 27, 27, 5, 90, m_diis=5, eps=1e-4),
        # the four-orbital 3D lattice in FP64, and with FP32 increments
        named("flex_4orb_16x16x8_w256", "flex", 4, 16, 16, 8, 256, m_diis=5, eps=1e-4),
        named("flex_4orb_16x16x8_w256_mixed", "flex", 4, 16, 16, 8, 256, prec=1, eps=1e-6),
        # spin-orbit FLEX: two orbitals with spin, 16 orbital pairs
        named("soc_flex_2orb_16x16_w128", "soc", 2, 16, 16, 1, 128, tail=False, m_diis=5, eps=1e-4),
        # the RPA scan of a five-orbital 2D model: tail-corrected chi0 on all
        # bosonic frequencies, Stoner factor, static chi_s and chi_c
        named("rpa_5orb_32x32_w64", "rpa", 5, 32, 32, 1, 64),
        # the same steps with FP32 transforms on a 3D mesh of mixed radices
        named("rpa_3orb_24x24x6_w100_f32", "rpa", 3, 24, 24, 6, 100, prec=1, tail=False),
        # Eliashberg eigenvalue by the power method (one orbital, d wave)
        named("eliash_1orb_64x64_w1024_power", "eliash", 1, 64, 64, 1, 1024, tail=False, arnoldi=0),
        # Eliashberg with the drivers' default Arnoldi on a multi-orbital model
        named("eliash_3orb_20x20x4_w128", "eliash", 3, 20, 20, 4, 128, tail=False),
    ]


def draw(rng):
    """One more case of the same ranges."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    most = 0.4 * max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["flex"] * 5 + ["soc", "rpa", "rpa", "eliash", "eliash"])
        norb = 2 if kind == "soc" else rng.choice([1, 1, 2, 3, 4, 5] if kind == "rpa" else [1, 1, 2, 2, 3, 4])
        nx = log_int(8, 64)
        ny = nx if rng.random() < 0.6 else log_int(8, 64)
        if nx % 2 and not ny % 2:  # the mesh tables take an odd first axis with an odd second one only
            nx, ny = ny, nx
        nz = 1 if rng.random() < 0.5 else log_int(2, 10)
        nw = log_int(32, 1024 if norb == 1 else 256)
        if nw > 256:
            nw -= nw % 8
        prec = 1 if kind in ("flex", "rpa") and rng.random() < 0.25 else 0
        tail = kind in ("flex", "rpa") and rng.random() < 0.6
        tight = rng.random() < 0.4
        c = _case(kind, norb, nx, ny, nz, nw, prec=prec, tail=tail, m_diis=1 if tight or prec else 5,
                  eps=1e-6 if tight or prec else 1e-4, arnoldi=rng.choice([0, 10]) if norb == 1 else 10)
        if _cost(c) <= most:
            return c


# --------------------------------------------------------------------------- inputs
def _lattice(case, seed):
    """(rvec, ham_r, filling per spin) of the case's model: the repository's
    synthetic lattices, hoppings from the seed."""
    rng = np.random.default_rng(1000 + seed)
    norb, nz = case["norb"], case["nz"]
    if norb == 1:
        rvec, ham_r = L.square_lattice(1.0, -0.25 + 0.05 * rng.uniform(-1, 1), tz=0.1 if nz > 1 else 0.0)
        fill = 0.425
    else:
        in_plane = [(1, 0, 0), (0, 1, 0), (1, 1, 0), (1, -1, 0)]
        inter = [(0, 0, 1), (1, 0, 1)] if nz > 1 else []
        rvec, ham_r = L.synthetic_lattice(norb, in_plane, 0.4, 0.3, L.SEED_BASE + norb, inter=inter, inter_scale=0.2)
        # one material, its amplitudes changed by a few per cent (pressure, doping, another fit); H(-R) = H(R)^T
        for i in range(1, len(rvec), 2):
            ham_r[i] *= 1.0 + 0.05 * rng.uniform(-1, 1, ham_r[i].shape)
            ham_r[i + 1] = ham_r[i].T
        fill = 0.45 * norb
    return rvec, ham_r, fill


def _spinful(rvec, ham_r, rng):
    """The spinful basis (spin up first) with an atomic term lambda L_z s_z
    and a Rashba hopping, both time-reversal symmetric."""
    hs = np.array([np.kron(np.eye(2), h) for h in ham_r])
    sx, sy, sz = (np.array(m, dtype=complex) for m in ([[0, 1], [1, 0]], [[0, -1j], [1j, 0]], [[1, 0], [0, -1]]))
    lam, alpha = 0.1 * rng.uniform(0.5, 1.0), 0.05 * rng.uniform(0.5, 1.0)
    rashba = {(1, 0, 0): 1j * alpha * sy, (0, 1, 0): -1j * alpha * sx}
    for i, R in enumerate(rvec):
        R = tuple(int(v) for v in R)
        minus = tuple(-v for v in R)
        if R == (0, 0, 0):
            hs[i] += 0.5 * lam * np.kron(sz, np.array([[0, -1j], [1j, 0]]))
        elif R in rashba:
            hs[i] += np.kron(rashba[R], np.eye(2))
        elif minus in rashba:
            hs[i] += np.kron(rashba[minus], np.eye(2)).conj().T
    return hs


def prepare(case, seed):
    F.set_precision(0)
    rvec, ham_r, fill = _lattice(case, seed)
    if case["kind"] == "soc":
        ham_r = _spinful(rvec, ham_r, np.random.default_rng(2000 + seed))
        fill *= 2
    st = L.build(rvec, ham_r, case["nx"], case["ny"], case["nz"], case["nw"], case["temp"], case["U"], case["J"],
                 fill)
    state = {"case": dict(case), "st": st}
    if case["kind"] == "soc":
        No = st["Norb"]
        slist = np.array([1] * (No // 2) + [-1] * (No // 2), dtype=np.int64)
        invs = np.array(list(range(No // 2, No)) + list(range(No // 2)), dtype=np.int64) + 1
        state.update(slist=slist, invs=invs,
                     Vmat=F.gen_Vmatrix(st["olist"], slist, st["site"], invs, case["U"], case["J"]))
    if case["kind"] in ("rpa", "eliash"):
        state["G"] = F.gen_Green0(st["eig"], st["uni"], st["mu"], st["temp"], st["Nw"])
    if case["kind"] == "eliash":
        state["chi"], _ = F.get_chi0(st["Smat"], st["Cmat"], state["G"], st["olist"], st["kmap"], st["invk"],
                                     st["temp"], st["Nx"], st["Ny"], st["Nz"])
        state["vertex"] = np.empty_like(state["chi"])
        gap = L.gap_symms(st["klist"], st["Norb"], 1)
        rng = np.random.default_rng(3000 + seed)
        state["init"] = gap * rng.uniform(0.8, 1.2, (st["Norb"], 1))
    return state


# --------------------------------------------------------------------------- one pass
def run(state):
    case, st = state["case"], state["st"]
    mesh = (st["Nx"], st["Ny"], st["Nz"])
    F.set_precision(case["prec"])
    if case["kind"] == "flex":
        sigma, mu = L.flex(st, eps=case["eps"], pp=0.5, m_diis=case["m_diis"], scf_loop=60, sw_tail=case["tail"])
        return {"sigma": sigma, "mu": mu}
    if case["kind"] == "soc":
        sigma, mu = F.mkself_soc(state["Vmat"], st["kmap"], st["invk"], state["invs"], st["olist"], state["slist"],
                                 st["hamk"], st["eig"], st["uni"], st["mu"], st["fill"], st["temp"], st["Nw"], *mesh,
                                 False, False, scf_loop=60, eps=case["eps"], pp=0.5, m_diis=case["m_diis"],
                                 sw_rescale=True)
        return {"sigma": sigma, "mu": mu}
    if case["kind"] == "rpa":
        if case["tail"]:
            chi, stoner = F.get_chi0_tail(st["Smat"], st["Cmat"], state["G"], st["eig"], st["uni"], st["olist"],
                                          st["kmap"], st["invk"], st["mu"], st["temp"], *mesh)
        else:
            chi, stoner = F.get_chi0(st["Smat"], st["Cmat"], state["G"], st["olist"], st["kmap"], st["invk"],
                                     st["temp"], *mesh)
        chis, chic = F.get_chis_chic(chi, st["Smat"], st["Cmat"])
        return {"chi0": chi, "stoner": stoner, "chis": chis, "chic": chic}
    # the solver leaves the pairing vertex in the array that held chi0
    np.copyto(state["vertex"], state["chi"])
    delta, lam = F.linearized_eliashberg(state["vertex"], state["G"], st["uni"], state["init"], st["Smat"],
                                         st["Cmat"], st["olist"], st["plist"], st["kmap"], st["invk"], *mesh,
                                         st["temp"], 1, eps=1e-5, arnoldi_m=case["arnoldi"])
    return {"delta": delta, "lambda": lam, "vertex": state["vertex"]}


def _sizes(case):
    """(irreducible (k, w) points, full (k, tau) grid points, orbitals, orbital pairs)"""
    no = case["norb"] * (2 if case["kind"] == "soc" else 1)
    nk = case["nx"] * case["ny"] * case["nz"]
    return (nk // 2 + 1) * case["nw"], 2 * nk * case["nw"], no, no * no


#: iterations that the loops typically take: linear mixing (one history entry)
#: gains a factor of two each, DIIS more; both Arnoldi passes or a power run
def _iterations(case):
    if case["kind"] in ("flex", "soc"):
        return round(4 - math.log2(case["eps"])) if case["m_diis"] == 1 else 12
    return {"rpa": 1, "eliash": 20}[case["kind"]]


def _cost(case):
    """Rough seconds at full rates; lengths with large prime factors, whose
    transforms take many more operations, count for more"""
    rough = 1.0
    for n in (case["nx"], case["ny"], case["nz"], 2 * case["nw"]):
        for p in (2, 3, 5, 7):
            while n % p == 0:
                n //= p
        rough = max(rough, n / 2)
    w = work(case)
    return rough * (w["bytes"] / 5e12 + w["flops"] / 2e13)


def work(case):
    """Bytes and operations that the path cannot do without.  An iteration
    reads and writes its fields once (G and Sigma: No^2 numbers per (k, w),
    chi0 and the vertex: Nchi^2; a gap iteration: Delta, F and the vertex) and
    transforms each once (5 n log2 n per transform of the full grid); the
    vertex takes two inversions and six products of Nchi x Nchi matrices."""
    nkw, n, no, nchi = _sizes(case)
    it = _iterations(case)
    fft = 5.0 * n * math.log2(n)
    pairs = nchi * (nchi + 1) / 2
    gemm = 8.0 * nchi ** 3
    if case["kind"] in ("flex", "soc"):
        by = it * 16.0 * nkw * (2 * no * no + 2 * nchi * nchi)
        fl = it * (fft * (2 * no * no + 2 * pairs) + nkw * gemm * 4)
    elif case["kind"] == "rpa":
        by = 16.0 * nkw * (no * no + nchi * nchi)
        fl = fft * (no * no + pairs)
    else:
        by = 16.0 * nkw * 3 * nchi * nchi + it * 16.0 * (n / 2) * (2 * no * no) + it * 16.0 * nkw * nchi * nchi
        fl = fft * (nchi * nchi + it * 2 * no * no) + nkw * gemm * 4
    return {"bytes": by, "flops": fl}


# --------------------------------------------------------------------------- the same in plain torch, 64 bits
class _Grid:
    """The mesh of a case on the GPU: unfolding of irreducible k points to the
    full zone by time reversal, and the transforms over (tau, z, y, x)."""

    def __init__(self, st, spin=None, inv=None):
        dev = "cuda"
        self.Nx, self.Ny, self.Nz, self.Nw = st["Nx"], st["Ny"], st["Nz"], st["Nw"]
        self.S, self.M, self.T = self.Nx * self.Ny * self.Nz, 2 * self.Nw, st["temp"]
        kmap, invk = st["kmap"], st["invk"]
        sp = kmap[:, 0] + self.Nx * (kmap[:, 1] + self.Ny * kmap[:, 2])
        irr, flag, self.Nk = np.empty(self.S, np.int64), np.empty(self.S, bool), len(st["klist"])
        irr[sp], flag[sp] = invk[:, 0] - 1, invk[:, 1] == 1
        first = np.empty(self.Nk, np.int64)
        d = invk[:, 1] == 0
        first[invk[d, 0] - 1] = sp[d]
        self.irr, self.flag = torch.from_numpy(irr).to(dev), torch.from_numpy(flag).to(dev)
        self.first = torch.from_numpy(first).to(dev)
        self.spin, self.inv = spin, inv
        self.kw = torch.from_numpy(np.bincount(invk[:, 0] - 1, minlength=self.Nk).astype(np.float64)).to(dev)
        ol = np.asarray(st["olist"]).ravel(order="K").reshape(2, -1).T - 1
        self.ol = [tuple(int(v) for v in r) for r in ol]
        self.wn = (2 * torch.arange(self.Nw, device=dev, dtype=torch.float64) + 1) * math.pi * self.T

    def turned(self, G, a, b):
        """G_ab at the -k image of an irreducible point: the transpose, with
        the spins flipped in a spinful basis"""
        if self.spin is None:
            return G[b, a]
        return G[self.inv[b], self.inv[a]] * (self.spin[a] * self.spin[b])

    def zone(self, direct, turned):
        return torch.where(self.flag, turned[:, self.irr], direct[:, self.irr])

    def fft(self, x, inverse=False, space_only=False):
        y = x.reshape(-1, self.Nz, self.Ny, self.Nx)
        dims = (1, 2, 3) if space_only else (0, 1, 2, 3)
        return (torch.fft.ifftn(y, dim=dims) if inverse else torch.fft.fftn(y, dim=dims)).reshape(x.shape)

    def back(self, x, tau=True):
        """x(-r, -tau) (or x(-r, tau))"""
        y = x.reshape(self.M, self.Nz, self.Ny, self.Nx)
        dims = (0, 1, 2, 3) if tau else (1, 2, 3)
        return torch.roll(torch.flip(y, dims), [1] * len(dims), dims).reshape(x.shape)

    def greens(self, G):
        """Transforms of G_ab, [a][b]: slots w_j, then the negative ones"""
        no = len(G)
        pos = [[self.zone(G[a, b], self.turned(G, a, b)) for b in range(no)] for a in range(no)]
        return [[self.fft(torch.cat([pos[a][b], pos[b][a].conj().flip(0)])) for b in range(no)] for a in range(no)]

    def boson(self, V, m, l, static):
        pos, neg = self.zone(V[m, l], V[l, m]), self.zone(V[l, m], V[m, l])
        return torch.cat([pos, torch.full_like(pos[:1], static), neg[1:].conj().flip(0)])

    def gather(self, x):
        return x[: self.Nw, self.first]


def _threshold(x):
    return torch.complex(torch.where(x.real.abs() < 1e-9, 0.0, x.real), torch.where(x.imag.abs() < 1e-9, 0.0, x.imag))


def _inverse(A):
    """Inverses of A[n, n, ...] by Gauss-Jordan elimination with row pivoting."""
    n = len(A)
    A = torch.cat([A, torch.zeros_like(A)], 1)
    for k in range(n):
        A[k, n + k] = 1.0
    for k in range(n):
        if k + 1 < n:
            p = A[k:, k].abs().argmax(0, keepdim=True) + k
            take = p.expand(1, *p.shape[1:])
            pivot = torch.gather(A, 0, take.unsqueeze(1).expand(1, 2 * n, *p.shape[1:]))[0]
            A.scatter_(0, take.unsqueeze(1).expand(1, 2 * n, *p.shape[1:]), A[k : k + 1].clone())
            A[k] = pivot
        row = A[k] / A[k, k].clone()
        for i in range(n):
            if i != k:
                A[i] -= A[i, k].clone() * row
        A[k] = row
    return A[:, n:]


def _mul(A, B):
    """Products of matrices held as [n, n, ...]; either may be a plain n x n one"""
    n = len(A)
    out = []
    for i in range(n):
        row = None
        for k in range(n):
            a, b = A[i, k], B[k]
            if a.ndim == 0 and float(a.abs()) == 0.0:
                continue
            if a.ndim == 0:
                t = a * b
            elif b.ndim == 1:
                t = a.unsqueeze(0) * b.reshape(-1, *([1] * a.ndim))
            else:
                t = a.unsqueeze(0) * b
            row = t if row is None else row + t
        out.append(torch.zeros_like(out[0]) if row is None and out else row)
    like = next(r for r in out if r is not None)
    return torch.stack([torch.zeros_like(like) if r is None else r for r in out])


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda")


def _fields(py):
    """[p, q, w, k] of an array in the library's layout [q, p, w, k]"""
    return _dev(py).transpose(0, 1).contiguous()


def _green0(g, st, mu):
    e, U = _dev(st["eig"]), _dev(st["uni"])  # U[k, band, orbital]
    den = 1.0 / (mu + 1j * g.wn[None, :, None] - e.T[:, None, :])
    no = e.shape[1]
    c = [[U[:, :, a] * U[:, :, b].conj() for b in range(no)] for a in range(no)]
    return torch.stack([torch.stack([sum(c[a][b][:, n] * den[n] for n in range(no)) for b in range(no)])
                        for a in range(no)])


def _pairs(g):
    """The computed orbital pairs (l, m) and the partner (l', m') of each:
    chi_{1234} = chi*_{4321}, with the spins flipped in a spinful basis"""
    inv = g.inv if g.inv is not None else list(range(1 + max(max(p) for p in g.ol)))
    where = {p: i for i, p in enumerate(g.ol)}
    seen, out = set(), []
    for l, (l1, l2) in enumerate(g.ol):
        for m, (m1, m2) in enumerate(g.ol):
            q = (where[(inv[m2], inv[m1])], where[(inv[l2], inv[l1])])
            if q not in seen:
                seen.add((l, m))
                out.append(((l, m), q))
    return out


def _chi0(g, G, st, mu, tail):
    """chi[m, l, w, k] of G by convolution; with the tail, minus that of G0
    plus the analytic one of G0 on the tau grid"""
    Fg = g.greens(G)
    n = len(g.ol)
    chi = torch.zeros((n, n, g.Nw, g.Nk), dtype=torch.complex128, device="cuda")
    w = g.T / g.S
    if tail:
        F0 = g.greens(_green0(g, st, mu))
        e, U = _dev(st["eig"]), _dev(st["uni"])
        no, beta = e.shape[1], 1.0 / g.T
        xi = (e - mu).T[:, None, :]  # [band, 1, k]
        tau = (torch.arange(g.M, device="cuda", dtype=torch.float64) * (beta / g.M))[None, :, None]
        up = xi >= 0
        d = 1.0 + torch.exp(-beta * xi.abs())
        fall, rise = torch.exp(-xi.abs() * tau) / d, torch.exp(-xi.abs() * (beta - tau)) / d
        gp, gm = -torch.where(up, fall, rise), torch.where(up, rise, fall)
        f = (torch.where(up, d - 1.0, torch.ones_like(d)) / d)[:, 0]
        TA, TB = [[None] * no for _ in range(no)], [[None] * no for _ in range(no)]
        rho = torch.zeros((no, no), dtype=torch.complex128, device="cuda")
        for a in range(no):
            for b in range(no):
                c = U[:, :, a] * U[:, :, b].conj()
                ab, ba = (sum((x[:, k] * y[k]) for k in range(no)) for x, y in ((c, gp), (c.conj(), gp)))
                TA[a][b] = g.fft(g.zone(ab, ba), space_only=True)
                ab, ba = (sum((x[:, k] * y[k]) for k in range(no)) for x, y in ((c, gm), (c.conj(), gm)))
                TB[a][b] = g.fft(g.zone(ab, ba), space_only=True)
                dens = (c.T * f).sum(0)
                rho[a, b] = g.zone(dens[None], dens.conj()[None]).mean()
        j = torch.arange(1, g.Nw, device="cuda", dtype=torch.float64)
        dtau = beta / g.M
        saw = torch.zeros(g.Nw, dtype=torch.complex128, device="cuda")
        saw[0] = -0.5 * dtau
        saw[1:] = 1j / (2 * math.pi * j * g.T) - dtau * (0.5 + 0.5j / torch.tan(math.pi * j / g.M))
        del fall, rise, gp, gm
    for (l, m), (pl, pm) in _pairs(g):
        a, b, c, d = g.ol[l][0], g.ol[m][0], g.ol[m][1], g.ol[l][1]
        x = (-w) * (Fg[a][b] * g.back(Fg[c][d]))
        sign = 1.0 if g.spin is None else float(np.prod([g.spin[o] for o in (*g.ol[l], *g.ol[m])]))
        if not tail:
            x = g.gather(g.fft(x, inverse=True))
        else:
            x = x - (TA[a][b] * g.back(TB[c][d], tau=False)) / (g.T * g.S)
            bare = w * (F0[a][b] * g.back(F0[c][d]))
            Jc = (rho[c, d] if a == b else 0.0) - (rho[a, b] if c == d else 0.0)
            if (pl, pm) == (l, m):  # conjugated between the sums
                x = (g.gather(g.fft(x, inverse=True)) + Jc * saw[:, None]).conj() + g.gather(g.fft(bare, inverse=True))
                chi[m, l] = x
                continue
            x = g.gather(g.fft(x + bare, inverse=True)) + Jc * saw[:, None]
        chi[m, l] = x
        chi[pm, pl] = sign * x.conj()
    return _threshold(chi)


def _stoner(chi, W):
    A = chi[:, :, 0].permute(2, 0, 1).cpu().numpy() @ W
    return float(np.linalg.eigvals(A).real.max())


def _rpa(chi, W, sign):
    """(1 + sign chi W)^-1 chi W"""
    X = _mul(chi, W)
    n = len(X)
    A = sign * X
    for i in range(n):
        A[i, i] += 1.0
    return X, _mul(_inverse(A), X)


class _Mu:
    """The loop's search of the chemical potential: a bracket (kept between
    the iterations while it still holds the root), then inverse quadratic
    interpolation safeguarded by bisection down to a tenth of the loop's
    residual, and a last secant step."""

    def __init__(self, fill):
        self.fill, self.kept = fill, None

    def bracket(self, n_of, mu, step):
        if self.kept:
            a, b = n_of(self.kept[0]), n_of(self.kept[1])
            if a < self.fill < b:
                return (*self.kept, a, b)
        ends = []
        for sign in (1.0, -1.0):
            x = mu + sign * step
            for _ in range(100):
                n = n_of(x)
                off = sign * (self.fill - n)
                if off <= 0:
                    break
                x += sign * (1.0 if off > 0.5 else 0.5 if off > step else step)
            ends.append((x, n))
            mu = mu if sign > 0 else x
        (hi, nhi), (lo, nlo) = ends
        return lo, hi, nlo, nhi

    def __call__(self, n_of, mu, mu_old, residual):
        eps = 1e-8 if residual > 1e-2 else 0.1 * residual
        lo, hi, flo, fhi = self.bracket(n_of, mu, max(2.0 * abs(mu - mu_old), 4.0 * eps))
        self.kept = (lo, hi)
        flo, fhi = flo - self.fill, fhi - self.fill
        fc, c, d, halved = flo, lo, 0.0, False
        for _ in range(100):
            if fc != flo and fc != fhi:
                x = (hi * flo * fc * (flo - fc) + lo * fhi * fc * (fc - fhi) + c * fhi * flo * (fhi - flo)) / (
                    (fhi - flo) * (fc - fhi) * (fc - flo))
            else:
                x = hi - fhi * (hi - lo) / (fhi - flo)
            last = abs(hi - c) if halved else abs(c - d)
            halved = 0.25 * (3.0 * lo + hi) > x or x > hi or abs(x - hi) >= 0.5 * last or last < 1e-8
            if halved:
                x = 0.5 * (hi + lo)
            if abs(hi - x) < eps:
                break
            fx = n_of(x) - self.fill
            d, c, fc = c, hi, fhi
            if flo * fx < 0:
                hi, fhi = x, fx
            else:
                lo, flo = x, fx
            if abs(flo) < abs(fhi):
                lo, hi, flo, fhi = hi, lo, fhi, flo
        return 0.5 * (lo + hi) if fhi == flo else (lo * fhi - hi * flo) / (fhi - flo)


def _exact_flex(state):
    case, st = state["case"], state["st"]
    soc = case["kind"] == "soc"
    g = _Grid(st, spin=[int(s) for s in state["slist"]], inv=[int(i) - 1 for i in state["invs"]]) if soc else _Grid(st)
    no, n = st["Norb"], len(g.ol)
    H = _dev(st["hamk"]).permute(2, 1, 0)  # [p, q, k]
    e = _dev(st["eig"])
    if soc:
        V0 = _dev(state["Vmat"].T).to(torch.complex128)
        static, stoner_of = -state["Vmat"].T, -state["Vmat"].T
    else:
        S, C = _dev(st["Smat"].T).to(torch.complex128), _dev(st["Cmat"].T).to(torch.complex128)
        static, stoner_of = (1.5 * st["Smat"] - 0.5 * st["Cmat"]).T, st["Smat"].T

    def dyson(sig, mu):
        A = -(H[:, :, None, :] + sig)
        for p in range(no):
            A[p, p] += mu + 1j * g.wn[:, None]
        return _inverse(A)

    def filling(sig, mu):
        G = dyson(sig, mu)
        dn = sum(G[p, p].real.sum() for p in range(no))
        dn = dn - (1.0 / (mu + 1j * g.wn[None, :, None] - e.T[:, None, :])).real.sum()
        return float(((0.5 - 0.5 * torch.tanh(0.5 * (e - mu) / g.T)).sum() + 2 * g.T * dn) / g.Nk)

    search, mu, hist = _Mu(st["fill"]), st["mu"], []
    mu_old = 1.2 * mu
    G = _green0(g, st, mu)
    old = torch.zeros_like(G)
    for _ in range(60):
        chi = _chi0(g, G, st, mu, case["tail"])
        alpha = _stoner(chi, stoner_of)
        if alpha >= 1.0:
            chi = chi * ((1.0 - 1e-4) / alpha)
        if soc:
            V = _mul(V0, _rpa(chi, V0, 1.0)[1])
            for i in range(n):
                for j in range(n):
                    V[i, j] -= V0[i, j]
        else:
            (AS, X), (AC, Y) = _rpa(chi, S, -1.0), _rpa(chi, C, 1.0)
            V = 1.5 * _mul(S, X) + 0.5 * _mul(C, Y) - 0.25 * _mul(S + C, AS + AC)
            for i in range(n):
                for j in range(n):
                    V[i, j] += 1.5 * S[i, j] - 0.5 * C[i, j]
            del AS, X, AC, Y
        del chi
        Fg = g.greens(G)
        acc = [[0.0] * no for _ in range(no)]
        for l in range(n):
            for m in range(n):
                a, b = g.ol[m][0], g.ol[l][0]
                v = g.fft(g.boson(V, m, l, complex(static[m, l])))
                acc[a][b] = acc[a][b] + v * Fg[g.ol[m][1]][g.ol[l][1]]
        sig = torch.stack([torch.stack([g.gather(g.fft(acc[a][b], inverse=True)) for b in range(no)])
                           for a in range(no)]) * (g.T / g.S)
        del V, Fg, acc
        sig = _threshold(sig)
        base = sig[:, :, :1]
        sig = sig - 0.5 * (base + base.transpose(0, 1).conj())
        hist = (hist + [(sig, sig - old)])[-case["m_diis"]:]
        k = len(hist)
        if case["m_diis"] > 1:
            B = np.ones((k + 1, k + 1))
            B[k, k] = 0.0
            for i in range(k):
                for j in range(k):
                    B[i, j] = float((hist[i][1].conj() * hist[j][1]).sum().real) + (1e-12 if i == j else 0.0)
            c = np.linalg.solve(B, np.array([0.0] * k + [1.0]))
            sig = sum(float(c[i]) * hist[i][0] for i in range(k))
        big = sig.abs() > 1e-10
        err = float(((old - sig).abs() / sig.abs())[big].max())
        if k < 2 or case["m_diis"] == 1:
            sig = 0.5 * sig + 0.5 * old
        if err < case["eps"]:
            break
        mu = mu_old = search(lambda x: filling(sig, x), mu, mu_old, err)
        G = dyson(sig, mu)
        old = sig
    mu = search(lambda x: filling(sig, x), mu, mu_old, err)
    return {"sigma": sig.transpose(0, 1).cpu().numpy(), "mu": mu}


def _exact_rpa(state):
    case, st = state["case"], state["st"]
    g = _Grid(st)
    chi = _chi0(g, _fields(state["G"]), st, st["mu"], case["tail"])
    S, C = st["Smat"].T, st["Cmat"].T
    A = chi[:, :, 0].permute(2, 0, 1).cpu().numpy()
    one = np.eye(len(S))
    chis, chic = np.linalg.solve(one - A @ S, A), np.linalg.solve(one + A @ C, A)
    return {"chi0": chi.transpose(0, 1).cpu().numpy(), "stoner": _stoner(chi, S),
            "chis": np.ascontiguousarray(chis.transpose(2, 1, 0)), "chic": np.ascontiguousarray(chic.transpose(2, 1, 0))}


def _exact_eliash(state):
    """The power method; of the Arnoldi solver only the vertex is restated
    (its Ritz pair after ten steps is no converged value)"""
    case, st = state["case"], state["st"]
    g = _Grid(st)
    n, no = len(g.ol), st["Norb"]
    S, C = _dev(st["Smat"].T).to(torch.complex128), _dev(st["Cmat"].T).to(torch.complex128)
    chi = _fields(state["chi"])
    V = 1.5 * _mul(S, _rpa(chi, S, -1.0)[1]) - 0.5 * _mul(C, _rpa(chi, C, 1.0)[1])
    for i in range(n):
        for j in range(n):
            V[i, j] += 0.5 * (S[i, j] + C[i, j])
    out = {"delta": None, "lambda": None, "vertex": V.transpose(0, 1).cpu().numpy()}
    if case["arnoldi"] or no > 1:
        return out
    Vf = g.fft(g.boson(V, 0, 0, complex(0.5 * (S[0, 0] + C[0, 0]))))
    G = _fields(state["G"])[0, 0]

    def apply(D):
        f = -(G * D * G.conj()).real.to(torch.complex128)
        z = g.zone(f, f)
        x = g.gather(g.fft(Vf * g.fft(torch.cat([z, z.conj().flip(0)])), inverse=True))
        return x.real.to(torch.complex128) * (g.T / g.S)

    def inner(u, v):
        return 2.0 * float((g.kw * (u.conj() * v).real).sum())

    D = _dev(state["init"][0]).to(torch.complex128)[None].expand(g.Nw, -1)
    D = D / math.sqrt(inner(D, D))
    before = 0.0
    for _ in range(300):
        new = apply(D)
        norm, lam = math.sqrt(inner(new, new)), inner(D, new)
        far = min(inner(new / norm - D, new / norm - D), inner(new / norm + D, new / norm + D)) ** 0.5
        if lam < 0.0 and far < 1e-5:
            return out  # the solver goes on with a shifted operator
        if far < 1e-5 and abs(lam - before) < 1e-5 * (abs(lam) + 1e-10):
            break
        before, D = lam, new / norm
    if lam < 0.0:
        return out
    out.update({"delta": (new / norm)[None, None].cpu().numpy(), "lambda": lam})
    return out


def exact(case, seed):
    if _cost(case) > 1.5 * max(_cost(c) for c in listed()):
        return None
    state = prepare(case, seed)
    torch.cuda.empty_cache()
    return {"flex": _exact_flex, "soc": _exact_flex, "rpa": _exact_rpa, "eliash": _exact_eliash}[case["kind"]](state)
