"""The K-build work of this framework's users, as cases to be timed.

A case is a system (water-like molecules, optionally spdf centres; positions,
exponents and contraction coefficients from the number `system`), a share of
its screened set quartets (1 in `sample` by index hash, the part of one rank
among many), and the way a program drives the library:

  plan       the screened call stream recorded once as a resident plan; one
             SCF step is set_P, plan_execute, get_K on host arrays
  stream     the call stream sent anew every step through the per-call ABI
             (add_prm / add_shell / add_qrt / add_qrtt / add_set), CP2K's way
  noalloc    the resident plan into the program's own device arrays
  server     a K-build request to the device-resident request loop
  integrals  the spherical integrals of every class instead of K

The seed of a state gives the densities of its SCF step (for the integrals,
another molecule).
"""
import math

import numpy as np
import torch

from libgint_amd import driver, load

C0_TABLE = None


def _case(path, **kw):
    c = {"path": path, "waters": 1, "centres": 0, "box_A": 10.0, "images": 0, "basis": 0, "np_min": 1, "np_max": 6,
         "np_centre": 16, "zmin": 0.1, "system": 0, "sample": 1, "spins": 1, "truncated": True, "tau": 0.0}
    c.update(kw)
    return c


def _workload(index, path, **kw):
    """one of the framework's own workloads"""
    p = dict(driver.CONFIGS[index])
    return _case(path, waters=p["n_water"], centres=p["n_tm"], box_A=p["box_A"], images=p["image_shells"],
                 basis=p["basis"], np_min=p["np_min"], np_max=p["np_max"], system=p["seed"], **kw)


def listed():
    cases = {
        # one molecule, one SCF step: the latency of the calls, launches and copies
        "water1_plan": _case("plan", waters=1, box_A=4.0, np_min=2, np_max=4, system=2),
        # an unrestricted dimer with the plain Coulomb operator through the per-call ABI
        "water2_coulomb_uhf_stream": _case("stream", waters=2, box_A=6.0, np_max=4, system=0, spins=2, truncated=False),
        # the integrals of one molecule, every class, in the transposed output order
        "water1_integrals": _case("integrals", waters=1, box_A=4.0, np_min=5, system=3),
        # a small periodic box, P and K in the program's own device arrays (tight loops)
        "water2_pbc27_noalloc": _case("noalloc", waters=2, box_A=7.0, images=1, np_max=3, system=0),
        # a request of a serving client: 21 atoms at liquid density, up to 3 primitives
        "water7_pbc27_server": _case("server", waters=7, box_A=5.94, images=1, np_max=3, zmin=0.6, system=3003),
        # CP2K's protocol on a small periodic system, the stream sent every step
        "water3_pbc27_stream": _case("stream", waters=3, box_A=8.0, images=1, np_max=4, system=4, sample=4),
        # the 8-molecule cluster, every set quartet, one cell
        "water8_cluster_plan": _workload(0, "plan"),
        # liquid water, 27 cells, unrestricted
        "water16_pbc27_uhf_plan": _case("plan", waters=16, box_A=9.84, images=1, np_max=8, system=1, spins=2, sample=16),
        # 32 molecules, 27 cells
        "water32_pbc27_plan": _workload(1, "plan", sample=32),
        # 64 molecules and 8 centres with f shells, 16 primitives and 4 contractions; 125 cells
        "water64_spdf8_pbc125_plan": _workload(2, "plan", sample=192),
        # the same under the mixed-precision route
        "water64_spdf8_pbc125_mixed": _workload(2, "plan", sample=1024, tau=1e-7),
        # O 4s3p2d1f / H 3s2p1d, 256 cells
        "water64_f_pbc256_plan": _case("plan", waters=64, box_A=12.4, images=3, basis=4, np_max=16, system=4, sample=4096),
    }
    return [{"name": name, **case} for name, case in cases.items()]


def draw(rng):
    """one more case of the same ranges: sizes over their logarithm, odd ones among them"""
    kind = rng.choice(("cluster", "cluster", "liquid", "liquid", "liquid", "centres", "f"))
    between = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    spins, system = rng.choice((1, 1, 2)), rng.randrange(1, 1 << 20)
    if kind == "cluster":
        w = between(1, 8)
        path = rng.choice(("plan", "stream", "noalloc", "integrals")) if w <= 2 else "plan"
        c = _case(path, waters=w, box_A=round(rng.uniform(4.0, 5.0) * w ** (1.0 / 3.0), 2), np_max=rng.randint(2, 6),
                  basis=rng.choice((0, 0, 1)), spins=1 if path == "integrals" else spins, truncated=rng.random() < 0.7)
    elif kind == "liquid":
        w = between(2, 32)
        path = rng.choice(("plan", "stream", "noalloc", "server") if w <= 4 else ("plan", "plan", "server"))
        few = path == "server"
        c = _case(path, waters=w, box_A=round((29.9 * w) ** (1.0 / 3.0) * rng.uniform(1.0, 1.5), 2), images=1,
                  np_max=rng.randint(2, 3 if few else 8), zmin=0.6 if few else 0.1, spins=1 if few else spins)
    elif kind == "centres":
        w = between(8, 64)
        m = max(1, w // 8)
        c = _case("plan", waters=w, centres=m, box_A=round((52.7 * (w + m)) ** (1.0 / 3.0), 2), images=rng.choice((1, 2)),
                  np_max=rng.randint(2, 8), np_centre=rng.randint(3, 16), spins=spins, tau=rng.choice((0.0, 0.0, 1e-7)))
    else:
        w = between(4, 64)
        c = _case("plan", waters=w, box_A=round((29.7 * w) ** (1.0 / 3.0), 2), images=rng.choice((1, 2, 3)), basis=4,
                  np_max=rng.randint(2, 8), spins=spins)
    c["system"] = system
    # the share of the list that takes about `most` operations; fewer where every quartet is sent or returned
    most = {"plan": 1e10, "server": 4e9, "noalloc": 1e9, "stream": 5e8, "integrals": 5e8}[c["path"]]
    most = math.exp(rng.uniform(math.log(0.02 * most), math.log(most)))
    c["sample"] = max(1, c["waters"] ** 3 // 8) if c["images"] else 1
    for _ in range(4):
        c["sample"] = max(1, math.ceil(c["sample"] * work(c)["flops"] / most))
    while work(c)["flops"] > most:
        c["sample"] = math.ceil(1.3 * c["sample"])
    return c if work(c)["flops"] > 1e6 else draw(rng)


def _system(case, seed=0):
    # without a density, another seed is another molecule
    other = seed if case["path"] == "integrals" else 0
    return driver.System(n_water=case["waters"], n_tm=case["centres"], box_A=case["box_A"], image_shells=case["images"],
                         basis=case["basis"], np_min=case["np_min"], np_max=case["np_max"], np_tm=case["np_centre"],
                         zmin=case["zmin"], seed=case["system"] + other)


def _densities(case, system, seed):
    """the density the list was screened with, moved as between SCF steps"""
    rng = np.random.default_rng(seed)
    P0 = system.P()
    return [P0 + 1e-3 * rng.standard_normal(P0.size) for _ in range(case["spins"])]


def _table():
    global C0_TABLE
    if C0_TABLE is None:
        C0_TABLE = driver.tcg_table()
    return C0_TABLE


class State:
    """a program's handle on its system, with its density and the array K goes to"""

    def __init__(self, case, seed):
        self.case = case
        self.lib = load()
        self.system = _system(case, seed)
        self.stream = self.system.record(sample=case["sample"])
        self.n = self.system.P_size
        self.P = _densities(case, self.system, seed)
        self.K = [np.zeros(self.n) for _ in self.P]
        self.server = None
        path = case["path"]
        self.h, self.table = driver.setup_handle(
            self.lib, "libgint_", self.system, truncated=case["truncated"], c0=_table(), P=self.P[0],
            Pb=self.P[1] if case["spins"] == 2 else None)
        if case["tau"] > 0:
            self.lib.libgint_amd_set_mixed_precision(self.h, case["tau"])
        if path in ("plan", "noalloc", "server"):
            self.lib.libgint_amd_plan_begin(self.h)
            self.stream.replay(self.table, self.h, blocks=True)
            self.lib.libgint_amd_plan_end(self.h)
        if path == "noalloc":
            self.dP = [torch.from_numpy(p).cuda() for p in self.P]
            self.dK = [torch.zeros_like(p) for p in self.dP]
        elif path == "server":
            self.server = self.lib.libgint_amd_server_create(8192, 1)
            self.client = self.lib.libgint_amd_server_add_client(self.server, self.h, self.n)
            self.times = np.zeros(3)
        elif path == "integrals":
            self.out = np.zeros(driver.tra_size(self.system, self.stream.sets()))
            self.lib.libgint_amd_set_output(self.h, driver._ptr(self.out), self.out.size)

    def __del__(self):
        if getattr(self, "server", None):
            self.lib.libgint_amd_server_destroy(self.server)
        if getattr(self, "h", None):
            self.lib.libgint_amd_destroy_handle(self.h)


def prepare(case, seed):
    return State(case, seed)


def run(s):
    lib, h, ptr, n = s.lib, s.h, driver._ptr, s.n
    path = s.case["path"]
    if path == "integrals":
        s.stream.replay_tra(s.table, h)
        lib.libgint_amd_get_output(h)
        return s.out
    if path == "server":
        request = lib.libgint_amd_server_submit(s.server, s.client, ptr(s.P[0]), ptr(s.K[0]))
        if lib.libgint_amd_server_wait(s.server, request, ptr(s.times)) != 0:
            raise RuntimeError("request refused")
        return s.K[0]
    if path == "noalloc":
        for k in s.dK:
            k.zero_()
        torch.cuda.synchronize()   # the library works on a stream of its own
        p = [x.data_ptr() for x in s.dP] + [None]
        k = [x.data_ptr() for x in s.dK] + [None]
        if lib.libgint_amd_plan_execute_noalloc(h, p[0], p[1], k[0], k[1], n) != 0:
            raise RuntimeError("plan_execute_noalloc refused the plan")
        lib.libgint_amd_synchronize(h)
        return s.dK
    if len(s.P) == 2:
        lib.libgint_set_P_polarized(h, ptr(s.P[0]), ptr(s.P[1]), n)
    else:
        lib.libgint_set_P(h, ptr(s.P[0]), n)
    if path == "stream":
        s.stream.replay(s.table, h)
    else:
        lib.libgint_amd_plan_execute(h)
    if len(s.P) == 2:
        lib.libgint_get_K_polarized(h, ptr(s.K[0]), ptr(s.K[1]))
    else:
        lib.libgint_get_K(h, ptr(s.K[0]))
    return s.K


def work(case):
    """A lower bound: the records of the screened list, P and K once; G_m of
    one cell per primitive quartet, its blocks formed and contracted once, and
    the four K updates of every integral (none for the integral output)."""
    s = _system(case)
    st = s.record(sample=case["sample"])
    _, kind, _ = s.atoms()
    shells = {k: s.kind_basis(k)[1] for k in set(kind.tolist())}
    lmax = {k: max(l for l, _, _ in v) for k, v in shells.items()}
    nfun = {k: sum(nl * (2 * l + 1) for l, nl, _ in v) for k, v in shells.items()}
    quartets, counts = np.unique(kind[st.sets()].reshape(-1, 4), axis=0, return_counts=True)
    integrals = flops = 0.0
    for q, n in zip(quartets.tolist(), counts.tolist()):
        integrals += n * float(np.prod([nfun[k] for k in q]))
        L = sum(lmax[k] for k in q)
        cols = math.comb(lmax[q[0]] + lmax[q[1]] + 3, 3) * math.comb(lmax[q[2]] + lmax[q[3]] + 3, 3)
        flops += st.n_prm * (n / max(1, st.n_sets)) * (211.0 * (L + 1) + 2.0 * cols)
    out = 8.0 * integrals if case["path"] == "integrals" else 16.0 * s.P_size * case["spins"]
    updates = 0.0 if case["path"] == "integrals" else 8.0 * case["spins"] * integrals
    return {"bytes": out + 4.0 * st.n_prm + 16.0 * st.n_rows, "flops": flops + updates}


# ---------------------------------------------------------------------------
# The same in 64 bits by plain numpy: McMurchie-Davidson integrals of the
# unscreened molecule, for small clusters
# ---------------------------------------------------------------------------
_NODES, _WEIGHTS = np.polynomial.legendre.leggauss(64)
_NODES, _WEIGHTS = 0.5 * (_NODES + 1.0), 0.5 * _WEIGHTS


def _aux(L, rho, T, r_cut):
    """G_0 .. G_L of the operator 1/r (r_cut None) or theta(r_cut - r)/r: [L+1, *T.shape]"""
    b = np.minimum(1.0, 7.5 / np.sqrt(np.maximum(T, 1e-300)))
    v2 = _NODES ** 2
    e = np.exp(-(T * b * b)[..., None] * v2) * _WEIGHTS
    F = np.stack([b ** (2 * m + 1) * (e * v2 ** m).sum(-1) for m in range(L + 1)])
    if r_cut is None:
        return F
    # minus the part beyond the cut-off: 2 int_R^inf s e^(-s^2-T) i_0(2 s sqrt(T)) ds and its
    # derivatives by -T, (1/z d/dz) (i_k / z^k) = i_{k+1} / z^{k+1}
    R, t = r_cut * np.sqrt(rho), np.sqrt(T)
    near = R - t < 8.0
    R, t, T = R[near][:, None], t[near][:, None], T[near][:, None]
    s = R + 8.0 * _NODES
    z = 2.0 * s * t
    g = _scaled_bessel(L, z)
    w = 16.0 * _WEIGHTS * s * np.exp(-(s - t) ** 2)
    for m in range(L + 1):
        f = sum(math.comb(m, k) * (-2.0 * s * s) ** k * g[k] for k in range(m + 1))
        F[m][near] -= (w * f).sum(-1)
    return F


def _scaled_bessel(L, z):
    """e^-z i_k(z) / z^k, k = 0..L"""
    small = np.minimum(z, 6.0)
    out = []
    for k in range(L + 1):
        term = np.ones_like(z) / np.prod(np.arange(1.0, 2 * k + 2, 2))
        tot = term.copy()
        for j in range(1, 40):
            term = term * (0.5 * small * small) / (j * (2 * k + 2 * j + 1))
            tot += term
        out.append(tot * np.exp(-small))
    big = np.maximum(z, 6.0)
    q = np.exp(-2.0 * big)
    up = [(1.0 - q) / (2.0 * big), (1.0 + q - (1.0 - q) / big) / (2.0 * big)]
    for k in range(1, L):
        up.append(up[k - 1] - (2 * k + 1) / big * up[k])
    return [np.where(z < 6.0, out[k], up[k] / big ** k) for k in range(L + 1)]


def _components(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


_S3 = 1.0 / math.sqrt(3.0)
_SPHERICAL = {0: [[1.0]], 1: [[0, 1, 0], [0, 0, 1], [1, 0, 0]],
              2: [[0, 1, 0, 0, 0, 0], [0, 0, 0, 0, 1, 0], [-0.5 * _S3, 0, 0, -0.5 * _S3, 0, _S3],
                  [0, 0, 1, 0, 0, 0], [0.5, 0, 0, -0.5, 0, 0]]}


def _hermite_e(l, za, zb, A, B):
    """Hermite expansion along one axis of x_A^i x_B^j, i, j <= l: [i][j][t], each an array over primitive pairs"""
    p = za + zb
    P = (za * A + zb * B) / p
    zero = np.zeros_like(p)
    E = {(0, 0): [np.exp(-za * zb / p * (A - B) ** 2)]}
    for i in range(l + 1):
        for j in range(l + 1):
            if i + j == 0:
                continue
            low, x = (E[i - 1, j], P - A) if i else (E[i, j - 1], P - B)
            get = lambda t: low[t] if 0 <= t < len(low) else zero  # noqa: E731
            E[i, j] = [x * get(t) + get(t - 1) / (2 * p) + (t + 1) * get(t + 1) for t in range(i + j + 1)]
    return E


class _Exact:
    def __init__(self, s, r_cut):
        R, kind, self.first = s.atoms()
        self.r_cut, self.lmax, atoms = r_cut, 0, []
        for a in range(s.natom):
            Z, shells = s.kind_basis(int(kind[a]))
            rows = []
            for l, nl, K in shells:
                self.lmax = max(self.lmax, l)
                pair = np.pi ** 1.5 / 2.0 ** l / (Z[:, None] + Z[None, :]) ** (1.5 + l)
                Kn = K / np.sqrt(np.einsum("ni,nj,ij->n", K, K, pair))[:, None]
                rows += [(l, k, c) for k in Kn for c in _SPHERICAL[l]]
            atoms.append((R[a], Z, rows))
        self.atoms = atoms
        self.shells = [[(l, nl) for l, nl, _ in s.kind_basis(int(k))[1]] for k in kind]
        self.nfun = [len(r) for _, _, r in atoms]
        self.tuv = [c for n in range(2 * self.lmax + 1) for c in _components(n)]
        self.pairs = {}

    def pair(self, i, j):
        """Hermite coefficients of every function pair: [pairs of primitives, functions i x j, tuv], exponent sums and centres"""
        if (i, j) not in self.pairs:
            (A, za, fa), (B, zb, fb) = self.atoms[i], self.atoms[j]
            a, b = (x.ravel() for x in np.meshgrid(za, zb, indexing="ij"))
            E = [_hermite_e(self.lmax, a, b, A[k], B[k]) for k in range(3)]
            cart = {}
            for la in {f[0] for f in fa}:
                for lb in {f[0] for f in fb}:
                    M = np.zeros((a.size, len(_components(la)), len(_components(lb)), len(self.tuv)))
                    for x, ca in enumerate(_components(la)):
                        for y, cb in enumerate(_components(lb)):
                            e = [E[k][ca[k], cb[k]] for k in range(3)]
                            for n, t in enumerate(self.tuv):
                                if all(t[k] < len(e[k]) for k in range(3)):
                                    M[:, x, y, n] = e[0][t[0]] * e[1][t[1]] * e[2][t[2]]
                    cart[la, lb] = M
            H = np.zeros((a.size, len(fa), len(fb), len(self.tuv)))
            for x, (la, ka, ca) in enumerate(fa):
                for y, (lb, kb, cb) in enumerate(fb):
                    w = np.outer(ka, kb).ravel()
                    H[:, x, y] = w[:, None] * np.einsum("x,y,pxyn->pn", np.array(ca, float), np.array(cb, float), cart[la, lb])
            p = a + b
            self.pairs[i, j] = (p, (a[:, None] * A + b[:, None] * B) / p[:, None], H.reshape(a.size, -1, len(self.tuv)))
        return self.pairs[i, j]

    def integrals(self, i, j, k, l):
        """(ij|kl) of every function of four atoms"""
        (p, P, Hp), (q, Q, Hq) = self.pair(i, j), self.pair(k, l)
        L = 4 * self.lmax
        X = P[:, None, :] - Q[None, :, :]
        rho = p[:, None] * q[None, :] / (p[:, None] + q[None, :])
        G = _aux(L, rho, rho * (X ** 2).sum(-1), self.r_cut)
        R = {(m, (0, 0, 0)): (-2 * rho) ** m * G[m] for m in range(L + 1)}
        for N in range(1, L + 1):
            for c in _components(N):
                d = next(x for x in range(3) if c[x])
                c1 = tuple(v - (x == d) for x, v in enumerate(c))
                c2 = tuple(v - 2 * (x == d) for x, v in enumerate(c))
                for m in range(L - N + 1):
                    v = X[..., d] * R[m + 1, c1]
                    R[m, c] = v + (c[d] - 1) * R[m + 1, c2] if c[d] > 1 else v
        n = len(self.tuv)
        M = np.zeros((p.size, n, q.size, n))
        for x, t in enumerate(self.tuv):
            for y, u in enumerate(self.tuv):
                M[:, x, :, y] = (-1) ** sum(u) * R[0, tuple(a + b for a, b in zip(t, u))]
        M *= (2 * np.pi ** 2.5 / (p[:, None] * q[None, :] * np.sqrt(p[:, None] + q[None, :])))[:, None, :, None]
        left = Hp.transpose(1, 0, 2).reshape(Hp.shape[1], -1) @ M.reshape(p.size * n, -1)
        I = left @ Hq.transpose(1, 0, 2).reshape(Hq.shape[1], -1).T
        return I.reshape(self.nfun[i], self.nfun[j], self.nfun[k], self.nfun[l])


def exact(case, seed):
    # periodic lattice sums and clusters of many primitive quartets are beyond a few seconds of numpy
    if case["images"] or case["basis"] == 4 or case["centres"] or case["waters"] > 2:
        return None
    s = _system(case, seed)
    x = _Exact(s, s.rcut() if case["truncated"] else None)
    sets = s.record(sample=case["sample"]).sets().tolist()
    if case["path"] == "integrals":
        return np.concatenate([_transposed(x, q) for q in sets])
    P = _densities(case, s, seed)
    # blocks of atom pairs i <= j, column-major, one after the other
    na, at, off = s.natom, {}, 0
    for i in range(na):
        for j in range(i, na):
            at[i, j] = (off, x.nfun[i], x.nfun[j])
            off += x.nfun[i] * x.nfun[j]

    def block(v, a, b):
        o, r, c = at[min(a, b), max(a, b)]
        m = v[o:o + r * c].reshape(c, r).T
        return m if a <= b else m.T

    K = [np.zeros(s.P_size) for _ in P]
    for i, j, k, l in sets:
        I = x.integrals(i, j, k, l) * (2.0 / 2 ** ((i == j) + (k == l) + ((i, j) == (k, l))))
        for p, v in zip(P, K):
            block(v, j, l)[...] -= np.einsum("abcd,ac->bd", I, block(p, i, k))
            block(v, j, k)[...] -= np.einsum("abcd,ad->bc", I, block(p, i, l))
            block(v, i, l)[...] -= np.einsum("abcd,bc->ad", I, block(p, j, k))
            block(v, i, k)[...] -= np.einsum("abcd,bd->ac", I, block(p, j, l))
    return [torch.from_numpy(v) for v in K] if case["path"] == "noalloc" else K


def _transposed(x, q):
    """the classes of a set quartet, each [ila, isa, ilb, isb, ilc, isc, ild, isd]"""
    I, out, start = x.integrals(*q), [], []
    for a in q:
        n = np.cumsum([0] + [nl * (2 * l + 1) for l, nl in x.shells[a]])
        start.append([slice(u, v) for u, v in zip(n[:-1], n[1:])])
    for a in start[0]:
        for b in start[1]:
            for c in start[2]:
                out += [I[a, b, c, d].ravel() for d in start[3]]
    return np.concatenate(out)
