"""Performance cases of the exact-diagonalisation engine.

What a program that diagonalises a Hubbard cluster does with this package: it applies H to
device vectors (its own Lanczos, time evolution or a check), asks for the ground state of a
sector with its observables, and runs the continued-fraction chains of the Green's functions
and of the spin susceptibility from a state it has.  The sizes are those of the package's
workloads (lattice.CONFIGS), of its tests and of bench.py: the 8-site ring, the 3x4 and 4x4
tori, the open 3x6 cluster with disorder.
"""
import math

import numpy as np
import torch

from ed_lattice_amd import EDLattice, lattice

DEV = "cuda"


def listed():
    return [
        # H v on device vectors, the operator a program with its own Krylov loop calls:
        # the smallest sector (launch latency), the 8-ring at half filling
        dict(name="hxv_ring8_f64", kind="hxv", lx=8, ly=1, pbc=True, disorder=False, u=4.0, nup=4, ndw=4, prec="fp64"),
        # the 3x4 cluster at half filling, an ordinary size
        dict(name="hxv_rect3x4_f64", kind="hxv", lx=3, ly=4, pbc=True, disorder=False, u=6.0, nup=6, ndw=6,
             prec="fp64"),
        # an odd, unbalanced sector of a disordered cluster, single precision
        dict(name="hxv_rect3x5_f32", kind="hxv", lx=3, ly=5, pbc=True, disorder=True, u=4.0, nup=7, ndw=4,
             prec="fp32"),
        # the headline sector, 4x4 at half filling (1.66e8 states), in both precisions
        dict(name="hxv_sq4x4_f32", kind="hxv", lx=4, ly=4, pbc=True, disorder=False, u=8.0, nup=8, ndw=8, prec="fp32"),
        dict(name="hxv_sq4x4_f64", kind="hxv", lx=4, ly=4, pbc=True, disorder=False, u=8.0, nup=8, ndw=8, prec="fp64"),
        # the largest: the disordered open 3x6 cluster (2.36e9 states)
        dict(name="hxv_obc3x6_f32", kind="hxv", lx=3, ly=6, pbc=False, disorder=True, u=4.0, nup=9, ndw=9,
             prec="fp32"),
        # ground state and observables of a small cluster (a parameter scan runs thousands)
        dict(name="gs_ring8_f64", kind="gs", lx=8, ly=1, pbc=True, disorder=False, u=4.0, nup=4, ndw=4, prec="fp64",
             niter=120),
        # ... of the 3x4 cluster
        dict(name="gs_rect3x4_f64", kind="gs", lx=3, ly=4, pbc=True, disorder=False, u=6.0, nup=6, ndw=6, prec="fp64",
             niter=120),
        # ... of the 3x5 cluster (4.1e7 states) with mixed precision, the engine's solve for large sectors
        dict(name="gs_rect3x5_mixed", kind="gs", lx=3, ly=5, pbc=True, disorder=False, u=8.0, nup=8, ndw=7,
             prec="mixed", niter=60),
        # local Green's functions of every site of the ring: particle and hole chains
        dict(name="gf_ring8_f64", kind="gf", lx=8, ly=1, pbc=True, disorder=False, u=4.0, nup=4, ndw=4, prec="fp64",
             sites=8, offdiag=False, nlanc=40),
        # all i <= j pairs of the 3x4 cluster, 156 chains in the N+1 and N-1 sectors
        dict(name="gf_rect3x4_f64", kind="gf", lx=3, ly=4, pbc=True, disorder=False, u=6.0, nup=6, ndw=6, prec="fp64",
             sites=12, offdiag=True, nlanc=40),
        # spin susceptibility of the 3x4 cluster in single precision: one chain per site
        dict(name="chi_rect3x4_f32", kind="chi", lx=3, ly=4, pbc=True, disorder=True, u=6.0, nup=6, ndw=6,
             prec="fp32", sites=12, offdiag=False, nlanc=30),
    ]


def draw(rng):
    kind = rng.choice(["hxv", "hxv", "hxv", "gs", "gf", "chi"])
    big = kind == "hxv"
    # clusters from 6 sites on; the operator up to 4x4, the Lanczos solves up to 12 sites
    shapes = [(6, 1), (7, 1), (8, 1), (9, 1), (3, 3), (10, 1), (11, 1), (12, 1), (3, 4)]
    if big:
        shapes += [(13, 1), (14, 1), (3, 5), (15, 1), (4, 4), (16, 1)]
    # sizes spread over the logarithm: a target dimension first, then the nearest of some sectors
    target = math.exp(rng.uniform(math.log(400.0), math.log(1.6e8 if big else 8.5e5)))
    best = None
    for _ in range(60):
        lx, ly = rng.choice(shapes)
        ns = lx * ly
        nup, ndw = rng.randint(2, ns - 2), rng.randint(2, ns - 2)
        d = math.comb(ns, nup) * math.comb(ns, ndw)
        if 400 <= d <= (1.66e8 if big else 8.6e5):
            off = abs(math.log(d / target))
            if best is None or off < best[0]:
                best = (off, lx, ly, nup, ndw)
    _, lx, ly, nup, ndw = best
    c = dict(kind=kind, lx=lx, ly=ly, pbc=rng.random() < 0.7, disorder=rng.random() < 0.4,
             u=round(rng.uniform(2.0, 10.0), 2), nup=nup, ndw=ndw)
    ns = lx * ly
    if kind == "hxv":
        c["prec"] = rng.choice(["fp32", "fp64"])
    elif kind == "gs":
        c["prec"] = rng.choice(["fp64", "fp64", "mixed"])
        c["niter"] = rng.randint(60, 160)
    elif kind == "gf":
        c["prec"] = "fp64"
        c["sites"] = rng.randint(1, ns)
        c["offdiag"] = rng.random() < 0.5
        c["nlanc"] = rng.randint(20, 40)
    else:
        c["prec"] = rng.choice(["fp32", "fp64"])
        c["sites"] = rng.randint(1, ns)
        c["offdiag"] = False
        c["nlanc"] = rng.randint(15, 30)
    return c


# ------------------------------------------------------------------ the model of a case
def _hij(case, seed=None):
    """Hopping matrix; the solves (seed given) also draw the onsite energies of their sample."""
    lx, ly = case["lx"], case["ly"]
    ns = lx * ly
    if case["disorder"]:
        H = lattice.disordered_rect(lx, ly, pbc=case["pbc"])
    elif ly == 1:
        H = lattice.hij_from_bonds(ns, lattice.bonds_rect(lx, 1, case["pbc"], False))
    else:
        H = lattice.square(lx, ly, pbc=case["pbc"])
    if seed is not None:
        eps = np.random.default_rng([11, seed]).uniform(-0.25, 0.25, ns)
        H[:, np.arange(ns), np.arange(ns)] += eps
    return H


def _seeds(case):
    n = case["sites"]
    pairs = [(i, 0) for i in range(1, n + 1)]
    if case["offdiag"]:
        pairs += [(i, j) for i in range(1, n + 1) for j in range(i + 1, n + 1)]
    if case["kind"] == "chi":
        return [("sz", 1, i, j) for i, j in pairs]
    return [(op, 1, i, j) for i, j in pairs for op in ("cdg", "c")]


class State:
    """What a program holds: the engine's handle, its sector and its vectors."""

    def __init__(self, case):
        self.case = case
        self.ed = EDLattice(0)

    def __del__(self):
        self.ed.close()


def prepare(case, seed):
    s = State(case)
    if case["kind"] == "hxv":
        s.ed.set_hamiltonian(_hij(case), [case["u"]])
        s.isec = s.ed.sector_index(case["nup"], case["ndw"])
        dim, _, _ = s.ed.build_sector(s.isec)
        s.v = _vector(case, seed, dim)
        s.hv = torch.empty_like(s.v)
    else:
        H = _hij(case, seed)
        s.ed.set_hamiltonian(H, [case["u"]])
        s.isec = s.ed.sector_index(case["nup"], case["ndw"])
        dim, _, _ = s.ed.build_sector(s.isec)
        s.seed = seed
        if case["kind"] != "gs":
            # the state of an earlier run, installed from its file
            e, x = _given_state(case, H)
            s.ed.set_state(s.isec, e, x.cpu().numpy().ravel())
            s.seeds = _seeds(case)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s.case
    if case["kind"] == "hxv":
        s.ed.hxv_device(s.isec, case["prec"], s.v.data_ptr(), s.hv.data_ptr())
        return s.hv
    if case["kind"] == "gs":
        r = s.ed.lanczos_eigh(s.isec, case["prec"], niter=case["niter"], seed=s.seed)
        o, c = s.ed.observables(), s.ed.correlations()
        # a mixed-precision state is good to the square root of its energy's tolerance
        t = np.float32 if case["prec"] == "mixed" else np.float64
        return {"e0": r["e0"], "dens_up": o["dens_up"].astype(t), "dens_dw": o["dens_dw"].astype(t),
                "docc": o["docc"].astype(t), "sz2": c["sz2"].astype(t), "n2": c["n2"].astype(t)}
    r = s.ed.tridiag_batched(s.seeds, case["nlanc"], case["prec"])
    t = np.float32 if case["prec"] == "fp32" else np.float64  # coefficients of single-precision chains
    return {"alpha": r["alpha"].astype(t), "beta": r["beta"].astype(t), "norm2": r["norm2"],
            "nsteps": r["nsteps"], "isector": r["isector"]}


def _vector(case, seed, dim):
    g = torch.Generator(device=DEV).manual_seed(seed)
    t = torch.float32 if case["prec"] == "fp32" else torch.float64
    v = torch.randn(dim, generator=g, device=DEV, dtype=t)
    return v.div_(math.sqrt(dim))


def work(case):
    ns = case["lx"] * case["ly"]
    H = _hij(case)[0]
    bonds = int(np.count_nonzero(np.triu(H, 1)))

    def sector(nup, ndw):
        d = math.comb(ns, nup) * math.comb(ns, ndw)
        # a bond moves an electron where exactly one of its two sites is occupied
        hops = sum(bonds * 2.0 * n * (ns - n) / (ns * (ns - 1)) for n in (nup, ndw))
        return d, hops

    d, hops = sector(case["nup"], case["ndw"])
    if case["kind"] == "hxv":
        size = 4 if case["prec"] == "fp32" else 8
        return {"bytes": 2.0 * d * size, "flops": d * (2.0 * hops + 2.0)}
    if case["kind"] == "gs":
        # a step reads q_k and q_k-1 and writes q_k+1; the state is a sum over the stored q_k
        size = 8 if case["prec"] == "fp64" else 4
        m = min(case["niter"], d)
        return {"bytes": 4.0 * m * d * size, "flops": m * d * (2.0 * hops + 10.0)}
    size = 4 if case["prec"] == "fp32" else 8
    total = {"bytes": 0.0, "flops": 0.0}
    for op, _, _, _ in _seeds(case):
        dj, hj = sector(case["nup"] + {"c": -1, "cdg": 1, "sz": 0}[op], case["ndw"])
        m = min(case["nlanc"], dj)
        total["bytes"] += 3.0 * m * dj * size
        total["flops"] += m * dj * (2.0 * hj + 8.0)
    return total


# ------------------------------------------- the same quantities in plain 64-bit torch
def _strings(ns, n):
    s = np.arange(1 << ns, dtype=np.int64)
    pop = np.zeros(1 << ns, dtype=np.int8)
    for k in range(ns):
        pop += ((s >> k) & 1).astype(np.int8)
    return s[pop == n], pop


class _Plain:
    """H of one sector on vectors [.., DimDw, DimUp] (up index fastest), 64 bits."""

    def __init__(self, H, u, nup, ndw):
        ns = H.shape[1]
        self.shape = (math.comb(ns, ndw), math.comb(ns, nup))
        self.hops, diag = [], []
        strs = []
        for n in (nup, ndw):
            s, pop = _strings(ns, n)
            strs.append(s)
            hops = []
            for p in range(ns):
                for q in range(p + 1, ns):
                    h = H[0, p, q]
                    if h == 0.0:
                        continue
                    one = ((s >> p) ^ (s >> q)) & 1
                    src = np.where(one == 1, s ^ ((1 << p) | (1 << q)), s)
                    between = ((1 << q) - 1) & ~((1 << (p + 1)) - 1)
                    sign = 1.0 - 2.0 * (pop[s & between] & 1)
                    at = torch.from_numpy(np.searchsorted(s, src)).to(DEV)
                    hops.append((at, torch.from_numpy(h * sign * one).to(DEV)))
            self.hops.append(hops)
            d = np.zeros(len(s))
            for p in range(ns):
                d += ((s >> p) & 1) * (H[0, p, p] - 0.5 * u)
            diag.append(torch.from_numpy(d).to(DEV))
        self.diag = diag
        self.strs = [torch.from_numpy(s).to(DEV) for s in strs]
        self.u, self.ns = u, ns

    def site(self, spin, p):
        return ((self.strs[spin] >> p) & 1).double()

    def docc(self, v):
        """sum_p n_up,p n_dw,p times v."""
        w = torch.zeros_like(v)
        for p in range(self.ns):
            w += v * (self.site(1, p)[:, None] * self.site(0, p)[None, :])
        return w

    def __call__(self, v):
        w = self.diag[0][None, :] * v
        w += self.diag[1][:, None] * v
        for p in range(self.ns):
            w.addcmul_(v, self.site(1, p)[:, None] * (self.u * self.site(0, p))[None, :])
        for at, c in self.hops[0]:
            w.addcmul_(v.index_select(-1, at), c.expand_as(v))
        for at, c in self.hops[1]:
            w.addcmul_(v.index_select(-2, at), c[:, None].expand_as(v))
        return w


def _start(n, seed):
    """U[-1,1) from the SplitMix64 stream of `seed`, one output per element (the documented start vector)."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return torch.from_numpy(2.0 * ((z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53) - 1.0).to(DEV)


def _lowest(op, v, m):
    """Lowest Ritz pair of an m-step Lanczos run with full reorthogonalisation."""
    n = v.numel()
    m = min(m, n)
    Q = torch.empty(m, n, device=DEV, dtype=torch.float64)
    a, b = [], []
    q = v.reshape(-1) / v.norm()
    for k in range(m):
        Q[k] = q
        w = op(q.view(op.shape)).reshape(-1)
        a.append(float(w @ q))
        for _ in range(2):
            w -= Q[:k + 1].T @ (Q[:k + 1] @ w)
        nb = float(w.norm())
        if nb < 1e-12:
            break
        b.append(nb)
        q = w / nb
    k = len(a)
    e, z = np.linalg.eigh(np.diag(a) + np.diag(b[:k - 1], 1) + np.diag(b[:k - 1], -1))
    x = torch.from_numpy(z[:, 0].copy()).to(DEV) @ Q[:k]
    return float(e[0]), (x / x.norm()).view(op.shape)


def _given_state(case, H):
    op = _Plain(H, case["u"], case["nup"], case["ndw"])
    n = op.shape[0] * op.shape[1]
    return _lowest(op, _start(n, 7), 50)


def _apply(op_name, x, src, dst, site):
    """c+, c (spin up) or S^z on `site` (1-based) of x, in the target sector."""
    p = site - 1
    if op_name == "sz":
        return 0.5 * x * (src.site(0, p)[None, :] - src.site(1, p)[:, None])
    # the source string of each target string, its sign from the electrons below the site
    t = dst.strs[0]
    occupied = ((t >> p) & 1) == (1 if op_name == "cdg" else 0)
    low = t & ((1 << p) - 1)
    par = torch.zeros_like(t)
    for k in range(p):
        par ^= (low >> k) & 1
    at = torch.searchsorted(src.strs[0], torch.where(occupied, t ^ (1 << p), src.strs[0][0]))
    return x.index_select(-1, at) * ((1.0 - 2.0 * par) * occupied)[None, :]


def exact(case, seed):
    if case["kind"] == "hxv":
        op = _Plain(_hij(case), case["u"], case["nup"], case["ndw"])
        v = _vector(case, seed, op.shape[0] * op.shape[1]).double()
        return op(v.view(op.shape)).view(-1)
    H = _hij(case, seed)
    op = _Plain(H, case["u"], case["nup"], case["ndw"])
    n = op.shape[0] * op.shape[1]
    if case["kind"] == "gs":
        if n > 2_000_000:
            return None  # hundreds of stored vectors of 0.3 GB
        mixed = case["prec"] == "mixed"
        e, x = _lowest(op, _start(n, seed), 250 if mixed else case["niter"])
        p = x * x
        pu, pd = p.sum(0), p.sum(1)
        ns = case["lx"] * case["ly"]
        up = torch.stack([op.site(0, k) for k in range(ns)])
        dw = torch.stack([op.site(1, k) for k in range(ns)])
        uu, dd, ud = (up * pu) @ up.T, (dw * pd) @ dw.T, up @ p.T @ dw.T
        return {"e0": e, "dens_up": (up @ pu).cpu().numpy(), "dens_dw": (dw @ pd).cpu().numpy(),
                "docc": ud.diagonal().cpu().numpy(),
                "sz2": (0.25 * (uu + dd - ud - ud.T)).cpu().numpy(), "n2": (uu + dd + ud + ud.T).cpu().numpy()}
    _, x = _given_state(case, H)
    seeds, m = _seeds(case), case["nlanc"]
    alpha, beta, norm2 = np.zeros((len(seeds), m)), np.zeros((len(seeds), m)), np.zeros(len(seeds))
    for name in ("cdg", "c", "sz"):
        which = [k for k, sd in enumerate(seeds) if sd[0] == name]
        if not which:
            continue
        dst = _Plain(H, case["u"], case["nup"] + {"c": -1, "cdg": 1, "sz": 0}[name], case["ndw"])
        at_once = max(1, int(4e8 // (dst.shape[0] * dst.shape[1])))
        for b0 in range(0, len(which), at_once):
            part = which[b0:b0 + at_once]
            q = []
            for k in part:
                _, _, i, j = seeds[k]
                y = _apply(name, x, op, dst, i)
                q.append(y + _apply(name, x, op, dst, j) if j else y)
            q = torch.stack(q)
            n2 = (q * q).sum((1, 2))
            norm2[part] = n2.cpu().numpy()
            q /= n2.sqrt()[:, None, None]
            old, bk = torch.zeros_like(q), torch.zeros_like(n2)
            for k in range(min(m, dst.shape[0] * dst.shape[1])):
                w = dst(q) - bk[:, None, None] * old
                ak = (w * q).sum((1, 2))
                w -= ak[:, None, None] * q
                alpha[part, k] = ak.cpu().numpy()
                bk = (w * w).sum((1, 2)).sqrt()
                if k + 1 < m:
                    beta[part, k + 1] = bk.cpu().numpy()
                old, q = q, w / bk[:, None, None]
    return {"alpha": alpha, "beta": beta, "norm2": norm2, "nsteps": None, "isector": None}
