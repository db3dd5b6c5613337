"""Workloads of the exact-diagonalisation path, as a user's program runs them.

A case is one call (or a short fixed sequence of calls) of the public entry points in
diagham_amd.capi on vectors that live on the GPU: the product H.v of the sphere, the spin chain and
the momentum lattice, for one vector and for a block, one sector and every sector at once; the
adjoint of the sphere product (dE/dV of every pseudopotential channel); the full
reorthogonalisation of a Lanczos vector; and a whole Lanczos run to the lowest eigenvalues.

listed() names the cases, draw() takes others from the same ranges, prepare() builds the operator
and the input vectors, run() makes one pass, work() counts what a pass cannot do without, and
exact() gives the same outputs from plain torch in 64 bits.
"""
import math
from fractions import Fraction

import numpy as np
import torch

from diagham_amd import capi

_arch = None


def arch():
    """The device context of the program; its work goes to torch's current stream."""
    global _arch
    if _arch is None:
        _arch = capi.Arch(0)
    _arch.check(capi.gpu().dh_set_stream(_arch.ctx, torch.cuda.current_stream().cuda_stream), "dh_set_stream")
    return _arch


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one Lz sector of a small system: the bulk of a sector-after-sector run is calls like this,
        # and what counts is the latency of one product
        dict(name="sphere_n6", kind="sphere", n=6, lz_max=15, total_lz=0, k=1),
        # the sphere at nu = 1/3, Lz = 0, at the sizes of routine and of large studies: one product
        dict(name="sphere_n10", kind="sphere", n=10, lz_max=27, total_lz=0, k=1),
        dict(name="sphere_n12", kind="sphere", n=12, lz_max=33, total_lz=0, k=1),
        # the same operator on a block of eight vectors (block Lanczos, degenerate levels)
        dict(name="sphere_n10_k8", kind="sphere", n=10, lz_max=27, total_lz=0, k=8),
        # every Lz >= 0 sector of N = 10 in one product: a step of the batched sector solve
        dict(name="sectors_n10", kind="sectors", n=10, lz_max=27, k=1),
        # every momentum sector of the Chern band on 6 x 5 sites, complex vectors
        dict(name="lattice_6x5_n10", kind="lattice", n=10, nx=6, ny=5, k=1),
        # a Heisenberg chain at a size for dynamics and scans, and at the largest that is run
        dict(name="spin_l20", kind="spin", length=20, sz=0, k=1, periodic=True, uniform=True),
        dict(name="spin_l28", kind="spin", length=28, sz=0, k=1, periodic=True, uniform=True),
        # an open chain with bond-dependent couplings on a block of four vectors
        dict(name="spin_l24_open_k4", kind="spin", length=24, sz=0, k=4, periodic=False, uniform=False),
        # backward of the ground-state energy: dE/dV of every channel, and H psi
        dict(name="adjoint_n10", kind="adjoint", n=10, lz_max=27, total_lz=0),
        # one full reorthogonalisation deep in a Lanczos run (two passes over the Krylov basis)
        dict(name="reorth_100", kind="reorth", rows=2704156, vectors=100, k=1),
        # a whole run: the ten lowest eigenvalues of N = 8 at 2S = 21
        dict(name="lanczos_n8", kind="lanczos", n=8, lz_max=21, total_lz=0, nev=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kinds = ["sphere"] * 4 + ["sectors"] * 2 + ["lattice"] * 2 + ["spin"] * 3 + ["adjoint", "reorth", "lanczos"]
    while True:
        kind = rng.choice(kinds)
        if kind in ("sphere", "adjoint", "lanczos"):
            top = {"sphere": 12, "adjoint": 10, "lanczos": 8}[kind]
            n = rng.randint(5, top)
            lz_max = rng.randint(2 * n - 1, min(3 * n + 2, 33))
            total_lz = (n * lz_max) % 2 + 2 * rng.randint(0, n)
            c = dict(kind=kind, n=n, lz_max=lz_max, total_lz=total_lz)
            rows = _sphere_rows(n, lz_max, [total_lz])
            if kind == "sphere":
                c["k"] = rng.choice([1, 1, 4, 8])
                if rows * c["k"] > 7800000:
                    continue
            if rows < 200 or (kind == "lanczos" and rows > 12000) or (kind == "adjoint" and rows > 1500000):
                continue
            if kind == "lanczos":
                c["nev"] = rng.randint(2, 10)
            return c
        if kind == "sectors":
            n = rng.randint(5, 10)
            c = dict(kind=kind, n=n, lz_max=rng.randint(2 * n, 3 * n), k=rng.choice([1, 1, 4, 8]))
            if _sphere_rows(n, c["lz_max"], capi.sphere_sectors(n, c["lz_max"])) * c["k"] > 16000000:
                continue
            return c
        if kind == "lattice":
            nx, ny = rng.randint(3, 6), rng.randint(3, 6)
            c = dict(kind=kind, n=rng.randint(4, 10), nx=nx, ny=ny, k=rng.choice([1, 1, 2, 4]))
            if c["n"] > nx * ny - 4 or math.comb(nx * ny, c["n"]) * c["k"] > 31000000:
                continue
            return c
        if kind == "spin":
            length = rng.randint(10, 28)
            c = dict(kind=kind, length=length, sz=length % 2 + 2 * rng.randint(0, 3), k=rng.choice([1, 1, 2, 4, 8]),
                     periodic=rng.random() < 0.7, uniform=rng.random() < 0.6)
            if math.comb(length, (length + c["sz"]) // 2) * c["k"] > 40200000:
                continue
            return c
        k = rng.choice([1, 1, 1, 4, 8])
        rows = _log_int(rng, 5000, 4000000)
        vectors = rng.randint(4, 160) // k + 1
        if rows * vectors * k > 280000000:
            continue
        return dict(kind="reorth", rows=rows, vectors=vectors, k=k)


# ------------------------------------------------------------------------------------ sizes
def _sphere_counts(n, n_orb):
    """P[m][s]: m-subsets of the orbitals 0..n_orb-1 with index sum s, m <= n"""
    size = n * n_orb + 1
    p = np.zeros((n + 1, size))
    p[0, 0] = 1
    for a in range(n_orb):
        for m in range(n, 0, -1):
            p[m, a:] += p[m - 1, :size - a]
    return p


def _sphere_rows(n, lz_max, sectors):
    p = _sphere_counts(n, lz_max + 1)
    return int(sum(p[n, (lz + n * lz_max) // 2] for lz in sectors))


def _sphere_elements(n, lz_max, sectors):
    """matrix elements (row, annihilated pair, created pair) of the sectors: (n-2)-subsets that
    avoid both pairs, counted by removing their orbitals from the generating function"""
    n_orb, m = lz_max + 1, n - 2
    p = _sphere_counts(m, n_orb)
    size = p.shape[1]
    sums = [(lz + n * lz_max) // 2 for lz in sectors]

    def without(q, a):
        r = q.copy()
        for j in range(1, m + 1):
            r[j, a:] -= r[j - 1, :size - a]
        return r

    total = 0.0
    for s in range(1, 2 * lz_max):
        pairs = [(b, s - b) for b in range(s // 2 + 1, min(s, lz_max) + 1)]
        at = [t - s for t in sums if 0 <= t - s < size]
        for i, (a, b) in enumerate(pairs):
            q = without(without(p, a), b)
            total += q[m, at].sum()
            for c, d in pairs[i + 1:]:
                total += 2 * without(without(q, c), d)[m, at].sum()
    return total


def _lattice_elements(n, nx, ny):
    """matrix elements of all momentum sectors together: C(n-2 of the orbitals outside both pairs)"""
    orb = nx * ny
    sizes = np.zeros(orb)
    for a in range(orb):
        for b in range(a + 1, orb):
            sizes[((a // ny + b // ny) % nx) * ny + (a % ny + b % ny) % ny] += 1
    diag, off = sizes.sum(), (sizes * (sizes - 1)).sum()
    return diag * math.comb(orb - 2, n - 2) + off * math.comb(orb - 4, n - 2)


def work(case):
    c = case
    kind, k = c["kind"], c.get("k", 1)
    if kind in ("sphere", "adjoint", "sectors"):
        sectors = capi.sphere_sectors(c["n"], c["lz_max"]) if kind == "sectors" else [c["total_lz"]]
        rows = _sphere_rows(c["n"], c["lz_max"], sectors)
        elements = _sphere_elements(c["n"], c["lz_max"], sectors)
        return {"bytes": 16.0 * rows * k, "flops": 2.0 * float(elements) * k}
    if kind == "lattice":
        rows = math.comb(c["nx"] * c["ny"], c["n"])
        return {"bytes": 32.0 * rows * k, "flops": 8.0 * _lattice_elements(c["n"], c["nx"], c["ny"]) * k}
    if kind == "spin":
        up = (c["length"] + c["sz"]) // 2
        bonds = c["length"] - (0 if c["periodic"] else 1)
        rows = math.comb(c["length"], up)
        flips = 2 * bonds * math.comb(c["length"] - 2, up - 1)
        return {"bytes": 16.0 * rows * k, "flops": 2.0 * (rows + flips) * k}
    if kind == "reorth":  # the basis is needed by the dot products and again by the update
        block = 8.0 * c["rows"] * k
        return {"bytes": 2 * c["vectors"] * block + 2 * block, "flops": 4.0 * c["rows"] * c["vectors"] * k * k}
    rows = _sphere_rows(c["n"], c["lz_max"], [c["total_lz"]])
    steps = min(rows, 20 * c["nev"])  # a Krylov space of that size at least, each vector read by each later step
    return {"bytes": 8.0 * rows * steps * steps / 2 + 16.0 * rows * steps,
            "flops": 2.0 * _sphere_elements(c["n"], c["lz_max"], [c["total_lz"]]) * steps + 2.0 * rows * steps * steps}


# ------------------------------------------------------------------------------------ inputs
def _pseudo(case, seed):
    """Coulomb pseudopotentials of the lowest Landau level with a few per cent of variation, as in a
    scan over model interactions"""
    r = np.random.RandomState(seed % (1 << 31))
    v = capi.coulomb_pseudopotentials(case["lz_max"])
    return v * (1.0 + 0.05 * r.uniform(-1, 1, v.size))


def _couplings(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    length = case["length"]
    if case["uniform"]:
        return np.full(length, 1.0), np.full(length, r.uniform(0.5, 1.5))
    return r.uniform(0.5, 1.5, length), r.uniform(0.5, 1.5, length)


def _model(seed):
    r = np.random.RandomState(seed % (1 << 31))
    return dict(t1=1.0, t2=0.5, tpp=-0.5, mus=r.uniform(0.0, 0.1), u_potential=1.0, v_potential=0.0, flat_band=True)


def _vectors(rows, width, seed):
    """`width` normalised random vectors, one row after the other"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, width, dtype=torch.float64, device="cuda", generator=g)
    return x / math.sqrt(rows)


def _lattice_sectors(case):
    kx = [i // case["ny"] for i in range(case["nx"] * case["ny"])]
    ky = [i % case["ny"] for i in range(case["nx"] * case["ny"])]
    # a sector without states is not asked for
    keep = [i for i in range(len(kx))
            if capi.gpu().dh_momentum_sector_dimension(case["n"], case["nx"], case["ny"], kx[i], ky[i]) > 0]
    return [kx[i] for i in keep], [ky[i] for i in keep]


def prepare(case, seed):
    a, c, k = arch(), case, case.get("k", 1)
    kind = c["kind"]
    s = {"case": case, "arch": a}
    if kind in ("sphere", "adjoint", "lanczos"):
        s["op"] = capi.Problem.sphere(a, c["n"], c["total_lz"], c["lz_max"], _pseudo(c, seed))
        if kind == "lanczos":
            s["seed"] = seed
            return s
        s["x"] = _vectors(s["op"].dim, k, seed)
    elif kind == "sectors":
        s["op"] = capi.SphereSectorSet(a, c["n"], c["lz_max"], capi.sphere_sectors(c["n"], c["lz_max"]), _pseudo(c, seed))
        s["x"] = _vectors(s["op"].total, k, seed)
    elif kind == "lattice":
        s["op"] = capi.MomentumSectorSet(a, c["n"], c["nx"], c["ny"], *_lattice_sectors(c), **_model(seed))
        s["x"] = _vectors(s["op"].total, 2 * k, seed)
    elif kind == "spin":
        j, jz = _couplings(c, seed)
        s["op"] = capi.Problem.spin_chain(a, c["length"], c["sz"], j, jz, c["periodic"])
        s["x"] = _vectors(s["op"].dim, k, seed)
    else:
        # a Krylov basis as the solver stores it: block after block, [row][k] in each
        g = torch.Generator(device="cuda").manual_seed(seed)
        s["v"] = torch.empty(c["vectors"], c["rows"], k, dtype=torch.float64, device="cuda")
        s["v"].normal_(0.0, 1.0 / math.sqrt(c["rows"]), generator=g)
        s["x"] = _vectors(c["rows"], k, seed + 1)
    s["y"] = torch.empty_like(s["x"])
    return s


def run(state):
    s, c = state, state["case"]
    kind, k = c["kind"], c.get("k", 1)
    if kind in ("sphere", "sectors", "lattice", "spin"):
        s["op"].hv_device(s["x"].data_ptr(), s["y"].data_ptr(), k)
        return s["y"]
    if kind == "adjoint":
        return {"g": s["op"].adjoint_device(s["x"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr()), "hx": s["y"]}
    if kind == "lanczos":
        return s["op"].lanczos(c["nev"], block_size=1, seed=s["seed"])["eigenvalues"]
    a, lib = s["arch"], capi.gpu()
    h = np.empty(c["vectors"] * k * k)
    a.check(lib.dh_copy(a.ctx, s["y"].data_ptr(), s["x"].data_ptr(), c["rows"] * k), "dh_copy")
    a.check(lib.dh_block_dots(a.ctx, s["v"].data_ptr(), c["vectors"], s["y"].data_ptr(), c["rows"], k, capi.dptr(h)),
            "dh_block_dots")
    m = -h
    a.check(lib.dh_block_axpy(a.ctx, s["v"].data_ptr(), c["vectors"], s["y"].data_ptr(), c["rows"], k, capi.dptr(m)),
            "dh_block_axpy")
    return {"h": h, "w": s["y"]}


# ------------------------------------------------------------------------------------ 64-bit values
def _clebsch(tj, tm1, tm2, tJ):
    """<j m1 j m2 | J M> for integers twice their values, from Racah's formula in rational numbers"""
    f = math.factorial
    M2 = tm1 + tm2
    if abs(M2) > tJ:
        return 0.0
    a, b, cc = (2 * tj - tJ) // 2, tJ // 2, tJ // 2
    p1, q1, p2, q2 = (tj + tm1) // 2, (tj - tm1) // 2, (tj + tm2) // 2, (tj - tm2) // 2
    P, Q = (tJ + M2) // 2, (tJ - M2) // 2
    total = Fraction(0)
    for z in range(0, a + 1):
        d = (a - z, q1 - z, p2 - z, (tJ - tj + tm1) // 2 + z, (tJ - tj - tm2) // 2 + z)
        if min(d) < 0:
            continue
        den = f(z)
        for v in d:
            den *= f(v)
        total += Fraction((-1) ** z, den)
    square = Fraction((tJ + 1) * f(a) * f(b) * f(cc), f((2 * tj + tJ) // 2 + 1)) * f(p1) * f(q1) * f(p2) * f(q2) * f(P) * f(Q)
    square *= total * total
    return math.copysign(math.sqrt(square.numerator / square.denominator), total) if total else 0.0


def _sphere_pairs(case, seed):
    """per pair sum: the pairs (m1 > m2) and the channel amplitudes u[pair, L] of the odd relative
    momenta; the factor of two pairs is -4 sum_L V_L u[p, L] u[q, L]"""
    lz = case["lz_max"]
    v = _pseudo(case, seed)
    rel = [m for m in range(lz + 1) if m % 2 == 1]
    out = []
    for s in range(1, 2 * lz):
        pairs = [(b, s - b) for b in range(s // 2 + 1, min(s, lz) + 1)]
        u = np.array([[_clebsch(lz, 2 * a - lz, 2 * b - lz, 2 * (lz - m)) for m in rel] for a, b in pairs])
        out.append((pairs, torch.tensor(u, dtype=torch.float64, device="cuda")))
    return out, torch.tensor(v[rel], dtype=torch.float64, device="cuda"), rel


def _popc(x):
    x = x - ((x >> 1) & 0x5555555555555555)
    x = (x & 0x3333333333333333) + ((x >> 2) & 0x3333333333333333)
    x = (x + (x >> 4)) & 0x0F0F0F0F0F0F0F0F
    return (x + (x >> 8) + (x >> 16) + (x >> 24) + (x >> 32) + (x >> 40) + (x >> 48) + (x >> 56)) & 0xFF


def _subsets(n, n_orb, keep=None):
    """all n-subsets of n_orb orbitals as words, ascending; keep(sum so far, orbitals left, n left)
    drops branches without a member of the wanted sector"""
    words = {0: torch.zeros(1, dtype=torch.int64, device="cuda")}
    sums = {0: torch.zeros(1, dtype=torch.int64, device="cuda")}
    for a in range(n_orb - 1, -1, -1):  # highest orbital first
        for m in range(min(n, n_orb - a), 0, -1):
            if m - 1 in words:
                w, s = words[m - 1] | (1 << a), sums[m - 1] + a
                if m in words:
                    w, s = torch.cat([words[m], w]), torch.cat([sums[m], s])
                words[m], sums[m] = w, s
        for m in list(words):
            if n - m > a:  # too few orbitals left to complete
                del words[m], sums[m]
            elif keep is not None:
                ok = keep(sums[m], a, n - m)
                words[m], sums[m] = words[m][ok], sums[m][ok]
    return torch.sort(words[n])[0]


def _sum_of_orbitals(words, n_orb):
    s = torch.zeros_like(words)
    for a in range(n_orb):
        s += ((words >> a) & 1) * a
    return s


def _sign(words, m):
    """parity of the occupied orbitals at and above m"""
    return _popc(words >> m) & 1


def _elements(words, lookup, groups):
    """(rows, targets, coefficients) of every pair p occupied in the rows and every pair q of p's group:
    F(p, q) times both fermionic signs, zero where q is not free; groups: (pairs, F), pairs (high, low)"""
    for pairs, F in groups:
        masks = [(1 << a) | (1 << b) for a, b in pairs]
        for i, (a, b) in enumerate(pairs):
            rows = torch.nonzero((words & masks[i]) == masks[i]).flatten()
            s = words[rows]
            t = s ^ masks[i]
            sg = _sign(s, a) + _sign(s, b)
            for j, (c, d) in enumerate(pairs):
                free = (t & masks[j]) == 0
                par = (sg + _sign(t, c) + _sign(t, d)) & 1
                coef = torch.where(free, 1.0 - 2.0 * par.to(torch.float64), 0.0) * F[i, j]
                yield rows, lookup(torch.where(free, t | masks[j], s)), coef


def _two_body(words, lookup, groups, x):
    """the product: y[row] += coefficient x[target]"""
    y = torch.zeros_like(x)
    for rows, target, coef in _elements(words, lookup, groups):
        y.index_add_(0, rows, coef[:, None] * x[target])
    return y


def _sphere_exact(case, seed, sectors):
    n, lz = case["n"], case["lz_max"]
    sums = torch.tensor([(t + n * lz) // 2 for t in sectors], device="cuda")
    lo, hi = int(sums.min()), int(sums.max())
    words = _subsets(n, lz + 1, lambda s, a, m: (s + m * (m - 1) // 2 <= hi) & (s + m * a - m * (m + 1) // 2 >= lo))
    total = _sum_of_orbitals(words, lz + 1)
    sector = torch.searchsorted(sums, total)
    mine = sums[sector.clamp(max=len(sectors) - 1)] == total
    words, sector = words[mine], sector[mine]
    # sectors one after the other, descending words in each
    key = torch.argsort(sector * (1 << 40) + torch.arange(words.numel() - 1, -1, -1, device="cuda"))
    place = torch.empty_like(key)
    place[key] = torch.arange(key.numel(), device="cuda")
    groups, v, rel = _sphere_pairs(case, seed)
    return words[key], (lambda t: place[torch.searchsorted(words, t)]), groups, v, rel


def _lattice_groups(case, seed):
    """the projected nearest-neighbour repulsion of the checkerboard model in its lower flat band"""
    nx, ny, m = case["nx"], case["ny"], _model(seed)
    ns = nx * ny
    i = np.arange(ns)
    kx, ky = 2 * np.pi * (i // ny) / nx, 2 * np.pi * (i % ny) / ny
    c = math.cos(math.pi / 4)
    b1 = 4 * m["t1"] * c * (np.cos(kx / 2) * np.cos(ky / 2) + 1j * np.sin(kx / 2) * np.sin(ky / 2))
    d3 = m["mus"] + 2 * m["t2"] * (np.cos(kx) - np.cos(ky))
    r = np.sqrt(d3 ** 2 + abs(b1) ** 2)
    # lower eigenvector of [[d3, b1], [b1*, -d3]], first component real and not negative
    v0 = np.where(d3 >= 0, b1, r - d3)
    v1 = np.where(d3 >= 0, -(d3 + r), -b1.conj())
    norm = np.sqrt(abs(v0) ** 2 + abs(v1) ** 2)
    v0, v1 = v0 / norm, v1 / norm
    flip = abs(v0) > 1e-300
    phase = np.where(flip, v0.conj() / np.where(flip, abs(v0), 1), v1.conj() / abs(v1))
    ua, ub = (v0 * phase).conj(), (v1 * phase).conj()
    groups = []
    for s in range(ns):
        p = [(a, b) for a in range(ns) for b in range(a + 1, ns)
             if ((a // ny + b // ny) % nx) * ny + (a % ny + b % ny) % ny == s]
        if not p:
            continue
        lo, hi = np.array(p).T
        F = np.zeros((len(p), len(p)), complex)

        def term(a, b, cc, d):
            kk = (kx[d] - kx[cc]) / 2, (ky[d] - ky[cc]) / 2
            form = 2 * (np.cos(kk[0] - kk[1]) + np.cos(kk[0] + kk[1]))
            return ua[a].conj() * ua[b] * ub[cc].conj() * ub[d] * form

        a1, a2, b1_, b2 = lo[:, None], hi[:, None], lo[None, :], hi[None, :]
        F += term(a1, b1_, a2, b2) - term(a2, b1_, a1, b2) - term(a1, b2, a2, b1_) + term(a2, b2, a1, b1_)
        F *= -2 * 0.5 / ns
        # pairs high orbital first; creating both in the other order costs a sign on each side
        groups.append(([(b, a) for a, b in p], torch.tensor(F.conj(), device="cuda")))
    return groups


def _lanczos_exact(words, lookup, groups, case):
    """lowest eigenvalues from a Lanczos run with two orthogonalisations per step"""
    d = words.numel()
    h = torch.zeros(d, d, dtype=torch.float64, device="cuda")
    for rows, target, coef in _elements(words, lookup, groups):
        h.index_put_((rows, target), coef, accumulate=True)
    if d <= 2000:
        return torch.linalg.eigvalsh((h + h.T) / 2)[:case["nev"]].cpu().numpy()
    g = torch.Generator(device="cuda").manual_seed(5)
    q = [torch.randn(d, dtype=torch.float64, device="cuda", generator=g)]
    q[0] /= q[0].norm()
    alpha, beta, last = [], [], None
    for step in range(1, 1200):
        w = h @ q[-1]
        alpha.append(float(w @ q[-1]))
        basis = torch.stack(q, 1) if step % 50 == 1 else torch.cat([basis, q[-1][:, None]], 1)
        for _ in range(2):
            w = w - basis @ (basis.T @ w)
        beta.append(float(w.norm()))
        q.append(w / beta[-1])
        if step % 40 == 0 and step > 4 * case["nev"]:
            t = np.diag(alpha) + np.diag(beta[:-1], 1) + np.diag(beta[:-1], -1)
            e = np.linalg.eigvalsh(t)[:case["nev"]]
            if last is not None and np.max(abs(e - last)) < 1e-14 * np.max(abs(e)):
                return e
            last = e
    return last


def exact(case, seed):
    kind, k = case["kind"], case.get("k", 1)
    if kind == "reorth":
        g = torch.Generator(device="cuda").manual_seed(seed)
        v = torch.empty(case["vectors"], case["rows"], k, dtype=torch.float64, device="cuda")
        v.normal_(0.0, 1.0 / math.sqrt(case["rows"]), generator=g)
        w = _vectors(case["rows"], k, seed + 1)
        h = torch.stack([b.T @ w for b in v])
        for b, m in zip(v, h):
            w = w - b @ m
        return {"h": h.reshape(-1).cpu().numpy(), "w": w}
    if kind in ("sphere", "adjoint", "lanczos", "sectors"):
        sectors = capi.sphere_sectors(case["n"], case["lz_max"]) if kind == "sectors" else [case["total_lz"]]
        words, lookup, groups, v, rel = _sphere_exact(case, seed, sectors)
        full = [(pairs, -4.0 * (u * v) @ u.T) for pairs, u in groups]
        if kind == "lanczos":
            return _lanczos_exact(words, lookup, full, case)
        x = _vectors(words.numel(), k, seed)
        y = _two_body(words, lookup, full, x)
        if kind != "adjoint":
            return y
        each = [_two_body(words, lookup, [(p, -4.0 * u[:, m:m + 1] @ u[:, m:m + 1].T) for p, u in groups], x)
                for m in range(len(rel))]
        return {"g": np.array([float((x * e).sum()) for e in each]), "hx": y}
    if kind == "lattice":
        n, ns = case["n"], case["nx"] * case["ny"]
        words = _subsets(n, ns)
        kx, ky = torch.zeros_like(words), torch.zeros_like(words)
        for a in range(ns):
            bit = (words >> a) & 1
            kx += bit * (a // case["ny"])
            ky += bit * (a % case["ny"])
        sector = (kx % case["nx"]) * case["ny"] + ky % case["ny"]
        key = torch.argsort(sector * (1 << 40) + torch.arange(words.numel() - 1, -1, -1, device="cuda"))
        place = torch.empty_like(key)
        place[key] = torch.arange(key.numel(), device="cuda")
        x = torch.view_as_complex(_vectors(words.numel(), 2 * k, seed).reshape(-1, k, 2))
        y = _two_body(words[key], lambda t: place[torch.searchsorted(words, t)], _lattice_groups(case, seed), x)
        return torch.view_as_real(y).reshape(-1, 2 * k)
    # spin chain: site 0 is the most significant of the order, rows descending
    length, up = case["length"], (case["length"] + case["sz"]) // 2
    words = _subsets(up, length)
    rows = words.numel()
    j, jz = _couplings(case, seed)
    x = _vectors(rows, k, seed)
    y = torch.zeros_like(x)
    words = words.flip(0)  # bit length-1-i is site i
    ascending = words.flip(0).contiguous()
    for i in range(length if case["periodic"] else length - 1):
        m1, m2 = 1 << (length - 1 - i), 1 << (length - 1 - (i + 1) % length)
        anti = ((words & m1) != 0) != ((words & m2) != 0)
        y += (0.25 * jz[i] * (1.0 - 2.0 * anti.to(torch.float64)))[:, None] * x
        at = torch.nonzero(anti).flatten()
        target = rows - 1 - torch.searchsorted(ascending, words[at] ^ (m1 | m2))
        y.index_add_(0, at, 0.5 * j[i] * x[target])
    return y
