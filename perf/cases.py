"""Performance cases of the package: what each stands for in use, how its inputs are made, one pass of
it, the work it cannot do without, the tolerance of its results, and its values in plain torch.

Every case is a spin-1/2 ring of N sites (nearest neighbours J1 = 1, next-nearest J2, or the XXZ
ring), in the symmetry sectors of its translations, with the reflection or the spin flip where named:
the systems of the package's benchmark and tests. A seed draws the vectors, the couplings or the
random-vector seeds of a case, so that another seed is another input.

``exact`` restates each computation over torch arrays: the orbits of the ring's group by brute force
over its bit patterns, H as index and coefficient arrays, Lanczos with full reorthogonalisation.
"""

from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import qed_spin_amd as qs
from qed_spin_amd import dynamics as dyn
from qed_spin_amd import symmetry as sym
from qed_spin_amd import thermal as th

# ---- the cases ------------------------------------------------------------------------------------


def listed():
    return [
        # One apply of a sector of a few hundred states: the blocks at the edge of a momentum walk, and
        # the requests of a serving loop; launch latency.
        {"name": "apply_n16", "kind": "apply", "N": 16, "up": 8, "k": 3, "R": 0, "Z": 0},
        # One apply of the largest sector a single GPU is used for: the J1-J2 ring of 32 sites.
        {"name": "apply_n32", "kind": "apply", "N": 32, "up": 16, "k": 0, "R": 1, "Z": 0},
        # Four vectors through one apply, rows interleaved: block methods and several right-hand sides.
        {"name": "block4_n28", "kind": "block", "N": 28, "up": 14, "k": 5, "R": 0, "Z": 0, "nv": 4},
        # The on-the-fly apply, taken when a sector's CSR does not fit its budget.
        {"name": "gather_n28", "kind": "gather", "N": 28, "up": 14, "k": 0, "R": 1, "Z": 0},
        # Fully reorthogonalised Lanczos in a small sector: every step is short, latency counts.
        {"name": "lanczos_n20", "kind": "lanczos", "N": 20, "up": 10, "k": 0, "R": 0, "Z": 0, "steps": 200},
        # The same in a large sector: the time to a ground state energy with a kept basis.
        {"name": "lanczos_n30", "kind": "lanczos", "N": 30, "up": 15, "k": 0, "R": 1, "Z": 0, "steps": 100},
        # The lowest levels of a momentum block, as the levels walk solves each block.
        {"name": "levels_n24", "kind": "levels", "N": 24, "up": 12, "k": 7, "R": 0, "Z": 0, "want": 4},
        # One block of a streamed walk: the sector enumerated, its CSR built, its lowest level estimated.
        {"name": "block_walk_n28", "kind": "walk", "N": 28, "up": 14, "k": 3, "R": 0, "Z": 1},
        # Finite-temperature Lanczos over every (Sz, k) block with many random vectors per block.
        {"name": "ftlm40_n22", "kind": "ftlm", "N": 22, "samples": 40, "krylov": 80},
        # The same with a few random vectors per block: a larger ring, where few vectors suffice.
        {"name": "ftlm4_n24", "kind": "ftlm", "N": 24, "samples": 4, "krylov": 60},
        # Zero-temperature structure factor at every momentum: one continued fraction per momentum sector.
        {"name": "cf_n26", "kind": "cf", "N": 26, "krylov": 200},
        # Finite-temperature structure factor from every (Sz, k) source sector, kept bases and overlaps.
        {"name": "dynT_n18", "kind": "dynT", "N": 18, "samples": 5, "krylov": 60},
    ]


def draw(rng):
    """One more case of the listed kinds over the sizes they stand for."""
    kind = rng.choice(["apply", "apply", "block", "gather", "lanczos", "levels", "walk", "ftlm", "ftlm", "cf", "dynT"])
    if kind == "ftlm":
        N = rng.randint(14, 21)
        return {"kind": kind, "N": N, "samples": round(2 * 20 ** rng.random()), "krylov": rng.randint(40, 80)}
    if kind == "cf":
        return {"kind": kind, "N": 2 * rng.randint(8, 12), "krylov": rng.randint(100, 200)}
    if kind == "dynT":
        return {"kind": kind, "N": rng.randint(10, 16), "samples": rng.randint(2, 6), "krylov": rng.randint(30, 60)}
    top = {"apply": 30, "block": 28, "gather": 28, "lanczos": 28, "levels": 24, "walk": 28}[kind]
    N = rng.randint(16, top)
    up = N // 2 if rng.random() < 0.5 else N // 2 - rng.randint(0, 2)
    case = {"kind": kind, "N": N, "up": up, "k": rng.randrange(N), "R": 0, "Z": 0}
    sector = rng.random()
    if sector < 0.3:
        case.update(k=0, R=rng.choice([1, -1]))
    elif sector < 0.5 and 2 * up == N:
        case.update(Z=rng.choice([1, -1]))
    if kind == "block":
        case["nv"] = rng.choice([2, 4, 8])
    if kind == "lanczos":
        case["steps"] = rng.randint(40, 150)
    if kind == "levels":
        case["want"] = rng.randint(1, 6)
    return case


# ---- inputs ---------------------------------------------------------------------------------------


def _couplings(case, seed):
    """J2 of this seed (the XXZ ring of the thermal cases has its anisotropy instead)."""
    return 0.3 + 0.2 * float(np.random.default_rng(seed).random())


def _hamiltonian(case, seed):
    N, g = case["N"], _couplings(case, seed)
    b = qs.HamiltonianBuilder(N)
    if case["kind"] == "ftlm" and case["samples"] >= 8:
        b.xxz([(i, (i + 1) % N) for i in range(N)], 1.0, 0.3 + g)
    else:
        b.heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0)
        if case["kind"] != "cf":   # the continued fractions: the Heisenberg ring, one ground state at a known momentum
            b.heisenberg([(i, (i + 2) % N) for i in range(N)], g)
    return b.to_operator()


def _group(case):
    N = case["N"]
    g = sym.dihedral_group(N, case["k"], case["R"]) if case["R"] else sym.chain_group(N, case["k"])
    return sym.with_spin_flip(g, case["Z"]) if case["Z"] else g


class _Vector:
    """A torch tensor as a vector of the package (its ``ptr``)."""

    def __init__(self, t):
        self.t = t
        self.ptr = C.c_void_p(t.data_ptr())


def _random(n, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(n, dtype=dtype, device="cuda", generator=gen)


def _omega():
    return np.linspace(0.0, 4.0, 200)


def _cf_momentum(N):
    """The ground state's momentum of the Heisenberg ring: 0 for N = 4 n, pi for N = 4 n + 2."""
    return 0 if N % 4 == 0 else N // 2


def prepare(case, seed):
    kind, N = case["kind"], case["N"]
    H = _hamiltonian(case, seed)
    if kind == "walk":
        return {"case": case, "H": H, "group": _group(case)}
    if kind == "ftlm":
        blocks = [b for b in th.walk_blocks(H, qs.Symmetry(), tune=False, fold=True) if b[1].dim > 128]
        return {"case": case, "blocks": blocks, "seeds": _block_seeds(seed, len(blocks)), "betas": 1.0 / _temperatures()}
    if kind == "cf":
        blocks = th.walk_blocks(H, qs.Symmetry(sz=[N // 2]), tune=False)
        ground = [i for i, b in enumerate(blocks) if b[0].momentum == _cf_momentum(N)]
        # the probes of another seed are weighted differently: S^z(q) times 1 + its draw
        w = 0.5 + np.random.default_rng(seed).random(N)
        probes = []
        for m in range(N):
            op = qs.Operator(N)
            for ops, sites, c in dyn.sz_q(N, 2 * math.pi * m / N).products:
                op.add_product(ops, sites, c * w[m])
            probes.append(op)
        return {"case": case, "H": H, "blocks": blocks, "ground": ground, "probes": probes}
    if kind == "dynT":
        blocks = th.walk_blocks(H, qs.Symmetry(), tune=False)
        return {"case": case, "H": H, "blocks": blocks, "seed": 11 + seed,
                "probe": dyn.sz_q(N, 2 * math.pi * (N // 3) / N)}
    sector = qs.Sector(_group(case), case["up"])
    lane = qs.LANE_GATHER if kind == "gather" else qs.LANE_CSR
    m = qs.SectorMatvec(H, sector, lane=lane)
    state = {"case": case, "sector": sector, "m": m}
    dtype = torch.float64 if m.is_real else torch.complex128
    if kind in ("apply", "gather", "block"):
        n = sector.dim * case.get("nv", 1)
        state["x"], state["y"] = _Vector(_random(n, dtype, seed)), _Vector(torch.zeros(n, dtype=dtype, device="cuda"))
    if kind == "lanczos":
        state["v0"] = _random(sector.dim, dtype, seed).cpu().numpy()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("apply", "gather"):
        state["m"].apply(state["x"], state["y"])
        return state["y"].t
    if kind == "block":
        state["m"].apply_block(case["nv"], state["x"], state["y"])
        return state["y"].t
    if kind == "lanczos":
        alpha, beta, _ = state["m"].lanczos(state["v0"], case["steps"])
        return {"alpha": alpha, "beta": beta}
    if kind == "levels":
        values, converged, _ = state["m"].lowest(case["want"])
        return {"values": values, "converged": converged}
    if kind == "walk":
        sector = qs.Sector(state["group"], case["up"])
        m = qs.SectorMatvec(state["H"], sector, lane=qs.LANE_CSR)
        return {"dim": sector.dim, "nnz": int(m.info["nnz"]), "estimate": m.estimate()}
    if kind == "ftlm":
        lnZ, E, V, e_min, _ = th.ftlm_batched([b[2] for b in state["blocks"]], case["samples"], case["krylov"],
                                              state["seeds"], state["betas"])
        return {"lnZ": lnZ, "E": E, "V": V, "e_min": e_min}
    if kind == "cf":
        r = dyn.dynamics(state["H"], state["probes"], _omega(), eta=0.1, krylov=case["krylov"], blocks=state["blocks"],
                         ground_blocks=state["ground"])
        return {"S": np.array(r.S), "norms": r.norms, "e0": float(r.e0)}
    r = dyn.dynamics(state["H"], [state["probe"]], _omega(), eta=0.1, T=[0.5, 1.0], samples=case["samples"],
                     krylov=case["krylov"], seed=state["seed"], blocks=state["blocks"])
    # real parts: the autocorrelation's imaginary part is roundoff
    return {"S": np.ascontiguousarray(r.S[0].real), "e0": float(r.e0)}


def _temperatures():
    return np.linspace(0.2, 4.0, 20)


def _block_seeds(seed, n):
    s, out = 1 + int(seed), []
    for _ in range(n):
        s = th.next_block_seed(s)
        out.append(s)
    return out


# ---- work and tolerance ---------------------------------------------------------------------------


def _dim(case):
    """The sector's states, to a few per cent for the small ones."""
    G = case["N"] * (2 if case["R"] else 1) * (2 if case["Z"] else 1)
    return max(1, math.comb(case["N"], case["up"]) // G)


def _row(N, up, bonds):
    """Mean entries of a row of H: the diagonal and every antiparallel bond."""
    return 1 + bonds * 2 * up * (N - up) / (N * (N - 1))


def _blocks_rows(N, least):
    """Rows of the (Sz, k) blocks above `least` states, each time-reversal pair once; entries per row."""
    rows = nnz = 0.0
    for up in range(N + 1):
        d = math.comb(N, up) / N
        if d > least:
            rows += d * (N // 2 + 1)
            nnz += d * (N // 2 + 1) * _row(N, up, N)
    return rows, nnz


def work(case):
    N, kind = case["N"], case["kind"]
    if kind in ("ftlm", "cf", "dynT"):
        R, steps = case.get("samples", 1), case["krylov"]
        if kind == "ftlm":
            rows, nnz = _blocks_rows(N, 128)
            nnz *= 1 if case["samples"] >= 8 else 2
        elif kind == "cf":
            rows = float(math.comb(N, N // 2))
            nnz = rows * _row(N, N // 2, N)
        else:   # source and target runs of every source sector, their bases kept
            rows, steps = 2.0 ** (N + 1), case["krylov"]
            nnz = rows * (1 + N)
        # per step: the matrix once, the vector in, the next one out; full reorthogonalisation of the
        # kept bases reads them twice
        kept = rows * R * 16 * steps if kind == "dynT" else 0.0
        by = steps * (nnz * 6 + rows * 8 + 2 * rows * R * 16 + kept)
        return {"bytes": by, "flops": steps * (8 * nnz * R + 16 * rows * R + kept / 2)}
    real = case["Z"] in (0, 1, -1) and (2 * case["k"]) % N == 0
    s, D = (8 if real else 16), float(_dim(case))
    nnz = D * _row(N, case["up"], 2 * N)
    per = 2 if real else 8
    matrix = nnz * 5 + D * 2
    if kind in ("apply", "block"):
        nv = case.get("nv", 1)
        return {"bytes": matrix + 2 * D * s * nv, "flops": per * nnz * nv}
    if kind == "gather":   # no matrix: the representatives, the norms and the two vectors
        return {"bytes": D * 16 + 2 * D * s, "flops": per * nnz}
    if kind == "lanczos":   # a full Gram-Schmidt pass reads the kept basis twice
        m = case["steps"]
        return {"bytes": m * (matrix + 4 * D * s) + m * (m - 1) * D * s, "flops": m * per * nnz + m * m * 2 * per * D}
    if kind == "levels":
        m = 120
        return {"bytes": m * (matrix + 4 * D * s) + m * 40 * 2 * D * s, "flops": m * per * nnz + m * 80 * per * D}
    # the walk: the sector and the matrix written once, then 40 Lanczos steps
    return {"bytes": D * 16 + matrix + 40 * (matrix + 4 * D * s), "flops": 40 * per * nnz}


def tolerance(case):
    kind = case["kind"]
    if kind in ("apply", "block", "gather"):
        return {"rel": 1e-14, "max": 1e-12}
    if kind == "lanczos":
        return {"rel": 1e-12, "max": 1e-11}
    if kind == "levels":
        return {"rel": 1e-11, "max": 1e-10}
    if kind == "walk":
        return {"rel": 1e-11, "max": 1e-11}
    if kind == "ftlm":
        return {"rel": 1e-8, "max": 1e-5}
    if kind == "cf":
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 1e-6, "max": 1e-4}


# ---- the same values in plain torch ---------------------------------------------------------------

_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _popcount(x):
    x = x - ((x >> 1) & 0x5555555555555555)
    x = (x & 0x3333333333333333) + ((x >> 2) & 0x3333333333333333)
    x = (x + (x >> 4)) & 0x0F0F0F0F0F0F0F0F
    return (x * 0x0101010101010101) >> 56


def _key_bits(N, elements):
    """Where each site sits in the order that representatives are least in: from 24 sites and 16
    permutations on, the ring's sites mod b (b the least divisor from 2 to 8 with N / b <= 16) form
    blocks, block 0 on the highest bits; else the sites in order."""
    if N >= 24 and elements >= 16:
        for b in range(2, 9):
            if N % b == 0 and N // b <= 16:
                L = N // b
                return [N - (s % b + 1) * L + s // b for s in range(N)]
    return list(range(N))


class _Orbits:
    """The orbits of the ring's bit patterns under translations (reflections, the spin flip) with `up`
    set bits: ascending representatives, stabilisers as bit masks over the elements, and for each
    bond the representative and the element that a spin exchange leads to."""

    def __init__(self, N, up, reflect=False, flip=False):
        self.N, self.up = N, up
        perms = [[(i + a) % N for i in range(N)] for a in range(N)]
        if reflect:
            perms += [[(a - i) % N for i in range(N)] for a in range(N)]
        key = _key_bits(N, len(perms))
        self.elements = [(p, 0) for p in perms] + ([(p, 1) for p in perms] if flip else [])
        assert len(self.elements) <= 64
        half = 16
        v = torch.arange(1 << half, dtype=torch.int64, device=_DEV)

        def table(bit_of):   # input bit -> output bit, as two 16-bit lookup tables
            lo, hi = torch.zeros_like(v), torch.zeros_like(v)
            for i in range(N):
                t, j = (lo, i) if i < half else (hi, i - half)
                t |= ((v >> j) & 1) << bit_of[i]
            return lo, hi

        self.images = []
        full = (1 << N) - 1
        for p, z in self.elements:
            out = [0] * N
            for i in range(N):
                out[p[i]] = key[i]   # bit i of the image is bit p[i] of the state
            self.images.append((*table(out), full if z else 0))
        site_of = [0] * N
        for s in range(N):
            site_of[key[s]] = s
        self.unkey = table(site_of)
        self.key = table(key)
        reps = []
        step = 1 << min(N, 27)
        for base in range(0, 1 << N, step):
            s = torch.arange(base, min(base + step, 1 << N), dtype=torch.int64, device=_DEV)
            s = s[_popcount(s) == up]
            for im in self.images:
                if s.numel() == 0:
                    break
                s = s[self._map(im, s) >= self._look(self.key, s)]
            reps.append(s)
        self.reps = torch.cat(reps)
        k0 = self._look(self.key, self.reps)
        self.stab = torch.zeros_like(self.reps)
        for g, im in enumerate(self.images):
            self.stab |= (self._map(im, self.reps) == k0).to(torch.int64) << g

    @staticmethod
    def _look(tab, s):
        return tab[0][s & 0xFFFF] | tab[1][s >> 16]

    def _map(self, im, s):
        return self._look(im, s) ^ im[2]

    def norms(self, chars):
        """Sum of the characters over each stabiliser (0 where the sector holds no such state)."""
        masks, inverse = torch.unique(self.stab, return_inverse=True)
        S = []
        for mk in masks.tolist():
            t = sum((c for g, c in enumerate(chars) if (mk >> g) & 1), 0j)
            S.append(t.real if abs(t) > 1e-6 else 0.0)
        return torch.tensor(S, dtype=torch.float64, device=_DEV)[inverse]

    def exchange(self, i, j):
        """(antiparallel, representative index, element) of the spin exchange on sites i and j."""
        s = self.reps
        anti = ((s >> i) ^ (s >> j)) & 1 == 1
        t = torch.where(anti, s ^ ((1 << i) | (1 << j)), s)
        best = self._map(self.images[0], t)
        el = torch.zeros_like(t, dtype=torch.uint8)
        for g, im in enumerate(self.images[1:], 1):
            v = self._map(im, t)
            less = v < best
            best = torch.where(less, v, best)
            el[less] = g
        return anti, torch.searchsorted(self.reps, self._look(self.unkey, best)), el


class _Block:
    """H of one sector: y = diag x + sum_b val_b x[idx_b]."""

    def __init__(self, orbits, maps, chars, bonds, real):
        S = orbits.norms(chars)
        keep = S > 0.5
        self.keep, self.S = keep, S[keep]
        self.dim = int(keep.sum())
        place = torch.cumsum(keep.to(torch.int64), 0) - 1
        ch = torch.tensor(chars, dtype=torch.complex128, device=_DEV)
        if real:
            ch = ch.real
        w = 1.0 / torch.sqrt(self.S)
        reps = orbits.reps[keep]
        self.diag = torch.zeros(self.dim, dtype=torch.float64, device=_DEV)
        self.terms = []
        for (i, j, jxy, jz), (anti, to, el) in zip(bonds, maps):
            par = 1 - 2 * (((reps >> i) ^ (reps >> j)) & 1)
            self.diag += 0.25 * jz * par.to(torch.float64)
            a, t = anti[keep], to[keep]
            on = a & keep[t]
            c = torch.where(on, place[t], torch.zeros_like(t))
            # the orbit of the target is entered through element g: (w_r / w_c) J/2 chi(g)
            val = (0.5 * jxy) * (w / w[c]) * on.to(torch.float64) * ch[el[keep].to(torch.int64)]
            self.terms.append((c.to(torch.int32), val))

    def apply(self, x):
        wide = x.dim() == 2
        f = (lambda t: t[:, None]) if wide else (lambda t: t)
        y = f(self.diag) * x
        for c, val in self.terms:
            y += f(val) * x[c]
        return y


def _bonds(case, seed):
    N, g = case["N"], _couplings(case, seed)
    near = [(i, (i + 1) % N) for i in range(N)]
    if case["kind"] == "ftlm" and case["samples"] >= 8:
        return [(i, j, 1.0, 0.3 + g) for i, j in near]
    b = [(i, j, 1.0, 1.0) for i, j in near]
    return b if case["kind"] == "cf" else b + [(i, (i + 2) % N, g, g) for i in range(N)]


def _chars(N, k, R=0, Z=0):
    c = [sym_root(k * a, N) for a in range(N)]
    if R:
        c = c + [R * x for x in c]
    if Z:
        c = c + [Z * x for x in c]
    return c


def sym_root(p, L):
    th_ = 2 * math.pi * (p % L) / L
    return complex(math.cos(th_), math.sin(th_)) if (4 * p) % L else [1 + 0j, 1j, -1 + 0j, -1j][(4 * (p % L)) // L]


def _is_real(N, k):
    return (2 * k) % N == 0


def _block(case, seed, k=None):
    N = case["N"]
    k = case["k"] if k is None else k
    orbits = _Orbits(N, case["up"], reflect=bool(case["R"]), flip=bool(case["Z"]))
    bonds = _bonds(case, seed)
    maps = [orbits.exchange(i, j) for i, j, _, _ in bonds]
    return _Block(orbits, maps, _chars(N, k, case["R"], case["Z"]), bonds, _is_real(N, k))


def _lanczos(H, v, steps, least=1e-13):
    """Lanczos with two Gram-Schmidt passes against the whole basis: alpha, beta (beta[0] = 0), basis."""
    V = torch.empty((steps, v.numel()), dtype=v.dtype, device=v.device)
    V[0] = v / torch.linalg.vector_norm(v)
    alpha, beta = [], [0.0]
    for j in range(steps):
        w = H.apply(V[j])
        a = torch.vdot(V[j], w).real
        alpha.append(float(a))
        for _ in range(2):
            w = w - (V[: j + 1].conj() @ w) @ V[: j + 1]
        b = float(torch.linalg.vector_norm(w))
        beta.append(b)
        if b < least or j + 1 == steps:
            break
        V[j + 1] = w / b
    return np.array(alpha), np.array(beta), V[: len(alpha)]


def _tridiagonal(alpha, beta):
    m = len(alpha)
    return np.diag(alpha) + np.diag(beta[1:m], 1) + np.diag(beta[1:m], -1)


def _hash64(z):
    """splitmix64's output function over torch int64 words (wrapping products, logical shifts)."""
    def shr(x, n):
        return (x >> n) & ((1 << (64 - n)) - 1)

    def wrap(x):
        return x - (1 << 64) if x >= 1 << 63 else x

    z = z + wrap(0x9E3779B97F4A7C15)
    z = (z ^ shr(z, 30)) * wrap(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * wrap(0x94D049BB133111EB)
    return z ^ shr(z, 31)


def _box_muller(n, seed):
    """The fixed start vector of the block estimate: entry i from the hashes of seed ^ 2i and seed ^ (2i + 1)."""
    i = torch.arange(n, dtype=torch.int64, device=_DEV)
    a, b = _hash64(seed ^ (2 * i)), _hash64(seed ^ (2 * i + 1))
    u1 = ((((a >> 11) & ((1 << 53) - 1)).to(torch.float64)) + 0.5) * 2.0 ** -53
    u2 = ((b >> 11) & ((1 << 53) - 1)).to(torch.float64) * 2.0 ** -53
    r = torch.sqrt(-2.0 * torch.log(u1))
    return torch.complex(r * torch.cos(2 * math.pi * u2), r * torch.sin(2 * math.pi * u2))


def _splitmix(base, i):
    m = (1 << 64) - 1
    z = (int(base) + 0x9E3779B97F4A7C15 * (int(i) + 1)) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def _normals(n, seed32):
    """n complex normals by the polar method on a Mersenne Twister's 53-bit uniforms, two words each
    (the first normal of a pair is the imaginary part)."""
    words = np.random.RandomState(seed32)
    out, have = [], 0
    while have < n:
        c = int((n - have) * 1.3) + 64
        u = torch.from_numpy(words.randint(0, 1 << 32, size=4 * c, dtype=np.uint32).astype(np.int64)).to(_DEV)
        u = u.reshape(-1, 2)
        u = (u[:, 0].to(torch.float64) + u[:, 1].to(torch.float64) * 2.0 ** 32) * 2.0 ** -64
        u = torch.where(u >= 1.0, torch.full_like(u, 1.0 - 2.0 ** -53), u).reshape(-1, 2) * 2.0 - 1.0
        x, y = u[:, 0], u[:, 1]
        r2 = x * x + y * y
        ok = (r2 <= 1.0) & (r2 != 0.0)
        x, y, r2 = x[ok], y[ok], r2[ok]
        f = torch.sqrt(-2.0 * torch.log(r2) / r2)
        out.append(torch.complex(x * f, y * f))
        have += out[-1].numel()
    return torch.cat(out)[:n]


class _Union:
    """The blocks of a walk as one block-diagonal operator over stacked rows."""

    def __init__(self, blocks):
        self.dims = [b.dim for b in blocks]
        off = np.cumsum([0] + self.dims)
        self.of = torch.repeat_interleave(torch.arange(len(blocks), device=_DEV), torch.tensor(self.dims, device=_DEV))
        self.diag = torch.cat([b.diag for b in blocks])
        self.terms = []
        for t in range(len(blocks[0].terms)):
            self.terms.append((torch.cat([b.terms[t][0] + int(o) for b, o in zip(blocks, off)]),
                               torch.cat([b.terms[t][1].to(torch.complex128) for b in blocks])))

    def apply(self, x):
        y = self.diag[:, None] * x
        for c, val in self.terms:
            y += val[:, None] * x[c]
        return y

    def sums(self, x):
        """Per block and column."""
        out = torch.zeros((len(self.dims), x.shape[1]), dtype=x.dtype, device=_DEV)
        return out.index_add_(0, self.of, x)


def _exact_ftlm(case, seed):
    N, R, M = case["N"], case["samples"], case["krylov"]
    rows, _ = _blocks_rows(N, 128)
    if rows * R > 2.5e7:
        return None   # the start vectors alone take most of a minute
    bonds = _bonds(case, seed)
    blocks = []
    for up in range(N + 1):
        if math.comb(N, up) < 128:
            continue
        orbits = _Orbits(N, up)
        maps = [orbits.exchange(i, j) for i, j, _, _ in bonds]
        for k in range(N // 2 + 1):
            b = _Block(orbits, maps, _chars(N, k), bonds, _is_real(N, k))
            if b.dim > 128:
                blocks.append(b)
    seeds = _block_seeds(seed, len(blocks))
    U = _Union(blocks)
    del blocks
    V = torch.cat([torch.stack([_normals(d, _splitmix(s, i) & 0xFFFFFFFF) for i in range(R)], 1)
                   for d, s in zip(U.dims, seeds)])
    V = V / torch.sqrt(U.sums((V.conj() * V).real))[U.of]
    nb = len(U.dims)
    alpha, beta = torch.zeros((M, nb, R), device=_DEV, dtype=torch.float64), torch.zeros((M, nb, R), device=_DEV, dtype=torch.float64)
    prev = torch.zeros_like(V)
    for j in range(M):
        W = U.apply(V)
        if j:
            W -= beta[j - 1][U.of] * prev
        alpha[j] = U.sums((V.conj() * W).real)
        W -= alpha[j][U.of] * V
        W -= U.sums(V.conj() * W)[U.of] * V
        beta[j] = torch.sqrt(U.sums((W.conj() * W).real))
        prev, V = V, W / beta[j][U.of]
    T = torch.diag_embed(alpha.permute(1, 2, 0)) + torch.diag_embed(beta[:-1].permute(1, 2, 0), 1) + torch.diag_embed(beta[:-1].permute(1, 2, 0), -1)
    e, y = torch.linalg.eigh(T.cpu())
    e, w = e.numpy().reshape(nb, -1), (y[:, :, 0, :] ** 2).numpy().reshape(nb, -1)
    betas = 1.0 / _temperatures()
    lnZ, E, Var = (np.zeros((nb, betas.size)) for _ in range(3))
    low = e.min(1)
    for b in range(nb):
        g = w[b][:, None] * np.exp(-np.outer(e[b] - low[b], betas))
        Z = g.sum(0)
        lnZ[b] = np.log(U.dims[b] / R * Z) - betas * low[b]
        E[b] = (g * e[b][:, None]).sum(0) / Z
        Var[b] = (g * (e[b][:, None] - E[b]) ** 2).sum(0) / Z
    return {"lnZ": lnZ, "E": E, "V": Var, "e_min": None}


def _exact_cf(case, seed):
    N, M = case["N"], case["krylov"]
    bonds = _bonds(case, seed)
    orbits = _Orbits(N, N // 2)
    maps = [orbits.exchange(i, j) for i, j, _, _ in bonds]
    kg = _cf_momentum(N)
    H0 = _Block(orbits, maps, _chars(N, kg), bonds, True)
    v = torch.randn(H0.dim, dtype=torch.float64, device=_DEV, generator=torch.Generator(device=_DEV).manual_seed(1))
    a, b, V = _lanczos(H0, v, min(H0.dim, 160))
    e, y = np.linalg.eigh(_tridiagonal(a, b))
    g = torch.from_numpy(y[:, 0]).to(_DEV) @ V
    g = g / torch.linalg.vector_norm(g)
    e0 = float(torch.dot(g, H0.apply(g)))
    full = torch.zeros(orbits.reps.numel(), dtype=torch.float64, device=_DEV)
    full[H0.keep] = g * torch.sqrt(H0.S)
    wq = 0.5 + np.random.default_rng(seed).random(N)
    omega = _omega()
    S, norms = np.zeros((N, omega.size)), np.zeros(N)
    for m in range(N):
        lam = torch.zeros(orbits.reps.numel(), dtype=torch.complex128, device=_DEV)
        for j in range(N):
            lam += sym_root(-m * j, N) * (((orbits.reps >> j) & 1).to(torch.float64) - 0.5)
        k = (kg - m) % N
        H = _Block(orbits, maps, _chars(N, k), bonds, False)
        phi = (lam * full)[H.keep] / torch.sqrt(H.S) * (wq[m] / math.sqrt(N))
        n2 = float(torch.linalg.vector_norm(phi)) ** 2
        norms[m] = n2
        if n2 < 1e-20:
            continue
        a, b, _ = _lanczos(H, phi, min(M, H.dim))
        z = omega + 0.1j + e0
        G = np.zeros_like(z)
        for j in range(len(a) - 1, -1, -1):
            G = 1.0 / (z - a[j] - (b[j + 1] ** 2 * G if j + 1 < len(a) else 0.0))
        S[m] = -n2 * G.imag / math.pi
    return {"S": S, "norms": norms, "e0": e0}


def exact(case, seed):
    kind, N = case["kind"], case["N"]
    if kind == "ftlm":
        return _exact_ftlm(case, seed)
    if kind == "cf":
        return _exact_cf(case, seed)
    if kind == "dynT":
        return None   # every source sector's runs one after another: minutes in plain torch
    H = _block(case, seed)
    dtype = torch.float64 if _is_real(N, case["k"]) else torch.complex128
    if kind in ("apply", "gather", "block"):
        nv = case.get("nv", 1)
        x = _random(H.dim * nv, dtype, seed)
        return H.apply(x.reshape(H.dim, nv)).reshape(-1) if nv > 1 else H.apply(x)
    if kind == "lanczos":
        a, b, _ = _lanczos(H, _random(H.dim, dtype, seed), min(case["steps"], H.dim))
        return {"alpha": a, "beta": b}
    if kind == "levels":
        # a degenerate level needs a start of its own for each copy: deflate what is found
        found, vecs = [], []
        gen = torch.Generator(device=_DEV).manual_seed(5)

        class Deflated:
            def apply(self, x):
                y = H.apply(x)
                for e, v in vecs:
                    y = y + (1e3 - e) * v * torch.vdot(v, x)
                return y

        D = Deflated()
        for _ in range(min(case["want"], H.dim)):
            v = torch.randn(H.dim, dtype=dtype, device=_DEV, generator=gen)
            a, b, V = _lanczos(D, v, min(H.dim, 180))
            e, y = np.linalg.eigh(_tridiagonal(a, b))
            u = torch.from_numpy(y[:, 0]).to(V.dtype).to(_DEV) @ V
            u = u / torch.linalg.vector_norm(u)
            val = float(torch.vdot(u, H.apply(u)).real)
            found.append(val)
            vecs.append((val, u))
        return {"values": np.sort(np.array(found)), "converged": None}
    start = _box_muller(H.dim, 0x5EED0002)
    a, b, _ = _lanczos(H, start.real.contiguous() if dtype == torch.float64 else start, min(40, H.dim))
    e, y = np.linalg.eigh(_tridiagonal(a, b))
    return {"dim": None, "nnz": None, "estimate": float(e[0] - b[len(a)] * abs(y[-1, 0]))}
