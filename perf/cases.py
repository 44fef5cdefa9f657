"""The work whose speed is measured: what a program that uses this library has it do.

A case is a dict of plain values. Its "kind" is the call:

  solve         model tables -> basis -> ELL matrix -> Lanczos: the lowest energies of one sector
  assemble      basis -> ELL matrix -> one product: what a program pays that builds many sectors
  apply         y = H x on device vectors with a matrix that is kept (a caller's own iteration)
  batched       the lowest energies of many sectors in one call
  correlations  expectation values of two-site and structure-factor operators in a ground state
  train         loss and gradient of the learned start's network over a grid of ground states
  start         the learned start vector of one sector

Lattices are periodic: "n1" x "n2" sites (a chain has n2 = 1), nearest-neighbour XXZ coupling and,
with "next", a second-neighbour coupling along the chain. Delta, the second-neighbour coupling, start
vectors, network weights and x come from the seed. The sector is (n_up, momentum kx, ky, spin-flip
"parity" or -1 without it, "turn" = irrep of the quarter turns about a site or -1 without them).

`exact` restates the sector matrix, its lowest eigenpairs, the expectation values and the network in
64-bit torch, from the states' images under the group; it shares no code with the library.
"""
import math

import numpy as np
import torch

import qmbcuda_amd as q
from qmbcuda_amd import models as LM

_CTX = None


def _ctx():
    """The one context that a program keeps."""
    global _CTX
    if _CTX is None:
        _CTX = q.Context(0)
    return _CTX


def _case(name, kind, n1, n2=1, **kw):
    n = n1 * n2
    c = {"name": name, "kind": kind, "n1": n1, "n2": n2, "n_up": n // 2, "kx": 0, "ky": 0, "parity": -1, "turn": -1,
         "next": False, "locality": True, "n_eigs": 1, "vector": False, "tol": 1e-12}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest whole call: a 16-site ring, energy and ground-state vector; launches, copies and
        # synchronisations count, as in a scan over couplings on a small ring
        _case("solve_chain16", "solve", 16, parity=0, vector=True, tol=1e-13),
        # the single-sector workload of the benchmark: J1-J2 chain of 28 sites, 716,728 rows
        _case("solve_chain28_next", "solve", 28, parity=0, next=True),
        # several levels of a complex momentum sector of an odd ring (208,012 rows), kept vectors
        _case("solve_chain25_k4_three", "solve", 25, n_up=12, kx=4, n_eigs=3, vector=True, tol=1e-13),
        # the headline: 6x6 square lattice, 126,056,625 rows, selective orthogonalisation
        _case("solve_square6x6", "solve", 6, 6, parity=0, scheme=3, check_every=1, max_iter=100),
        # a sweep over point-group sectors: 100 permutations of 25 sites, no cyclic structure
        _case("assemble_square5x5_c4", "assemble", 5, 5, n_up=12, turn=0, locality=False),
        # products with a matrix that stays in the caches: 56,822 rows
        _case("apply_chain24", "apply", 24, parity=0, locality=False),
        # complex products, 1,432,860 rows, table-order slots (the default of the class interface)
        _case("apply_chain28_k5_next", "apply", 28, kx=5, next=True, locality=False),
        # products with a matrix that streams from memory: 4x8 lattice, 9.4 million rows
        _case("apply_square4x8", "apply", 4, 8, parity=0),
        # 72 momentum and magnetisation sectors of a 24-site ring, lowest four levels of each
        _case("batched_chain24_72", "batched", 24, n_eigs=4, tol=1e-13, sweep="12,14,16"),
        # spin correlations and the structure factor of the 28-site ground state
        _case("correlations_chain28", "correlations", 28, parity=0, next=True),
        # one step's loss and gradient over 192 ground states: rings of 20, 22 and 24 sites
        _case("train_rings_192", "train", 24, grid=8, sizes="20,22,24"),
        # inference: the learned start vector of the 30-site ring, 5,170,604 rows
        _case("start_chain30", "start", 30, next=True),
    ]


def draw(rng):
    kind = rng.choice(("solve", "solve", "assemble", "apply", "apply", "batched", "correlations", "train", "start"))
    square = rng.choice(((3, 3), (3, 4), (4, 4), (3, 5), (3, 6), (4, 5), (5, 5), (4, 6), (3, 9), (4, 7), (5, 6), (4, 8)))
    if kind == "batched":
        n = rng.randint(11, 23)
        ups = sorted(rng.sample(range(max(2, n // 2 - 3), n // 2 + 4), rng.randint(1, 3)))
        c = _case("", kind, n, n_eigs=rng.randint(1, 4), tol=1e-13, sweep=",".join(map(str, ups)),
                  next=rng.random() < 0.5)
    elif kind == "train":
        sizes = sorted(rng.sample(range(10, 24, 2), rng.randint(1, 3)))
        c = _case("", kind, sizes[-1], grid=rng.randint(2, 8), sizes=",".join(map(str, sizes)))
    elif kind == "start":
        c = _case("", kind, 2 * rng.randint(6, 15), next=rng.random() < 0.5)
    else:
        lattice = square if kind != "correlations" and rng.random() < 0.4 else (rng.randint(12, 30), 1)
        c = _case("", kind, *lattice, next=lattice[1] == 1 and rng.random() < 0.5, locality=rng.random() < 0.6)
        n = c["n1"] * c["n2"]
        c["n_up"] = n // 2 - rng.choice((0, 0, 0, 1, 2))
        if lattice[0] == lattice[1] and rng.random() < 0.6:
            c["turn"] = rng.choice((0, 2))
        elif kind != "correlations":
            c["kx"] = rng.choice((0, 0, rng.randrange(c["n1"])))
            c["ky"] = rng.choice((0, rng.randrange(c["n2"])))
        if 2 * c["n_up"] == n and c["turn"] < 0 and rng.random() < 0.6:
            c["parity"] = 0
        if kind == "solve":
            c["n_eigs"] = rng.choice((1, 1, 2, 3)) if n < 28 else 1
            c["vector"] = n < 28 and rng.random() < 0.5
            c["tol"] = 1e-13
    del c["name"]
    return c


# ---- what a program has in hand --------------------------------------------------


def _couplings(case, seed):
    r = np.random.default_rng([seed, 1])
    return float(r.uniform(0.8, 1.2)), float(r.uniform(0.1, 0.5)) if case["next"] else 0.0


def _lattice(case, delta, j2):
    return LM.square(case["n1"], case["n2"], 1.0, delta) if case["n2"] > 1 else LM.chain(case["n1"], 1.0, delta, j2)


def _group(case, lat):
    ge, fl, ch = LM.translation_group(lat, spin_flip=case["parity"] >= 0)
    irrep = LM.momentum_irrep(lat, case["kx"], case["ky"], case["parity"] if case["parity"] >= 0 else None)
    if case["turn"] >= 0:
        turns = LM.rotation_group(lat)
        ge, fl, ch, pairs = LM.product_group((ge, fl, ch), turns)
        irrep = pairs.index((irrep, case["turn"]))
    return q.Group(ge, ch, fl if case["parity"] >= 0 else None), irrep


def _model(case, seed):
    """The tables of one sector: group, irrep index and Hamiltonian terms."""
    lat, info = _lattice(case, *_couplings(case, seed))
    group, irrep = _group(case, lat)
    return {"lat": lat, "group": group, "irrep": irrep, "terms": q.Terms(lat.n_sites, LM.term_table(lat, info))}


def _basis(case, m):
    return q.Basis(_ctx(), m["group"], case["n_up"], m["irrep"], q.LAYOUT_COMPACT)


def _vector(case, seed, n, is_complex):
    """A unit vector like the ones of a Krylov iteration: every entry filled, no pattern."""
    g = torch.Generator(device="cuda").manual_seed(1000 + seed)
    x = torch.randn(n, dtype=torch.complex128 if is_complex else torch.float64, device="cuda", generator=g)
    return x / torch.linalg.vector_norm(x)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind, "seed": seed}
    if kind == "batched":
        lat, info = _lattice(case, *_couplings(case, seed))
        s["group"], _ = _group(case, lat)
        s["terms"] = q.Terms(lat.n_sites, LM.term_table(lat, info))
        s["ells"] = [q.Ell(_ctx(), q.Basis(_ctx(), s["group"], up, k), s["terms"], locality_slots=True)
                     for up in map(int, case["sweep"].split(",")) for k in range(case["n1"])]
    elif kind == "train":
        s.update(_training_set(case, seed))
    elif kind == "start":
        lat = LM.Lattice(case["n1"])
        group, irrep = _group(case, lat)
        s["basis"] = q.Basis(_ctx(), group, case["n_up"], irrep)
        s["net"] = q.Mlp(_ctx(), seed=seed)
        s["theta"] = s["net"].params()
        s["couplings"] = _couplings(case, seed)
    else:
        s.update(_model(case, seed))
        if kind in ("apply", "assemble"):
            basis = _basis(case, s)
            ell = q.Ell(_ctx(), basis, s["terms"], locality_slots=case["locality"])
            s["x"] = _vector(case, seed, basis.n_rows, ell.is_complex)
            s["y"] = torch.empty_like(s["x"])
            if kind == "apply":
                s["ell"] = ell
        elif kind == "correlations":
            s["basis"] = _basis(case, s)
            ell = q.Ell(_ctx(), s["basis"], s["terms"], locality_slots=True)
            s["x"] = q.lanczos(ell, max_iter=1000, tol=1e-12, want_eigvec=True)[3]
            n = case["n1"]
            s["operators"] = [q.Terms(n, LM.operator_table(LM.spin_spin(0, r))) for r in _distances(n)]
            s["operators"].append(q.Terms(n, LM.operator_table(LM.structure_factor_zz(s["lat"], n // 2))))
    torch.cuda.synchronize()
    return s


def _distances(n):
    return sorted({1, 2, 3, n // 4, n // 2})


def _training_set(case, seed):
    """Rings of several sizes, every one over a grid of couplings: bases, ground states, a fresh network."""
    r = np.random.default_rng([seed, 2])
    net, vectors, grid = q.Mlp(_ctx(), seed=seed), [], case["grid"]
    deltas = np.linspace(0.5, 1.5, grid) + r.uniform(-0.02, 0.02, grid)
    j2s = np.linspace(0.03, 0.6, grid) + r.uniform(-0.02, 0.02, grid)
    pairs = [(float(d), float(j)) for d in deltas for j in j2s]
    for n in map(int, case["sizes"].split(",")):
        ge, _, ch = LM.translation_group(LM.Lattice(n))
        basis = q.Basis(_ctx(), q.Group(ge, ch), n // 2, 0)
        tables = [q.Terms(n, LM.term_table(*LM.chain(n, 1.0, d, j))) for d, j in pairs]
        ells = [q.Ell(_ctx(), basis, t, locality_slots=True) for t in tables]
        _, _, found = q.lanczos_batched(ells, max_iter=200, tol=1e-9, reorth=2, want_eigvec=True)
        for (d, j), u in zip(pairs, found):
            net.add_sample(basis, u, d, j)
            vectors.append((n, d, j, u))
    return {"net": net, "vectors": vectors, "theta": net.params()}


# ---- one pass ---------------------------------------------------------------------


def _product(ell, x, y):
    q._check(q.lib().qmb_spmv_device(ell.ctx.h, ell.h, x.data_ptr(), y.data_ptr()))


def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "solve":
        ell = q.Ell(_ctx(), _basis(case, state), state["terms"], locality_slots=case["locality"])
        energies, _, _, vector = q.lanczos(ell, n_eigs=case["n_eigs"], max_iter=case.get("max_iter", 1000 if case["n_eigs"] == 1 else 300),
                                           tol=case["tol"], seed=state["seed"], reorth=case.get("scheme"),
                                           check_every=case.get("check_every", 10), want_eigvec=case["vector"])
        return {"energies": energies, "vector": vector}
    if kind == "assemble":
        basis = _basis(case, state)
        ell = q.Ell(_ctx(), basis, state["terms"], locality_slots=case["locality"])
        _product(ell, state["x"], state["y"])
        return {"rows": basis.n_rows, "entries": int(ell.info().nnz), "y": state["y"]}
    if kind == "apply":
        _product(state["ell"], state["x"], state["y"])
        return {"y": state["y"]}
    if kind == "batched":
        energies, _ = q.lanczos_batched(state["ells"], n_eigs=case["n_eigs"], max_iter=400, tol=case["tol"],
                                        seed=state["seed"], reorth=2)
        return {"energies": energies}
    if kind == "correlations":
        return {"values": np.array([state["basis"].expectation(a, state["x"])[0] for a in state["operators"]])}
    if kind == "train":
        loss, grad = state["net"].loss_grad()
        return {"loss": loss, "gradient": grad}
    x, fallback = state["net"].start_vector(state["basis"], *state["couplings"])
    return {"x": x, "fallback": int(fallback)}


# ---- what a pass cannot do without ------------------------------------------------


def _counts(case):
    """(states of the sector, rows, entries off the diagonal), the last two as averages."""
    n = case["n1"] * case["n2"]
    dim = math.comb(n, case["n_up"])
    rows = dim / (n * (2 if case["parity"] >= 0 else 1) * (4 if case["turn"] >= 0 else 1))
    bonds = n * ((2 if case["n2"] > 1 else 1) + (1 if case["next"] else 0))
    return dim, rows, rows * bonds * 2 * case["n_up"] * (n - case["n_up"]) / (n * (n - 1))


def _is_complex(case):
    return (2 * case["kx"]) % case["n1"] != 0 or (2 * case["ky"]) % case["n2"] != 0


def work(case):
    """The matrix counts at four bytes an entry (column and value index in one word) and a diagonal; a
    product reads it and x once and writes y; a Lanczos step reads three vectors and writes two more. The
    steps of a solve are taken as 2.2 a chain site (42 on a square lattice); a table of the basis takes two
    bits a state. The network is 256 window patterns a coupling, three passes over its layers for a gradient."""
    kind = case["kind"]
    if kind == "batched":
        sectors = [dict(case, n_up=int(u), kx=k) for u in case["sweep"].split(",") for k in range(case["n1"])]
        parts = [_solve_work(dict(c, kind="solve"), built=False) for c in sectors]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if kind == "train":
        sizes = [int(n) for n in case["sizes"].split(",")]
        pairs = case["grid"] ** 2
        rows = sum(math.comb(n, n // 2) / n for n in sizes)
        lookups = sum(math.comb(n, n // 2) for n in sizes)
        return {"bytes": pairs * 8.0 * rows + 9.0 * rows,
                "flops": len(sizes) * pairs * 256 * 3 * 2.0 * (10 * 128 + 128 * 128 + 2 * 128) + pairs * 4.0 * lookups}
    dim, rows, entries = _counts(case)
    s = 16.0 if _is_complex(case) else 8.0
    if kind == "start":
        return {"bytes": 17.0 * rows, "flops": 2.0 * rows * case["n1"] + 256 * 2.0 * (10 * 128 + 128 * 128 + 2 * 128)}
    if kind == "apply":
        return {"bytes": 4 * entries + rows * 3 * s, "flops": 2.0 * (s / 8) ** 2 * (entries + rows)}
    if kind == "assemble":
        return {"bytes": dim / 4 + 2 * 4 * entries + rows * (10 + 4 * s), "flops": 2.0 * (s / 8) ** 2 * (entries + rows)}
    if kind == "correlations":
        return {"bytes": (len(_distances(case["n1"])) + 1) * rows * 17.0,
                "flops": rows * case["n1"] * (10.0 * len(_distances(case["n1"])) + 2.0 * case["n1"])}
    b, f = _solve_work(case)
    return {"bytes": b, "flops": f}


def _solve_work(case, built=True):
    dim, rows, entries = _counts(case)
    s = 16.0 if _is_complex(case) else 8.0
    steps = 42 if case["n2"] > 1 else 2.2 * case["n1"]
    steps = min(steps, rows) * (1 + 0.3 * (case["n_eigs"] - 1))
    step_bytes = 4 * entries + rows * (2 * s + 5 * s)
    once = dim / 4 + 4 * entries + rows * (10 + s) if built else 0.0
    return once + steps * step_bytes, steps * (2.0 * (s / 8) ** 2 * (entries + rows) + 10.0 * rows * s / 8)


# ---- the same in plain 64-bit torch -----------------------------------------------


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _sector_states(n, k):
    """All n-bit integers with k bits set, ascending."""
    level = {0: torch.zeros(1, dtype=torch.int64, device=_dev())}
    for m in range(1, n + 1):
        new = {}
        for j in range(max(0, k - (n - m)), min(m, k) + 1):
            parts = [level[j]] if j in level else []
            if j - 1 in level:
                parts.append(level[j - 1] | (1 << (m - 1)))
            new[j] = torch.cat(parts)
        level = new
    return level[k]


class _Images:
    """The group of a case: for every element the states' images and the character of the irrep."""

    def __init__(self, case):
        n1, n2 = case["n1"], case["n2"]
        self.n, self.elements, self.chi = n1 * n2, [], []
        for turn in range(4 if case["turn"] >= 0 else 1):
            for dx in range(n1):
                for dy in range(n2):
                    move = [0] * self.n
                    for i in range(n1):
                        for j in range(n2):
                            x, y = i, j
                            for _ in range(turn):
                                x, y = (-y) % n1, x
                            move[((x + dx) % n1) * n2 + (y + dy) % n2] = i * n2 + j
                    chi = np.exp(2j * np.pi * (case["kx"] * dx / n1 + case["ky"] * dy / n2 + max(case["turn"], 0) * turn / 4))
                    for flip in range(2 if case["parity"] >= 0 else 1):
                        self.elements.append((move, flip))
                        self.chi.append(-chi if flip and case["parity"] == 1 else chi)
        self.chi = torch.tensor(np.array(self.chi), dtype=torch.complex128, device=_dev())
        self.tables = [self._tables(move) for move, _ in self.elements]

    def _tables(self, move):
        v = torch.arange(1 << 16, dtype=torch.int64, device=_dev())
        out = []
        for low in range(0, self.n, 16):
            t = torch.zeros_like(v)
            for b in range(min(16, self.n - low)):
                t |= ((v >> b) & 1) << move[low + b]
            out.append(t)
        return out

    def image(self, g, states):
        out = self.tables[g][0][states & 0xFFFF]
        for c in range(1, len(self.tables[g])):
            out = out | self.tables[g][c][(states >> (16 * c)) & 0xFFFF]
        return out ^ ((1 << self.n) - 1) if self.elements[g][1] else out

    def representatives(self, states):
        """The orbit minima among the states, and how many elements leave each as it is."""
        kept = []
        for part in states.split(1 << 26):
            for g in range(1, len(self.elements)):
                part = part[self.image(g, part) >= part]
            kept.append(part)
        reps = torch.cat(kept)
        stab = torch.zeros_like(reps)
        total = torch.zeros(len(reps), dtype=torch.complex128, device=reps.device)
        for g in range(len(self.elements)):
            same = self.image(g, reps) == reps
            stab += same
            total += same * self.chi[g]
        fits = total.abs() > 0.5
        return reps[fits], stab[fits]

    def to_minimum(self, states):
        """(minimum of the orbit, character of an element that takes the minimum to the state)."""
        best, which = states.clone(), torch.zeros_like(states)
        for g in range(1, len(self.elements)):
            im = self.image(g, states)
            less = im < best
            best = torch.where(less, im, best)
            which = torch.where(less, torch.full_like(which, g), which)
        return best, self.chi[which].conj()


class _Sector:
    def __init__(self, case):
        self.case, self.group = case, _Images(case)
        self.n = case["n1"] * case["n2"]
        self.reps, self.stab = self.group.representatives(_sector_states(self.n, case["n_up"]))
        self.real = not _is_complex(case)

    def bonds(self, delta, j2):
        n1, n2 = self.case["n1"], self.case["n2"]
        if n2 > 1:
            return [(i * n2 + j, t, 1.0, delta) for i in range(n1) for j in range(n2)
                    for t in (((i + 1) % n1) * n2 + j, i * n2 + (j + 1) % n2)]
        return [(i, (i + d) % n1, jd, jd * delta) for d, jd in ((1, 1.0), (2, j2)) if jd for i in range(n1)]

    def diagonal(self, bonds):
        d = torch.zeros(len(self.reps), dtype=torch.float64, device=self.reps.device)
        for i, j, _, jz in bonds:
            d += jz * (0.25 - 0.5 * (((self.reps >> i) ^ (self.reps >> j)) & 1).double())
        return d

    def entries(self, bonds):
        """For every bond the column and value of the row's entry (value 0 where there is none)."""
        for i, j, jxy, _ in bonds:
            differ = (((self.reps >> i) ^ (self.reps >> j)) & 1) == 1
            low, chi = self.group.to_minimum(torch.where(differ, self.reps ^ ((1 << i) | (1 << j)), self.reps))
            col = torch.searchsorted(self.reps, low).clamp_(max=len(self.reps) - 1)
            there = differ & (self.reps[col] == low)
            val = torch.where(there, jxy / 2 * torch.sqrt(self.stab[col] / self.stab.double()), 0.0)
            yield col, val * chi.real if self.real else val * chi

    def product(self, bonds, x):
        y = self.diagonal(bonds) * x
        for col, val in self.entries(bonds):
            y += val * x[col]
        return y

    def matrix(self, bonds):
        """H as a function of x, its entries kept."""
        diag = self.diagonal(bonds)
        cols, vals = zip(*self.entries(bonds))
        cols, vals = torch.stack(cols), torch.stack(vals)
        return lambda x: diag * x + (vals * x[cols]).sum(0)


def _lowest(matrix, rows, real, k, device):
    """The k lowest eigenvalues that a Krylov space holds and the ground state (Lanczos, every vector kept)."""
    g = torch.Generator(device=device).manual_seed(5)
    w = torch.randn(rows, dtype=torch.float64 if real else torch.complex128, device=device, generator=g)
    most = min(rows, 400)
    vs = torch.zeros(most, rows, dtype=w.dtype, device=device)
    a, b = [], [torch.linalg.vector_norm(w)]
    for m in range(most):
        vs[m] = w / b[-1]
        w = matrix(vs[m])
        a.append(torch.vdot(vs[m], w).real)
        for _ in range(2):
            w = w - vs[: m + 1].T @ (vs[: m + 1].conj() @ w)
        b.append(torch.linalg.vector_norm(w))
        if (m + 1) % 8 == 0 or m + 1 == most or float(b[-1]) < 1e-10:
            off = torch.stack(b[1:-1]).cpu().numpy() if m else np.zeros(0)
            t, z = np.linalg.eigh(np.diag(torch.stack(a).cpu().numpy()) + np.diag(off, 1) + np.diag(off, -1))
            last = float(b[-1]) * np.abs(z[-1, : min(k, m + 1)])
            if m + 1 == most or float(b[-1]) < 1e-10 or (m + 1 > k and last.max() < 1e-9 * max(1.0, abs(t[0]))):
                break
    return t[:k], vs[: m + 1].T @ torch.tensor(z[:, 0], device=device).to(w.dtype)


def _start_stream(seed, n):
    """The seeded start vector: SplitMix64 (Steele, Lea, Flood 2014) as uniform numbers in (0, 1]."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return ((z >> np.uint64(11)) + np.uint64(1)).astype(np.float64) * 2.0 ** -53


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched":
        sectors = [dict(case, n_up=int(u), kx=k) for u in case["sweep"].split(",") for k in range(case["n1"])]
        found = []
        for c in sectors:
            s = _Sector(c)
            found.append(_lowest(s.matrix(s.bonds(*_couplings(case, seed))), len(s.reps), s.real, case["n_eigs"], s.reps.device)[0])
        return {"energies": np.array(found)}
    if kind == "train":
        return _exact_gradient(case, seed)
    dim, rows, entries = _counts(case)
    if dim > 1 << 30:
        return None  # the states of the 6x6 sector alone take 72 GB
    s = _Sector(case)
    if kind == "start":
        return _exact_start(case, seed, s)
    bonds = s.bonds(*_couplings(case, seed))
    if kind in ("apply", "assemble"):
        y = s.product(bonds, _vector(case, seed, len(s.reps), not s.real))
        return {"y": y} if kind == "apply" else {"rows": None, "entries": None, "y": y}
    if kind == "correlations":
        x = torch.tensor(prepare(case, seed)["x"], device=s.reps.device)
        n, found = case["n1"], []
        for r in _distances(n):  # the group's average of S_0 S_r
            ring = [(i, (i + r) % n, 1.0 / n, 1.0 / n) for i in range(n)]
            found.append(torch.vdot(x, s.product(ring, x)))
        up = [((s.reps >> i) & 1).double() - 0.5 for i in range(n)]
        wave = sum(u * complex(math.cos(2 * math.pi * i * (n // 2) / n), math.sin(2 * math.pi * i * (n // 2) / n)) for i, u in enumerate(up))
        found.append((x.abs() ** 2 * wave.abs() ** 2 / n).sum())
        return {"values": torch.stack([v.to(torch.complex128) for v in found])}
    if len(s.reps) * len(bonds) > 1 << 28:
        return None  # a kept matrix of over 4 GB, and several hundred products with it
    energies, v = _lowest(s.matrix(bonds), len(s.reps), s.real, case["n_eigs"], s.reps.device)
    if not case["vector"]:
        return {"energies": energies, "vector": None}
    first = _start_stream(seed, len(s.reps) * (1 if s.real else 2))
    first = torch.tensor(first if s.real else first.view(np.complex128), device=v.device)
    along = torch.vdot(first, v)  # the vector's phase: its product with the start vector is positive
    return {"energies": energies, "vector": v * (along.conj() / along.abs())}


def _network(theta, delta, j2):
    """(log-amplitude, phase) of the 256 patterns of an eight-site window: two tanh layers of 128."""
    at, part = 0, []
    for shape in ((128, 10), (128,), (128, 128), (128,), (2, 128), (2,)):
        size = math.prod(shape)
        part.append(theta[at: at + size].reshape(shape))
        at += size
    p = torch.arange(256, device=theta.device)
    spins = ((p[:, None] >> torch.arange(8, device=theta.device)) & 1) * 2.0 - 1.0
    x = torch.cat([spins.double(), torch.tensor([[delta, j2]], dtype=torch.float64, device=theta.device).expand(256, 2)], 1)
    h = torch.tanh(torch.tanh(x @ part[0].T + part[1]) @ part[2].T + part[3])
    return h @ part[4].T + part[5]


def _amplitudes(theta, s, windows, delta, j2):
    """log-amplitude and phase of every row: the sums over the ring's windows, and the sublattice's sign."""
    out = _network(theta, delta, j2)
    alpha = sum(out[:, 0][w] for w in windows)
    beta = sum(out[:, 1][w] for w in windows)
    even = sum((s.reps >> i) & 1 for i in range(0, s.n, 2))
    return alpha, beta + math.pi * even.double()


def _windows(s):
    ring = s.reps | (s.reps << s.n)
    return [(ring >> i) & 255 for i in range(s.n)]


def _exact_start(case, seed, s):
    theta = torch.tensor(q.Mlp(_ctx(), seed=seed).params(), dtype=torch.float64, device=s.reps.device)
    alpha, beta = _amplitudes(theta, s, _windows(s), *_couplings(case, seed))
    top = int(torch.argmax(alpha))
    size = torch.exp(alpha - alpha[top]) * torch.sqrt(s.case["n1"] / s.stab.double())
    return {"x": size * torch.cos(beta - beta[top]), "fallback": None}


def _exact_gradient(case, seed):
    state = _training_set(case, seed)
    theta = torch.tensor(state["theta"], dtype=torch.float64, device=_dev(), requires_grad=True)
    made, total = {}, 0.0
    for n, delta, j2, u in state["vectors"]:
        if n not in made:
            s = _Sector(_case("", "train", n))
            made[n] = (s, _windows(s))
        s, windows = made[n]
        alpha, beta = _amplitudes(theta, s, windows, delta, j2)
        u = torch.tensor(u, device=s.reps.device)
        c = torch.exp(alpha - alpha.max().detach()) * torch.sqrt(n / s.stab.double())
        overlap = (u * c * torch.cos(beta)).sum() ** 2 + (u * c * torch.sin(beta)).sum() ** 2
        loss = (1 - overlap / ((c * c).sum() * (u * u).sum())) / len(state["vectors"])
        loss.backward()
        total += float(loss)
    return {"loss": total, "gradient": theta.grad}
