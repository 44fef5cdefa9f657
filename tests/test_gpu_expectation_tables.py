"""Expectation values by the operator's distinct terms: the group average formed on
the host and by images on the GPU, more terms than the LDS holds, equal and
cancelling terms, states above 32 sites, against the oracle."""
import numpy as np
import pytest

import oracle
import qmbcuda_amd as q
from oracle import model as OM
from tests.helpers import chain_case, oracle_orbits, square_case

SP, SM, SZ = OM.OP_SP, OM.OP_SM, OM.OP_SZ


def operator(n, n_terms, seed):
    """Random hops, density products and products of Sz (also on one site, where they are
    constants), none of them symmetric, the first five repeated and the next three cancelled."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n_terms):
        i, j, k = (int(v) for v in rng.choice(n, 3, replace=False))
        c = complex(rng.normal(), rng.normal()) / np.sqrt(n_terms)
        out.append([[(i, SP, c), (j, SM, 1.0 + 0j)], [(i, SZ, c), (j, SZ, 1.0 + 0j)], [(i, SP, c), (i, SM, 1.0 + 0j)],
                    [(k, SZ, c), (i, SP, 1.0 + 0j), (j, SM, 1.0 + 0j)], [(i, SZ, c), (i, SZ, 1.0 + 0j)]]
                   [int(rng.integers(5))])
    minus = [[(t[0][0], t[0][1], -t[0][2])] + t[1:] for t in out[5:8]]
    return out + out[:5] + minus


CASES = [("few images, few rows", lambda: chain_case(12, 1.0, 1.0, 0.2, flip=True), 6, [0, 13], 12),
         ("many images, few rows: on the GPU", lambda: chain_case(12, 1.0, 1.0, 0.2, flip=True), 6, [0, 13, 5], 220),
         ("many images, many rows", lambda: chain_case(20, 1.0, 1.0, 0.2, flip=True), 10, [3], 150),
         ("torus, many rows", lambda: square_case(4, 5, 1.0, 1.0), 10, [2], 30),
         ("above 32 sites", lambda: chain_case(36, 1.0, 1.0, 0.0), 3, [0, 5], 20)]


@pytest.mark.gpu
@pytest.mark.parametrize("label,mk,n_up,alphas,n_terms", CASES, ids=[c[0] for c in CASES])
def test_tables_match_the_oracle(ctx, label, mk, n_up, alphas, n_terms):
    case = mk()
    n = case["n_sites"]
    orb = oracle_orbits(case, n_up)
    g = q.Group(case["group_el"], case["chars"], case["flip"])
    terms = operator(n, n_terms, 17)
    table = OM.conjugated_term_table(terms)
    t = q.Terms(n, table)
    for a in alphas:
        keep = ~orb.null_mask(a)
        rng = np.random.default_rng(a)
        x = rng.normal(size=orb.n_orb) + 1j * rng.normal(size=orb.n_orb)
        x[~keep] = 0.0
        x /= np.linalg.norm(x)
        print(f"[gpu-case] expectation tables {label} irrep={a}", flush=True)
        want = oracle.expectation(orb, table, a, x)
        for layout in (q.LAYOUT_REFERENCE, q.LAYOUT_COMPACT):
            b = q.Basis(ctx, g, n_up, a, layout)
            got, averaged = b.expectation(t, x if layout == q.LAYOUT_REFERENCE else x[keep])
            assert averaged
            # |A| < 10 (150 terms of size 1/12); sums of some 10^5 products of a unit vector
            assert abs(got - want) < 1e-12 * max(1.0, abs(want))


@pytest.mark.gpu
def test_no_terms_left(ctx):
    """An operator whose terms all cancel, and one that never acts."""
    case = chain_case(10, 1.0, 1.0, 0.0)
    b = q.Basis(ctx, q.Group(case["group_el"], case["chars"], case["flip"]), 5, 0)
    x = np.ones(b.n_rows)
    print("[gpu-case] expectation tables: nothing left", flush=True)
    gone = [[(0, SP, 0.7 + 0j), (3, SM, 1.0 + 0j)], [(0, SP, -0.7 + 0j), (3, SM, 1.0 + 0j)]]
    never = [[(0, SP, 1.0 + 0j), (0, SP, 1.0 + 0j), (1, SM, 1.0 + 0j), (1, SM, 1.0 + 0j)]]
    for op in (gone, never):
        assert b.expectation(q.Terms(10, OM.conjugated_term_table(op)), x)[0] == 0.0


def invariant(case, terms):
    """Whether every image of the terms (equal products summed, the order kept on one site) is the same sum."""
    def summed(perm, flip):
        out = {}
        for t in terms:
            c, ops = 1.0 + 0j, []
            for s, o, f in t:
                c *= f
                if flip:
                    c, o = (-c, o) if o == SZ else (c, SM if o == SP else SP)
                ops.append((int(perm[s]), o))
            key = tuple(sorted(ops, key=lambda p: p[0]))
            out[key] = out.get(key, 0) + c
        return {k: v for k, v in out.items() if abs(v) > 1e-9}
    n = case["n_sites"]
    flip = case["flip"] if case["flip"] is not None else np.zeros(len(case["group_el"]))
    base = summed(np.arange(n), False)
    return all(b.keys() == base.keys() and all(abs(b[k] - base[k]) < 1e-9 for k in b)
               for b in (summed(p, f) for p, f in zip(np.asarray(case["group_el"]), flip)))


@pytest.mark.gpu
@pytest.mark.parametrize("flip", [False, True])
def test_commutation(ctx, flip):
    """`averaged` for sums over the ring of products of 0 to 10 operators, several on one site,
    even and odd numbers of Sz, with one term missing and with a cancelling pair."""
    n = 10
    case = chain_case(n, 1.0, 1.0, 0.0, flip=flip)
    b = q.Basis(ctx, q.Group(case["group_el"], case["chars"], case["flip"]), 5, 0)
    x = np.random.default_rng(1).normal(size=b.n_rows)
    shapes = [[], [(0, SZ)], [(0, SZ), (1, SZ)], [(0, SZ), (0, SZ)], [(0, SP), (0, SM)], [(0, SM), (0, SP), (3, SZ)],
              [(2, SP), (0, SM)], [(3, SZ), (0, SP), (1, SM)], [(i, SZ) for i in range(8)],
              [(i // 2, SZ) for i in range(9)], [(i, (SP, SM)[i % 2]) for i in range(8)] + [(8, SZ), (4, SZ)]]
    for shape in shapes:
        both = [shape, [(s, {SP: SM, SM: SP, SZ: SZ}[o]) for s, o in shape]]
        ring = [[((s + r) % n, o, 1.0 + 0j) for s, o in t] for t in both for r in range(n)]
        extra = [[(0, SP, 0.4 + 0j), (5, SM, 1.0 + 0j)], [(0, SP, -0.4 + 0j), (5, SM, 1.0 + 0j)]]
        for terms in (ring, ring[1:], ring + extra, ring + extra[:1]):
            print(f"[gpu-case] commutation flip={flip} {shape} {len(terms)} terms", flush=True)
            _, averaged = b.expectation(q.Terms(n, OM.conjugated_term_table(terms)), x)
            assert averaged != invariant(case, terms)


def adjoint(t):
    """The product of the adjoint factors in reverse order."""
    return [(s, {SP: SM, SM: SP, SZ: SZ}[o], np.conj(c)) for s, o, c in reversed(t)]


@pytest.mark.gpu
@pytest.mark.parametrize("label,mk,n_up,alphas,n_terms", CASES, ids=[c[0] for c in CASES])
def test_hermitian_operators(ctx, label, mk, n_up, alphas, n_terms):
    """A + A^dagger: only the terms that raise the state are looked up where the average is formed."""
    case = mk()
    n = case["n_sites"]
    orb = oracle_orbits(case, n_up)
    g = q.Group(case["group_el"], case["chars"], case["flip"])
    half = operator(n, n_terms, 23)
    table = OM.conjugated_term_table(half + [adjoint(t) for t in half])
    for a in alphas:
        keep = ~orb.null_mask(a)
        rng = np.random.default_rng(a)
        x = rng.normal(size=orb.n_orb) + 1j * rng.normal(size=orb.n_orb)
        x[~keep] = 0.0
        x /= np.linalg.norm(x)
        print(f"[gpu-case] hermitian {label} irrep={a}", flush=True)
        want = oracle.expectation(orb, table, a, x)
        for layout in (q.LAYOUT_REFERENCE, q.LAYOUT_COMPACT):
            b = q.Basis(ctx, g, n_up, a, layout)
            got, _ = b.expectation(q.Terms(n, table), x if layout == q.LAYOUT_REFERENCE else x[keep])
            # |A| < 20, sums of some 10^5 products of a unit vector
            assert abs(got - want) < 1e-12 * max(1.0, abs(want))
