"""Element lists in which some elements appear more often than others. They are accepted;
stabiliser sizes count every appearance, so a size need not divide the length of the list
and the sector matrix of a symmetric operator need not be symmetric. Matrix and
expectation values against the plain formulas over all listed elements."""
import numpy as np
import pytest

import qmbcuda_amd as q
from oracle import model as OM

SP, SM, SZ = OM.OP_SP, OM.OP_SM, OM.OP_SZ


def ring_list(n, shifts):
    ge = np.array([[(s + sh) % n for s in range(n)] for sh in shifts], np.uint32)
    return ge, np.ones((1, len(shifts)), np.complex128)


def image(s, p):
    return sum(1 << int(p[i]) for i in range(len(p)) if s >> i & 1)


def act(s, table):
    """(image, coefficient) of every term that acts on s"""
    op, site, sc, n_ops, w = table
    for h in range(len(n_ops)):
        t, c = s, complex(sc[h])
        for k in range(n_ops[h]):
            o, i = op[h * w + k], int(site[h * w + k])
            up = t >> i & 1
            if o == SZ:
                c *= 0.5 if up else -0.5
            elif up == (o == SM):
                t ^= 1 << i
            else:
                break
        else:
            yield t, c


def least(s, ge):
    imgs = [image(s, p) for p in ge]
    return min(imgs), imgs.count(min(imgs))


def row(u, m_src, ge, table, reps):
    """[(row, value)] of the entries that state u gives, trivial characters"""
    out = []
    for t, c in act(u, table):
        if t == u:
            out.append((None, c))
            continue
        rep, mult = least(t, ge)
        out.append((reps.index(rep), c * np.sqrt(mult / m_src)))
    return out


def value(x, ge, table, reps, average):
    total = 0j
    for r, rep in enumerate(reps):
        m_src = sum(image(rep, p) == rep for p in ge)
        us = [image(rep, p) for p in ge] if average else [rep]
        mx = sum(v * x[r if t is None else t] for u in us for t, v in row(u, m_src, ge, table, reps)) / len(us)
        total += x[r] * np.conj(mx)
    return total


@pytest.mark.gpu
def test_matrix_with_a_size_that_does_not_divide(ctx, monkeypatch):
    print("[gpu-case] repeated elements: matrix", flush=True)
    ge, ch = ring_list(4, [0, 1, 2, 3, 2])  # state 0101 is left as it is by 3 of the 5
    table = OM.conjugated_term_table([[(2, SP, 0.7 + 0j), (1, SM, 1 + 0j)], [(0, SZ, 0.3 + 0j), (2, SZ, 1 + 0j)]])
    b = q.Basis(ctx, q.Group(ge, ch), 2, 0)
    reps = [int(v) for v in b.export()[0]]
    assert reps == [3, 5]
    got = []
    for codes in ("1", "0"):
        monkeypatch.setenv("QMB_VALUE_CODES", codes)
        e = q.Ell(ctx, b, q.Terms(4, table), max_terms=4)
        got.append(np.array([e.spmv(np.eye(2)[i]) for i in range(2)]).T)
    want = np.zeros((2, 2))
    for r, rep in enumerate(reps):
        for t, v in row(rep, sum(image(rep, p) == rep for p in ge), ge, table, reps):
            want[r, r if t is None else t] += v.real
    assert np.array_equal(got[0], got[1])
    assert np.abs(got[0] - want).max() < 1e-15


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [q.LAYOUT_COMPACT, q.LAYOUT_REFERENCE])
@pytest.mark.parametrize("n,shifts", [(4, [0, 1, 2, 3, 2]), (8, [0, 1, 2, 3, 4, 5, 6, 7, 4]),
                                      (8, list(range(8)) * 2)])  # the last: every element twice
def test_expectation(ctx, n, shifts, layout):
    print(f"[gpu-case] repeated elements: expectation n={n} G={len(shifts)} layout={layout}", flush=True)
    ge, ch = ring_list(n, shifts)
    b = q.Basis(ctx, q.Group(ge, ch), n // 2, 0, layout)
    reps = [int(v) for v in b.export()[0]]
    bonds = []
    for i in range(n):
        j = (i + 1) % n
        bonds += [[(i, SP, 0.5 + 0j), (j, SM, 1 + 0j)], [(i, SM, 0.5 + 0j), (j, SP, 1 + 0j)],
                  [(i, SZ, 1 + 0j), (j, SZ, 1 + 0j)]]
    r = np.random.default_rng(n)
    x = r.normal(size=len(reps)) + 1j * r.normal(size=len(reps))
    x /= np.linalg.norm(x)
    for terms, average in ((bonds, False), (bonds[:2], True)):
        table = OM.conjugated_term_table(terms)
        v, averaged = b.expectation(q.Terms(n, table), x)
        assert averaged == average
        # at most some 40 terms a row, each within 4 rounding units
        assert abs(v - value(x, ge, table, reps, average)) < 1e-13
