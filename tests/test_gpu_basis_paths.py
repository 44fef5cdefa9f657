"""Every route of the basis build against the oracle, at the sizes where the
route or its tiling changes: one kernel with 1 and more states per lane, two
kernels (group test, then one state per lane), last words and groups that are
partly full, few and many words per compaction wavefront; rings, torus products
and both times cosets of point operations, whose ELL rows also take the coset
form of the orbit minimum."""
import sys

import numpy as np
import pytest

import oracle
import qmbcuda_amd as q
import qmbcuda_amd.models as LM
from tests.helpers import oracle_ell
from oracle import model as OM


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


def group_of(lat, flip, point):
    T = LM.translation_group(lat, spin_flip=flip)
    if point is None:
        return T
    P = LM.reflection_group(lat) if point == "P" else LM.rotation_group(lat, point)
    return LM.product_group(T, P)[:3]


# (N1, N2, M, flip, point operation, n_up, irreps)
CASES = [
    (8, 1, 1, True, None, 4, [0, 3, 9]),         # 70 states: one word and a part
    (9, 1, 1, False, None, 1, [0, 4]),           # 9 states, width barely above a window
    (12, 1, 1, False, None, 0, [0, 1]),          # one state
    (20, 1, 1, True, None, 10, [0, 30]),         # 184,756: below the two-kernel limit
    (21, 1, 1, False, None, 10, [0, 7]),         # 352,716: two kernels, periods 7 and 3
    (22, 1, 1, True, None, 11, [0, 33]),
    (23, 1, 1, False, None, 8, [5]),             # prime length
    (20, 1, 1, True, "P", 10, [0, 3]),           # ring times the reflection
    (22, 1, 1, True, "P", 11, [0, 5]),
    (4, 5, 1, False, None, 10, [0, 7]),          # torus product
    (3, 7, 1, False, None, 10, [0, 4]),
    (7, 3, 1, False, None, 9, [2]),
    (4, 6, 1, True, None, 12, [0, 36]),
    (4, 4, 1, True, 4, 8, [0, 2, 5]),            # torus times quarter turns
    (4, 4, 1, True, 2, 8, [1, 6]),
    (3, 3, 1, False, 4, 4, [0, 1, 2, 3]),
    (5, 5, 1, False, 4, 10, [0, 1, 2]),          # 3,268,760: two kernels
    (5, 5, 1, False, 2, 12, [0, 1]),
    (3, 4, 2, False, None, 11, [0, 5]),          # two sites a cell: no cyclic form, runs of 2
]


@pytest.mark.gpu
@pytest.mark.parametrize("n1,n2,m,flip,point,n_up,irreps", CASES)
def test_basis_routes_match_the_oracle(ctx, n1, n2, m, flip, point, n_up, irreps):
    lat = LM.Lattice(n1, n2, m)
    n = lat.n_sites
    ge, fl, ch = group_of(lat, flip, point)
    fl = fl if flip else None
    ch = np.asarray(ch)[irreps]
    orb = oracle.Orbits(n, n_up, ge, ch, flip=fl)
    g = q.Group(ge, ch, fl)
    for a in range(len(irreps)):
        say(f"basis {n1}x{n2}x{m} flip={flip} point={point} n_up={n_up} irrep={irreps[a]}")
        keep = ~orb.null_mask(a)
        for layout in (q.LAYOUT_REFERENCE, q.LAYOUT_COMPACT):
            reps, stab, nul = q.Basis(ctx, g, n_up, a, layout).export()
            sel = np.ones(len(keep), bool) if layout == q.LAYOUT_REFERENCE else keep
            assert np.array_equal(reps, orb.reps[sel])
            assert np.array_equal(stab.astype(np.int32), orb.stab[sel])
            assert np.array_equal(nul.astype(bool), ~keep[sel])


@pytest.mark.gpu
@pytest.mark.parametrize("n1,flip,point,n_up", [(3, False, 4, 4), (4, True, 4, 8), (4, False, 4, 7), (4, True, 2, 8),
                                                (5, False, 4, 6), (5, False, 2, 5)])
def test_torus_cosets_ell_matches_the_oracle(ctx, n1, flip, point, n_up):
    """Translations times turns of an n1 x n1 torus: every irrep's ELL bit for bit."""
    lat, info = LM.square(n1, n1, 1.0, 0.7)
    ge, fl, ch = group_of(lat, flip, point)
    fl = fl if flip else None
    table = LM.term_table(lat, info)
    orb = oracle.Orbits(n1 * n1, n_up, ge, ch, flip=fl)
    g, t = q.Group(ge, ch, fl), q.Terms(n1 * n1, table)
    for a in range(np.asarray(ch).shape[0]):
        say(f"torus cosets {n1}x{n1} flip={flip} point={point} n_up={n_up} irrep={a}")
        ref = oracle_ell({"table": table, "chars": ch}, orb, a,
                         max_terms=OM.max_terms_rule(len(table[3]), n_up, n1 * n1) + 4)
        b = q.Basis(ctx, g, n_up, a, q.LAYOUT_REFERENCE)
        e = q.Ell(ctx, b, t, value_type=q.COMPLEX if ref.is_complex else q.REAL, max_terms=ref.W)
        ind, val, track = e.export_reference()
        assert np.array_equal(track, ref.track)
        assert np.array_equal(ind, ref.ind)
        assert np.array_equal(val.view(np.float64), ref.val)
