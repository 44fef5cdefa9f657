"""The ELL passes that share a row between lanes (few rows) against the oracle,
bit for bit: 16, 8, 4 and 2 lanes a row and one lane, more and fewer candidates
than lanes, more than 64 terms, null orbits (rounds with missing slots), packed
and FP64 values."""
import numpy as np
import pytest

import oracle
import qmbcuda_amd as q
import qmbcuda_amd.models as LM
from oracle import model as OM
from tests.helpers import oracle_ell

# (sites, n_up, J2, flip, irrep): rows decide the lanes per row
CASES = [(8, 1, 0.0, False, 3),      # 1 orbit, null for most irreps
         (10, 5, 0.3, True, 13),     # odd parity: null orbits
         (12, 6, 0.3, False, 0),     # 16 lanes a row
         (16, 8, 0.2, False, 8),     # real, null orbits, 96 terms
         (16, 8, 0.0, False, 3),     # complex
         (20, 10, 0.3, False, 10),   # 9,252 orbits, 120 terms
         (22, 10, 0.0, False, 5),    # 29,414 orbits: 8 lanes
         (23, 11, 0.0, False, 0)]    # 58,786 orbits: 4 lanes


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,j2,flip,a", CASES)
def test_split_rows_match_the_oracle(ctx, n, n_up, j2, flip, a):
    print(f"[gpu-case] ell split n={n} n_up={n_up} irrep={a}", flush=True)
    lat, info = LM.chain(n, 1.0, 0.7, j2)
    ge, fl, ch = LM.translation_group(lat, spin_flip=flip)
    ch = np.asarray(ch)[[a]]
    fl = fl if flip else None
    table = LM.term_table(lat, info)
    orb = oracle.Orbits(n, n_up, ge, ch, flip=fl)
    W = OM.max_terms_rule(len(table[3]), n_up, n) + 4
    ref = oracle_ell({"table": table, "chars": ch}, orb, 0, max_terms=W)
    g, t = q.Group(ge, ch, fl), q.Terms(n, table)
    b = q.Basis(ctx, g, n_up, 0, q.LAYOUT_REFERENCE)
    for keep in (False, True):
        e = q.Ell(ctx, b, t, value_type=q.COMPLEX if ref.is_complex else q.REAL, max_terms=W, keep_fp64_values=keep)
        ind, val, track = e.export_reference()
        assert np.array_equal(track, ref.track)
        assert np.array_equal(ind, ref.ind)
        assert np.array_equal(val.view(np.float64), ref.val)


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k", [(12, 6, 1), (20, 10, 0), (25, 12, 4), (26, 13, 0)])
def test_compact_rows_match_the_oracle(ctx, n, n_up, k):
    """Compact layout: 208,012 rows take one lane, 400,024 too (above the limit of two)."""
    print(f"[gpu-case] ell compact n={n} n_up={n_up} k={k}", flush=True)
    lat, info = LM.chain(n, 1.0, 0.7, 0.0)
    ge, fl, ch = LM.translation_group(lat)
    ch = np.asarray(ch)[[k]]
    table = LM.term_table(lat, info)
    orb = oracle.Orbits(n, n_up, ge, ch)
    ref = oracle_ell({"table": table, "chars": ch}, orb, 0)
    keep = ~orb.null_mask(0)
    b = q.Basis(ctx, q.Group(ge, ch), n_up, 0)
    e = q.Ell(ctx, b, q.Terms(n, table))
    ind, val, track = e.export_reference()
    W = int(e.info().max_terms)
    row_of = np.cumsum(keep) - 1
    assert np.array_equal(track, ref.track[keep])
    ri = ref.ind.reshape(-1, ref.W)[keep][:, :W]
    used = np.arange(W)[None, :] < track[:, None]
    assert np.array_equal(np.where(used, ind.reshape(-1, W), 0), np.where(used, row_of[ri], 0))
    rv = ref.val.view(np.complex128 if ref.is_complex else np.float64).reshape(-1, ref.W)[keep][:, :W]
    assert np.array_equal(np.where(used, val.reshape(-1, W), 0), np.where(used, rv, 0))
