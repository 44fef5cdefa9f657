"""The matrix build without a wait (small matrices, code classes for every divisor of
the group's order) against the route that collects the values, on both sides of the
size limit, and a row that is too long."""
import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM


def build(ctx, monkeypatch, b, t, codes, **kw):
    monkeypatch.setenv("QMB_VALUE_CODES", "1" if codes else "0")
    return q.Ell(ctx, b, t, **kw)


def same(e, f):
    assert e.info().stored == f.info().stored and e.info().device_bytes == f.info().device_bytes
    for u, v in zip(e.export_reference(), f.export_reference()):
        assert np.array_equal(np.asarray(u), np.asarray(v))


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k,j2,flip", [(2, 1, 0, 0.0, False), (8, 4, 0, 0.3, True), (16, 8, 3, 0.0, False),
                                              (20, 10, 10, 0.3, False), (24, 12, 0, 0.0, True),  # 2.8 million slots of room
                                              (23, 11, 5, 0.3, False),  # 5.5 million, complex
                                              (25, 12, 0, 0.0, False)])  # 10.6 million: with the wait
def test_groups_on_both_sides_of_the_limit(ctx, monkeypatch, n, n_up, k, j2, flip):
    print(f"[gpu-case] open build n={n} k={k}", flush=True)
    lat, info = LM.chain(n, 1.0, 0.7, j2)
    ge, fl, ch = LM.translation_group(lat, spin_flip=flip)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]], fl if flip else None), n_up, 0)
    t = q.Terms(n, LM.term_table(lat, info))
    same(build(ctx, monkeypatch, b, t, True), build(ctx, monkeypatch, b, t, False))


@pytest.mark.gpu
def test_row_too_long(ctx, monkeypatch):
    print("[gpu-case] open build: a row too long", flush=True)
    lat, info = LM.chain(12, 1.0, 0.7, 0.0)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[0]]), 6, 0)
    t = q.Terms(12, LM.term_table(lat, info))
    with pytest.raises(q.QMBError):
        build(ctx, monkeypatch, b, t, True, max_terms=3)
    same(build(ctx, monkeypatch, b, t, True), build(ctx, monkeypatch, b, t, False))
