"""Batches of real and complex sectors in the same launches, and of one kind alone,
under each scheme, rows below, at and above a block's range: against single solves."""
import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM


def sector(ctx, n, n_up, k, fp64=False):
    lat, info = LM.chain(n, 1.0, 0.8, 0.0)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0)
    return q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)), keep_fp64_values=fp64)


BATCHES = {"mixed": [(16, 8, 0), (16, 8, 3), (16, 7, 8), (18, 9, 1), (18, 9, 9), (10, 5, 2), (8, 4, 0)],
           "real": [(16, 8, 0), (18, 9, 0), (8, 4, 0)],
           "complex": [(17, 8, 3), (10, 5, 1)],
           "one": [(18, 8, 5)],
           "larger": [(20, 10, 0), (20, 10, 3), (21, 10, 4)]}


@pytest.mark.gpu
@pytest.mark.parametrize("reorth", [0, 1, 2])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batch_equals_single_solves(ctx, name, reorth):
    print(f"[gpu-case] batched mixed {name} reorth={reorth}", flush=True)
    ells = [sector(ctx, *s, fp64=i == 1) for i, s in enumerate(BATCHES[name])]
    ev, reports = q.lanczos_batched(ells, max_iter=200, tol=1e-13, reorth=reorth)
    assert all(r.converged for r in reports)
    for e, got in zip(ells, np.asarray(ev).reshape(len(ells), -1)):
        want = q.lanczos(e, max_iter=300, tol=1e-13)[0][0]
        # both stop when the error estimate r^2 / gap is below 1e-13 max(1, |E|), |E| < 10
        assert abs(got[0] - want) < 1e-11
