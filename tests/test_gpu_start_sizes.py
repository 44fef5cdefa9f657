"""Learned start vector on the two sides of the row count up to which it comes back
with its norms, against its own statement in double precision over the network's
outputs; and the reference phase where all amplitudes are the same."""
import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM
from oracle import mlp as OMLP


def ring(ctx, n):
    lat, _ = LM.chain(n, 1.0, 0.8, 0.3)
    ge, _, ch = LM.translation_group(lat)
    return q.Basis(ctx, q.Group(ge, np.asarray(ch)[[0]]), n // 2, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [3.0, 0.0])  # 0: every alpha is the same, the first row is the reference
@pytest.mark.parametrize("n", [8, 12, 18, 20,  # 10 to 9,252 rows: with the norms
                               22])            # 32,066 rows: by itself
def test_start_vector_states_its_formula(ctx, n, scale):
    print(f"[gpu-case] start vector n={n} scale={scale}", flush=True)
    b = ring(ctx, n)
    net = q.Mlp(ctx, seed=11)
    net.set_params((net.params() * np.float32(scale)).astype(np.float32))
    reps, stab, _ = b.export()
    out = net.forward([0.8], [0.3])[0].astype(np.float64)
    pats = OMLP.window_patterns(reps, n)
    alpha = out[:, 0][pats].sum(1)
    beta = out[:, 1][pats].sum(1) + OMLP.marshall_phase(reps, n)
    i = int(np.argmax(alpha))
    want = np.exp(alpha - alpha[i]) * np.sqrt(n / np.asarray(stab, np.float64)) * np.cos(beta - beta[i])
    x, fallback = net.start_vector(b, 0.8, 0.3)
    assert not fallback
    # sums of at most 22 terms below 10 and a cosine of an angle below 200, all in
    # double precision: some 1e-13 of values of at most 5
    assert np.abs(x - want).max() < 1e-11
