"""The training step's ring form (four windows per table read) against the form
that takes registered windows one at a time (pinned on the oracle elsewhere), at
ring sizes with every remainder of the windows and samples of a part of a
wavefront step, several steps and several blocks."""
import numpy as np
import pytest


def ring_basis(ctx, n):
    import qmbcuda_amd as q
    from qmbcuda_amd import models as LM

    ge, _, ch = LM.translation_group(LM.Lattice(n))
    return q.Basis(ctx, q.Group(ge, ch), n // 2, 0, q.LAYOUT_COMPACT)


# 8 and 10 sites: too short for the ring form; 22 sites: 32,066 rows, 8 blocks
@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(8,), (10,), (11,), (12,), (13,), (14,), (15,), (19,), (22,), (12, 9, 16, 22)])
def test_ring_form_equals_the_window_form(ctx, sizes):
    """Same windows in another order: the tables, the rows and their fixed-point
    gradients are the same but for the order of a few 64-bit sums, so the loss
    agrees to 1e-12 and the histograms to a unit of 2^-36 per row in 32-bit
    gradients of a relative 1e-5 (32-bit sums of 256 terms: 256 * 2^-24)."""
    import qmbcuda_amd as q

    print(f"[gpu-case] ring windows {sizes}", flush=True)
    rng = np.random.default_rng(sum(sizes))
    bases = [ring_basis(ctx, n) for n in sizes]
    vecs = [rng.normal(size=b.n_rows) for b in bases]
    got = []
    for ordered in (True, False):
        net = q.Mlp(ctx, seed=5)
        net.set_params(net.params() * 2.0)
        for i, (n, b, u) in enumerate(zip(sizes, bases, vecs)):
            if not ordered:
                w = [[(t + k) % n for k in range(8)] for t in reversed(range(n))]
                net.set_windows(b, w, sum(1 << s for s in range(0, n, 2)))
            net.add_sample(b, u, 0.7 + 0.1 * i, 0.3)
        L, g = net.loss_grad()
        assert net.loss_grad(want_grad=False)[0] == L
        x = [net.start_vector(b, 0.9, 0.2)[0] for b in bases]
        got.append((L, g.astype(np.float64), x))
    (L0, g0, x0), (L1, g1, x1) = got
    assert abs(L0 - L1) < 1e-12
    assert np.linalg.norm(g0 - g1) < 1e-5 * np.linalg.norm(g1)
    for a, b in zip(x0, x1):
        assert np.linalg.norm(a - b) < 1e-12 * np.linalg.norm(b)
