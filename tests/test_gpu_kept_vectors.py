"""Eigenvectors combined from the kept Lanczos vectors against the replay of all
steps (the route of a run with a checkpoint file), bit for bit: small sectors in one
workgroup and larger ones, step counts around a block of 16, real and complex."""
import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM


def matrix(ctx, n, n_up, k, j2=0.0):
    lat, info = LM.chain(n, 1.0, 0.8, j2)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0)
    return q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)))


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k,max_iter", [(8, 4, 0, 300),       # 10 rows, the space ends early
                                               (14, 7, 0, 300),      # 246 rows, four wavefronts
                                               (16, 8, 3, 300),      # complex
                                               (18, 9, 0, 300),      # 2,704 rows, four rows a thread
                                               (18, 9, 0, 4000),     # beyond what a small sector keeps: replayed
                                               (20, 10, 0, 300),     # larger, several blocks of 16
                                               (20, 10, 3, 300),
                                               (22, 11, 0, 1000)])
def test_kept_equals_replayed(ctx, tmp_path, n, n_up, k, max_iter):
    print(f"[gpu-case] kept vectors n={n} k={k} max_iter={max_iter}", flush=True)
    e = matrix(ctx, n, n_up, k)
    ev, rep, kr, vec = q.lanczos(e, max_iter=max_iter, tol=1e-13, want_eigvec=True, allow_unconverged=True)
    ev2, rep2, kr2, vec2, _ = q.lanczos_checkpointed(e, tmp_path / "run.ck", every=1000000, max_iter=max_iter,
                                                     tol=1e-13, want_eigvec=True)
    assert rep.iters == rep2.iters and np.array_equal(ev, ev2) and np.array_equal(kr, kr2)
    assert np.array_equal(vec, vec2)
    assert rep.eig_residual == rep2.eig_residual


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 15, 16, 17, 32, 33])
def test_step_counts_around_a_block(ctx, steps):
    """x = sum_n z[n] phi_n from vectors of a host recurrence on the same start."""
    print(f"[gpu-case] kept vectors steps={steps}", flush=True)
    e = matrix(ctx, 20, 10, 0)
    x0 = np.random.default_rng(4).normal(size=e.basis.n_rows)
    ev, rep, z, vec = q.lanczos(e, max_iter=steps, fixed_iter=True, tol=1e-30, start_vec=x0, want_eigvec=True,
                                allow_unconverged=True)
    phi, prev, beta, out = x0 / np.linalg.norm(x0), np.zeros_like(x0), 0.0, np.zeros_like(x0)
    for n in range(steps):
        out += z[n] * phi
        w = e.spmv(phi) - beta * prev
        w -= (w @ phi) * phi
        beta = np.linalg.norm(w)
        prev, phi = phi, w / beta
    # the two recurrences drift apart by rounding, amplified at most some 1e4 times in
    # 33 steps of a random start that is far from converged
    assert np.abs(vec - out).max() < 1e-10
