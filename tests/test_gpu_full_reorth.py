"""Full reorthogonalisation with its norms summed by the next launches against a run
that finishes every step by itself (a check after each), bit for bit: one row group,
several, the two sides of the row count where the folding stops, real and complex; and
the basis it keeps orthonormal, by the lowest levels of a run past convergence."""
import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM


def matrix(ctx, n, n_up, k):
    lat, info = LM.chain(n, 1.0, 0.8, 0.0)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0)
    return q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)))


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k", [(12, 6, 0),     # 80 rows: less than a block
                                      (18, 9, 0),     # 2,704 rows
                                      (20, 10, 3),    # complex
                                      (25, 12, 0),    # 208,012 rows: folded
                                      (26, 13, 0)])   # 400,024 rows: finished by its own launches
def test_folded_equals_finished(ctx, n, n_up, k):
    print(f"[gpu-case] full reorthogonalisation n={n} k={k}", flush=True)
    e = matrix(ctx, n, n_up, k)
    runs = [q.lanczos(e, n_eigs=2, max_iter=40, fixed_iter=True, tol=1e-30, reorth=1, check_every=c, want_eigvec=True,
                      allow_unconverged=True) for c in (1, 7, 40)]
    ev, rep, z, vec = runs[0]
    for ev2, rep2, z2, vec2 in runs[1:]:
        assert rep2.iters == rep.iters
        assert np.array_equal(ev, ev2) and np.array_equal(z, z2) and np.array_equal(vec, vec2)


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k", [(12, 6, 0), (14, 7, 3)])
def test_no_copies_of_a_level(ctx, n, n_up, k):
    """70 of at most 246 directions: a basis that loses its orthogonality shows the
    lowest level twice, an orthonormal one gives the dense spectrum's (to rounding: 1e-10
    of levels of some 10)."""
    print(f"[gpu-case] full reorthogonalisation levels n={n} k={k}", flush=True)
    e = matrix(ctx, n, n_up, k)
    rows = e.basis.n_rows
    H = np.stack([e.spmv(c) for c in np.eye(rows, dtype=np.complex128 if e.is_complex else np.float64)], axis=1)
    dense = np.linalg.eigvalsh(H)
    ev, _, _, _ = q.lanczos(e, n_eigs=2, max_iter=70, fixed_iter=True, tol=1e-30, reorth=1, allow_unconverged=True)
    assert np.abs(ev - dense[:2]).max() < 1e-10


# In one workgroup while the kept basis has at most 100,000 numbers, else (and with every
# product timed) by launches.
@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k,steps", [(9, 4, 0, 9),       # 14 rows
                                            (13, 4, 0, 33),     # 55 rows: less than a wavefront
                                            (16, 8, 0, 60),     # 810 rows
                                            (16, 8, 3, 60),     # complex, one row a thread
                                            (17, 8, 3, 60),     # complex, two rows; beyond the limit from step 34
                                            (17, 8, 0, 90)])    # two rows a thread; beyond the limit from step 69
def test_one_workgroup_equals_launches(ctx, tmp_path, n, n_up, k, steps):
    print(f"[gpu-case] full reorthogonalisation in one workgroup n={n} k={k}", flush=True)
    e = matrix(ctx, n, n_up, k)
    opts = dict(n_eigs=2, max_iter=steps, tol=1e-30, reorth=1, want_eigvec=True)
    ev, rep, z, vec = q.lanczos(e, fixed_iter=True, allow_unconverged=True, **opts)
    ev2, rep2, z2, vec2 = q.lanczos(e, fixed_iter=True, profile=True, allow_unconverged=True, **opts)
    assert rep.iters == rep2.iters and rep.n_reorth == rep2.n_reorth
    # the same start and an orthonormal basis on both sides: rounding, amplified by the
    # inverse gaps of levels of some 10 (at most some 1e3)
    assert np.abs(ev - ev2).max() < 1e-11
    assert abs(abs(np.vdot(vec, vec2)) / np.linalg.norm(vec) / np.linalg.norm(vec2) - 1.0) < 1e-10
    assert abs(rep.eig_residual - rep2.eig_residual) < 1e-9
    # windows of other lengths (they may end before `steps`), and a run taken up from a
    # file: the same bits as that many steps in one window
    for c in (1, 7):
        ev3, rep3, _, vec3 = q.lanczos(e, check_every=c, allow_unconverged=True, **opts)
        if c == 7:
            file = tmp_path / "run.ck"
            q.lanczos_checkpointed(e, file, every=1, stop_after=steps // 2, check_every=c, **opts)
            ev4, _, _, vec4, _ = q.lanczos_checkpointed(e, file, resume=True, check_every=c, **opts)
            assert np.array_equal(ev3, ev4) and np.array_equal(vec3, vec4)
        ev5, _, _, vec5 = q.lanczos(e, fixed_iter=True, allow_unconverged=True, **dict(opts, max_iter=rep3.iters))
        assert np.array_equal(ev3, ev5) and np.array_equal(vec3, vec5)
