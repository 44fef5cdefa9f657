"""Windows of the plain recurrence in one workgroup (small packed sectors) against
dense diagonalisation and the Krylov relations, at the sizes where the route
changes: one row, a part of a chunk, 16 and 17 chunks, the largest that fit and
the first that do not; real and complex, random and given start vectors, checks
in the middle of a window, breakdown, and stopped runs that resume."""
import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM


def sector(ctx, n, n_up, k=0, flip=False, delta=0.9, j2=0.2, layout=q.LAYOUT_COMPACT):
    lat, info = LM.chain(n, 1.0, delta, j2)
    ge, fl, ch = LM.translation_group(lat, spin_flip=flip)
    b = q.Basis(ctx, q.Group(ge, ch, fl if flip else None), n_up, k, layout)
    return b, q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)))


def dense(ell):
    n, W = ell.basis.n_rows, int(ell.info().max_terms)
    ind, val, track = ell.export_reference()
    H = np.zeros((n, n), val.dtype)
    for s in range(W):
        rows = np.nonzero(track > s)[0]
        np.add.at(H, (rows, ind[rows * W + s]), val[rows * W + s])
    return H


# (sites, n_up, momentum, flip, J2) and rows
CASES = [(8, 0, 0, False, 0.2),    # 1 (not packed)
         (9, 2, 0, False, 0.2),    # 4
         (12, 6, 0, True, 0.2),    # 44
         (12, 5, 1, False, 0.2),   # 66 complex
         (14, 6, 3, False, 0.2),   # 212 complex
         (16, 8, 0, True, 0.2),    # 415
         (16, 8, 0, False, 0.2),   # 810
         (16, 8, 3, False, 0.0),   # 800 complex
         (17, 8, 0, False, 0.0),   # 1430: 23 chunks
         (17, 7, 2, False, 0.0),   # 1144 complex: 18 chunks
         (18, 9, 0, True, 0.0),    # 1367
         (25, 5, 0, False, 0.0),   # 2126: 34 chunks
         (18, 9, 0, False, 0.2)]   # 2704: beyond the LDS, kernel by kernel


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k,flip,j2", CASES)
def test_small_sector_ground_state(ctx, n, n_up, k, flip, j2):
    """The bounds of the single solver's tests: E0 to 1e-10 of the dense one, the
    rebuilt vector's residual and norm, a seeded start equal to the same start given."""
    print(f"[gpu-case] small sector n={n} n_up={n_up} k={k} flip={flip}", flush=True)
    b, e = sector(ctx, n, n_up, k, flip, j2=j2)
    H = dense(e)
    w = np.linalg.eigvalsh(H)
    for every in (10, 3):
        ev, rep, _, x = q.lanczos(e, max_iter=300, tol=1e-13, check_every=every, want_eigvec=True)
        assert rep.converged
        assert abs(ev[0] - w[0]) < 1e-10 * max(1.0, abs(w[0]))
        assert abs(np.linalg.norm(x) - 1.0) < 1e-10
        r = np.linalg.norm(H @ x - ev[0] * x)
        assert r < 2 * np.sqrt(1e-13) * max(1.0, abs(w[0]))
        assert abs(r - rep.eig_residual) < 1e-12
    f = q.Ell(ctx, b, e.terms, keep_fp64_values=True)  # unpacked: the same route, the same bits
    evf, repf, _, xf = q.lanczos(f, max_iter=300, tol=1e-13, check_every=3, want_eigvec=True)
    assert evf[0] == ev[0] and repf.iters == rep.iters and np.array_equal(x, xf)
    rng = np.random.default_rng(3)
    v = rng.normal(size=b.n_rows) + (1j * rng.normal(size=b.n_rows) if e.is_complex else 0.0)
    ev2, rep2, _, _ = q.lanczos(e, max_iter=300, tol=1e-13, start_vec=v)
    assert rep2.converged and abs(ev2[0] - w[0]) < 1e-10 * max(1.0, abs(w[0]))


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k", [(16, 8, 0), (16, 7, 3), (18, 9, 0)])
def test_small_sector_recurrence(ctx, n, n_up, k):
    """Fixed steps: the tridiagonal matrix's lowest eigenvalue and Krylov vector
    are those of a NumPy Lanczos from the same start (12 steps: orthogonality is
    still at rounding, so 1e-12 of the spectrum's size)."""
    print(f"[gpu-case] small recurrence n={n} k={k}", flush=True)
    b, e = sector(ctx, n, n_up, k)
    H = dense(e)
    rng = np.random.default_rng(11)
    v = rng.normal(size=b.n_rows) + (1j * rng.normal(size=b.n_rows) if e.is_complex else 0.0)
    ev, rep, kr, _ = q.lanczos(e, max_iter=12, fixed_iter=True, start_vec=v)
    phi, prev, beta, T = v / np.linalg.norm(v), 0.0, 0.0, np.zeros((12, 12))
    for j in range(12):
        y = H @ phi
        T[j, j] = np.vdot(phi, y).real
        y = y - T[j, j] * phi - beta * prev
        beta = np.linalg.norm(y)
        if j < 11:
            T[j, j + 1] = T[j + 1, j] = beta
        prev, phi = phi, y / beta
    w, Z = np.linalg.eigh(T)
    scale = abs(T).sum(1).max()
    assert abs(ev[0] - w[0]) < 1e-12 * scale
    z = Z[:, 0] * np.sign(Z[0, 0])
    assert np.abs(kr - z).max() < 1e-9


@pytest.mark.gpu
@pytest.mark.parametrize("k", [0, 3])
def test_small_sector_checkpoint_and_breakdown(ctx, tmp_path, k):
    print(f"[gpu-case] small checkpoint k={k}", flush=True)
    b, e = sector(ctx, 16, 8, k)
    ref, rep, _, x = q.lanczos(e, max_iter=200, tol=1e-13, check_every=5, want_eigvec=True)
    path = tmp_path / "c"
    _, _, _, _, done = q.lanczos_checkpointed(e, path, stop_after=10, max_iter=200, tol=1e-13, check_every=5)
    assert not done
    ev, rep2, _, x2, done = q.lanczos_checkpointed(e, path, resume=True, max_iter=200, tol=1e-13, check_every=5,
                                                   want_eigvec=True)
    assert done and ev[0] == ref[0] and rep2.iters == rep.iters and np.array_equal(x, x2)
    ev, rep3, _, _ = q.lanczos(e, max_iter=50, start_vec=np.linalg.eigh(dense(e))[1][:, 0])
    assert rep3.breakdown and abs(ev[0] - ref[0]) < 1e-11 * abs(ref[0])
