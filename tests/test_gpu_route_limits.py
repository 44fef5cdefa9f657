"""Routes that only certain sizes take: vectors of a small sector that are too many to
keep, four rows a thread in the one-workgroup kernels, and read-backs just below and
above the sizes where their pieces and threads change."""
import math

import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM
from tests.helpers import DeviceBuffer


def matrix(ctx, n, n_up, k):
    lat, info = LM.chain(n, 1.0, 0.8, 0.0)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0)
    return q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)))


def in_one_workgroup(e):
    """The LDS rule of the one-workgroup kernels."""
    i, vs = e.info(), 2 if e.is_complex else 1
    return i.n_rows * vs * 8 + i.stored * 4 <= 140 * 1024 and -(-i.n_rows // 64) <= (32 if vs == 2 else 64)


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k", [(25, 5, 0),   # 2,126 rows: four rows a thread
                                      (18, 7, 1)])  # 1,768 complex rows: two
def test_kept_equals_replayed_in_one_workgroup(ctx, tmp_path, n, n_up, k):
    print(f"[gpu-case] kept in one workgroup n={n} n_up={n_up} k={k}", flush=True)
    e = matrix(ctx, n, n_up, k)
    assert in_one_workgroup(e)
    opts = dict(max_iter=300, tol=1e-13, want_eigvec=True)
    ev, rep, kr, vec = q.lanczos(e, **opts)
    ev2, rep2, kr2, vec2, done = q.lanczos_checkpointed(e, tmp_path / "run.ck", every=1000000, **opts)
    assert done and rep.iters == rep2.iters and np.array_equal(ev, ev2) and np.array_equal(kr, kr2)
    assert np.array_equal(vec, vec2) and rep.eig_residual == rep2.eig_residual


@pytest.mark.gpu
def test_small_sector_with_too_many_vectors_to_keep(ctx):
    """max_iter vectors of 28 KB: 300 are kept, 3,537 (100 MB) are not and the steps are
    repeated. Both runs converge at the same step: the same bits."""
    print("[gpu-case] small sector, vectors not kept", flush=True)
    e = matrix(ctx, 18, 7, 1)
    cnt = 2 * e.basis.n_rows
    assert in_one_workgroup(e) and 300 * cnt * 8 <= 64 << 20 < (cnt + 1) * cnt * 8
    ev, rep, kr, vec = q.lanczos(e, max_iter=300, tol=1e-13, want_eigvec=True)
    ev2, rep2, kr2, vec2 = q.lanczos(e, max_iter=5000, tol=1e-13, want_eigvec=True)
    assert rep.converged and rep.iters == rep2.iters and np.array_equal(ev, ev2)
    assert np.array_equal(kr, kr2) and np.array_equal(vec, vec2) and rep.eig_residual == rep2.eig_residual


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k,steps", [(25, 5, 0, 40),   # within the limit of kept numbers (47 steps)
                                            (25, 5, 0, 60),   # beyond it from step 47
                                            (18, 7, 1, 40)])  # complex, beyond it from step 28
def test_full_reorthogonalisation_in_one_workgroup(ctx, n, n_up, k, steps):
    """Against the launches of a run with every product timed; the bounds are those of the
    smaller sectors: rounding, amplified by the inverse gaps of levels of some 10 (at
    most some 1e3)."""
    print(f"[gpu-case] full reorthogonalisation in one workgroup n={n} k={k} steps={steps}", flush=True)
    e = matrix(ctx, n, n_up, k)
    assert in_one_workgroup(e)
    opts = dict(n_eigs=2, max_iter=steps, tol=1e-30, reorth=1, want_eigvec=True, fixed_iter=True,
                allow_unconverged=True)
    ev, rep, _, vec = q.lanczos(e, **opts)
    ev2, rep2, _, vec2 = q.lanczos(e, profile=True, **opts)
    assert rep.iters == rep2.iters == steps and rep.n_reorth == rep2.n_reorth
    assert np.abs(ev - ev2).max() < 1e-11
    assert abs(abs(np.vdot(vec, vec2)) / np.linalg.norm(vec) / np.linalg.norm(vec2) - 1.0) < 1e-10
    assert abs(rep.eig_residual - rep2.eig_residual) < 1e-9
    # windows of other lengths: the same bits
    for every in (1, 7):
        ev3, _, _, vec3 = q.lanczos(e, check_every=every, **opts)
        assert np.array_equal(ev, ev3) and np.array_equal(vec, vec3)


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up", [(16, 6), (18, 5),    # 64,064 and 68,544 bytes: around 64 KB
                                    (23, 7), (52, 4),    # 1,961,256 and 2,165,800: around 2 MB
                                    (61, 4), (62, 4)])   # 4,174,840 and 4,462,760: around 4 MB
def test_read_backs_around_the_limits(ctx, n, n_up):
    """A product of the whole sector read back into ordinary memory, off a page's start
    too, against the same product left on the device."""
    print(f"[gpu-case] read-back n={n} n_up={n_up}", flush=True)
    lat, info = LM.chain(n, 1.0, 0.8, 0.0)
    b = q.Basis(ctx, q.Group(np.arange(n, dtype=np.uint32)[None], np.ones((1, 1))), n_up, 0)
    assert b.n_rows == math.comb(n, n_up)
    e = q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)))
    x = np.random.default_rng(n).normal(size=b.n_rows)
    dx, dy = DeviceBuffer.from_array(x), DeviceBuffer(x.nbytes)
    q._check(q.lib().qmb_spmv_device(ctx.h, e.h, dx.ptr, dy.ptr))
    ctx.synchronize()
    want = dy.to_array(np.float64, x.size)
    odd = np.zeros(b.n_rows + 1)
    for out in (np.zeros(b.n_rows), odd[1:]):
        q._check(q.lib().qmb_spmv_host(ctx.h, e.h, x.ctypes.data, out.ctypes.data))
        assert np.array_equal(out, want)
    assert odd[0] == 0.0
