"""The launch shapes of the SpMV (interleaved and XCD-contiguous chunks, and the
16-wavefront blocks of a matrix past the memory-side cache) against the exported
rows: the row sums in slot order, bit for bit, and four Lanczos steps."""
import numpy as np
import pytest
import torch

import qmbcuda_amd as q
import qmbcuda_amd.models as LM

# (n1, n2, J2, flip, irrep, FP64 values)
CASES = [(24, 1, 0.0, True, 0, False),     # interleaved, one pass
         (28, 1, 0.3, True, 0, False),     # interleaved, several passes
         (27, 1, 0.3, False, 3, False),    # contiguous, complex, odd number of sites
         (28, 1, 0.0, False, 5, False),    # contiguous, complex
         (28, 1, 0.0, False, 14, False),   # contiguous, real, null orbits dropped
         (28, 1, 0.3, True, 0, True),      # wide, FP64
         (28, 1, 0.0, False, 5, True),     # wide, FP64 complex
         (30, 1, 0.0, True, 0, False),     # wide, packed
         (4, 7, 0.0, False, 1, False)]     # wide, packed complex


def product(ind, val, track, x):
    """The row sums in slot order, in FP64, one rounding per operation."""
    n = track.numel()
    w = ind.numel() // n
    ind, val = ind.view(n, w), val.view((n, w) + tuple(val.shape[1:]))
    y = torch.zeros_like(x)
    for k in range(w):
        g, v, on = x[ind[:, k].long()], val[:, k], track > k
        if x.dim() == 1:
            y = torch.where(on, y + v * g, y)
        else:
            re = v[:, 0] * g[:, 0] - v[:, 1] * g[:, 1]
            im = v[:, 0] * g[:, 1] + v[:, 1] * g[:, 0]
            y = torch.where(on[:, None], y + torch.stack((re, im), 1), y)
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("n1,n2,j2,flip,a,fp64", CASES)
def test_products_and_steps(ctx, n1, n2, j2, flip, a, fp64):
    print(f"[gpu-case] spmv shape {n1}x{n2} j2={j2} irrep={a} fp64={fp64}", flush=True)
    n = n1 * n2
    lat, info = LM.chain(n, 1.0, 0.7, j2) if n2 == 1 else LM.square(n1, n2, 1.0, 0.7)
    ge, fl, ch = LM.translation_group(lat, spin_flip=flip)
    ch = np.asarray(ch)[[a]]
    g, t = q.Group(ge, ch, fl if flip else None), q.Terms(n, LM.term_table(lat, info))
    b = q.Basis(ctx, g, n // 2, 0)
    e = q.Ell(ctx, b, t, keep_fp64_values=fp64)
    ind, val, track = e.export_reference()
    ind = torch.from_numpy(ind.view(np.int32)).cuda()
    val = torch.from_numpy(val.view(np.float64)).cuda()
    track = torch.from_numpy(track).cuda()
    x = np.random.default_rng(5).normal(size=b.n_rows * (2 if e.is_complex else 1))
    tx = torch.from_numpy(x).cuda()
    if e.is_complex:
        val, tx = val.view(-1, 2), tx.view(-1, 2)
    y = e.spmv(x.view(np.complex128) if e.is_complex else x)
    assert np.array_equal(np.ascontiguousarray(y).view(np.float64),
                          product(ind, val, track, tx).reshape(-1).cpu().numpy())
    # four steps of the recurrence: each a and b is a sum of up to 2.6 million
    # products, accumulated to better than 1e-14 of |H|, and four steps from a random
    # vector lose at most a few digits of that
    ev, _, _, _ = q.lanczos(e, max_iter=4, fixed_iter=True, check_every=4, allow_unconverged=True, tol=1e-30,
                            start_vec=x.view(np.complex128) if e.is_complex else x)
    v0, v1, beta = torch.zeros_like(tx), tx / tx.norm(), 0.0
    al, be = [], []
    for _ in range(4):
        w = product(ind, val, track, v1) - beta * v0
        al.append(float((w * v1).sum()))
        w -= al[-1] * v1
        beta = float(w.norm())
        be.append(beta)
        v0, v1 = v1, w / beta
    low = np.linalg.eigvalsh(np.diag(al) + np.diag(be[:3], 1) + np.diag(be[:3], -1))[0]
    assert abs(ev[0] - low) < 1e-11 * abs(low)
