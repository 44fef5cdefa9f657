"""Read-backs into ordinary and pinned memory around the sizes where pieces and
threads change: spmv into host arrays against spmv on the device, bit for bit."""
import numpy as np
import pytest
import torch

import qmbcuda_amd as q
import qmbcuda_amd.models as LM


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up,k", [(26, 13, 0),    # 3.2 MB: one transfer
                                      (26, 13, 3),    # 6.4 MB: four pieces, the last one short
                                      (27, 13, 2),    # 11.9 MB: six pieces, two threads with two
                                      (29, 14, 0)])   # 21.4 MB: eleven pieces, slots used again
def test_host_products_equal_device_products(ctx, n, n_up, k):
    print(f"[gpu-case] download n={n} n_up={n_up} k={k}", flush=True)
    lat, info = LM.chain(n, 1.0, 0.7, 0.0)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0)
    e = q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)))
    x = np.random.default_rng(n).normal(size=b.n_rows * (2 if e.is_complex else 1))
    dx = torch.from_numpy(x).cuda()
    dy = torch.empty_like(dx)
    torch.cuda.synchronize()
    q._check(q.lib().qmb_spmv_device(ctx.h, e.h, dx.data_ptr(), dy.data_ptr()))
    y = e.spmv(x.view(np.complex128) if e.is_complex else x).view(np.float64)
    torch.cuda.synchronize()
    assert np.array_equal(y, dy.cpu().numpy())
    # pinned memory, and ordinary memory off a page's start
    pinned = torch.zeros(x.size, dtype=torch.float64, pin_memory=True).numpy()
    odd = np.zeros(x.size + 1)[1:]
    for out in (pinned, odd):
        q._check(q.lib().qmb_spmv_host(ctx.h, e.h, x.ctypes.data, out.ctypes.data))
        assert np.array_equal(out, y)
