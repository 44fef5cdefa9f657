"""Device memory that handles hold and that calls leave with the context, by the free
memory of the device."""
import ctypes as C
import time

import numpy as np
import pytest

import qmbcuda_amd as q
import qmbcuda_amd.models as LM
from tests.helpers import DeviceBuffer


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert DeviceBuffer.hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def sector(ctx, n, n_up, k, j2=0.0):
    lat, info = LM.chain(n, 1.0, 0.7, j2)
    ge, _, ch = LM.translation_group(lat)
    return q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0), q.Terms(n, LM.term_table(lat, info))


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_up", [(24, 12), (30, 6)])  # half and low filling: 5.5 and 1.2 million slots of room
def test_kept_matrices_hold_what_they_report(n, n_up):
    """Matrices that are kept take the device memory that their info states: the room
    that a small build fills its columns in does not stay with the matrix."""
    print(f"[gpu-case] kept matrices n={n} n_up={n_up}", flush=True)
    c = q.Context(0)
    b, t = sector(c, n, n_up, 1)
    kept = [q.Ell(c, b, t) for _ in range(3)]  # the context's temporary blocks exist
    c.synchronize()
    before = free_bytes()
    more = max(12, 200_000_000 // int(kept[0].info().device_bytes))
    kept += [q.Ell(c, b, t) for _ in range(more)]
    c.synchronize()
    held = before - free_bytes()
    # six arrays a matrix; the pool hands out blocks up to 1/8 larger for the columns and
    # the device rounds each to 4 KB
    limit = more * (int(kept[0].info().device_bytes) * 1.125 + 6 * 4096) + (32 << 20)
    print(f"held {held / 1e6:.1f} MB, limit {limit / 1e6:.1f} MB", flush=True)
    assert held <= limit
    del kept, b, t
    c.close()


@pytest.mark.gpu
def test_kept_lanczos_vectors_are_given_back():
    """A plain run for a vector keeps some 2.6 GB of Lanczos vectors while it runs; at most
    1 GiB of them stays with the context."""
    print("[gpu-case] kept Lanczos vectors given back", flush=True)
    c = q.Context(0)
    b, t = sector(c, 30, 15, 0)
    e = q.Ell(c, b, t)
    steps = 60
    block = 16 * b.n_rows * 8
    assert -(-steps // 16) * block > 2 * (1 << 30)
    run = lambda vec: q.lanczos(e, max_iter=steps, fixed_iter=True, want_eigvec=vec, allow_unconverged=True)
    run(False)
    before = free_bytes()
    run(True)
    for _ in range(50):  # the device clears freed memory before it counts it as free
        held = before - free_bytes()
        if held <= (1 << 30) + (256 << 20):
            break
        time.sleep(0.1)
    print(f"held {held / 1e6:.1f} MB", flush=True)
    assert held <= (1 << 30) + (256 << 20)  # and the vector's own buffers
    del e, b, t
    c.close()
