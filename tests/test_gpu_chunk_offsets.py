"""Chunk offsets and statistics by one block (at most 1024 chunks) and by three
kernels: matrices c I with rows of 1 to 5 slots, whose extra slots hold zeros."""
import numpy as np
import pytest

import qmbcuda_amd as q


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 64, 65, 8 * 64 + 1, 1024 * 64 - 1, 1024 * 64, 1024 * 64 + 1, 2048 * 64 + 3])
def test_constant_matrix(ctx, n):
    print(f"[gpu-case] chunk offsets n={n}", flush=True)
    W, r = 5, np.random.default_rng(n)
    track = r.integers(1, W + 1, n).astype(np.int16)
    ind = r.integers(0, n, (n, W)).astype(np.uint32)
    ind[:, 0] = np.arange(n)
    val = np.zeros((n, W))
    val[:, 0] = -1.75
    val[np.arange(W)[None, :] >= track[:, None]] = np.nan  # past the row's end: never read
    out = q.eigvals_ref(1, 1, n, W, 11, ind.reshape(-1), val.reshape(-1), track, False)
    energy = out[0] if isinstance(out, tuple) else out
    # one step: E = <x, c x> of a normalised x, a sum of n rounded squares
    assert abs(energy + 1.75) < 1e-12
