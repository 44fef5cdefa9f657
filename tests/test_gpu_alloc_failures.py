"""Allocations that fail inside a call: kept Lanczos vectors that no longer fit. Each case
runs in a process of its own whose hipMalloc fails for the blocks' size
(tests/cpp/fail_alloc.cpp)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "cpp", "libfail_alloc.so")

HEAD = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
w = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
w.fail_device.argtypes = w.fail_host.argtypes = [C.c_size_t, C.c_size_t, C.c_int, C.c_int]
import numpy as np
import qmbcuda_amd as q
import qmbcuda_amd.models as LM
OOM, UNKNOWN = 2, 999

def matrix(ctx, n, n_up, k, **kw):
    lat, info = LM.chain(n, 1.0, 0.8, 0.0)
    ge, _, ch = LM.translation_group(lat)
    b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[k]]), n_up, 0)
    return q.Ell(ctx, b, q.Terms(n, LM.term_table(lat, info)), **kw)
"""


def run(body):
    if not os.path.exists(LIB):
        pytest.fail("tests/cpp/libfail_alloc.so is not built (run __graft_entry__.build())")
    out = subprocess.run([sys.executable, "-u", "-c", HEAD.format(root=ROOT, lib=LIB) + body], capture_output=True,
                         text=True, timeout=100)
    print(out.stdout, out.stderr[-2000:], flush=True)
    assert out.returncode == 0 and "done" in out.stdout


@pytest.mark.gpu
def test_reference_call_without_room_for_a_kept_block():
    """The reference-signature call keeps its vectors outside any pool: a block that does
    not fit sends it back to repeating the steps, with the same bits; another error of
    the allocation is the call's error."""
    print("[gpu-case] reference call, third kept block fails", flush=True)
    run("""
ctx = q.Context(0)
e = matrix(ctx, 20, 10, 0)
ind, val, track = e.export_reference()
n, W = e.basis.n_rows, int(e.info().max_terms)
block = 16 * n * 8
solve = lambda: q.eigvals_ref(None, 60, n, W, 5, ind, val, track, False)
E, r, kr = solve()
w.fail_device(block, block, 2, OOM)
E2, r2, kr2 = solve()
assert w.failed_device() >= 1
assert E2 == E and r2 == r and np.array_equal(kr2, kr)
w.fail_device(block, block, 2, UNKNOWN)
try:
    solve()
    raise SystemExit("the error of an allocation was lost")
except q.QMBError as err:
    assert err.status == 2, err
w.fail_device(1, 0, 0, 0)
E3, r3, kr3 = solve()
assert E3 == E and r3 == r
print("done")
""")


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [16, 17, 31, 32, 33, 49])
@pytest.mark.parametrize("k", [0, 3])
def test_vectors_kept_up_to_a_block(k, steps):
    """Runs whose vectors are kept for one block of 16 steps (two for k = 3) and
    repeated beyond, against runs that keep all of them, bit for bit."""
    print(f"[gpu-case] kept up to a block k={k} steps={steps}", flush=True)
    run(f"""
ctx = q.Context(0)
e = matrix(ctx, 20, 10, {k}, keep_fp64_values=True)  # leaves no large block with the context
block = 16 * e.basis.n_rows * 8 * {2 if k else 1}
skip = {2 if k else 1}
x0 = np.random.default_rng(4).normal(size=2 * e.basis.n_rows).view(np.complex128)
x0 = x0 if {k} else x0.real.copy()
solve = lambda: q.lanczos(e, max_iter={steps}, fixed_iter=True, tol=1e-30, start_vec=x0, want_eigvec=True,
                          allow_unconverged=True)
w.fail_device(block, block, skip, OOM)
ev, rep, kr, vec = solve()
assert (w.failed_device() > 0) == ({steps} > 16 * skip)
w.fail_device(1, 0, 0, 0)
ev2, rep2, kr2, vec2 = solve()
assert np.array_equal(ev, ev2) and np.array_equal(kr, kr2) and np.array_equal(vec, vec2)
assert rep.eig_residual == rep2.eig_residual
print("done")
""")
