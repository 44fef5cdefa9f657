"""Allocations that fail inside a call: kept Lanczos vectors that no longer fit, and slots
in page-locked memory that are not to be had. Each case runs in a process of its own
whose hipMalloc or hipHostMalloc fails for chosen sizes (tests/cpp/fail_alloc.cpp)."""
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
w.fail_device.argtypes = w.fail_host.argtypes = [C.c_size_t, C.c_size_t, C.c_int, C.c_int, C.c_int]
EVER = 1 << 30
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
w.fail_device(block, block, 2, OOM, EVER)
E2, r2, kr2 = solve()
assert w.failed_device() >= 1
assert E2 == E and r2 == r and np.array_equal(kr2, kr)
w.fail_device(block, block, 2, UNKNOWN, EVER)
try:
    solve()
    raise SystemExit("the error of an allocation was lost")
except q.QMBError as err:
    assert err.status == 2, err
w.fail_device(1, 0, 0, 0, 0)
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
w.fail_device(block, block, skip, OOM, EVER)
ev, rep, kr, vec = solve()
assert (w.failed_device() > 0) == ({steps} > 16 * skip)
w.fail_device(1, 0, 0, 0, 0)
ev2, rep2, kr2, vec2 = solve()
assert np.array_equal(ev, ev2) and np.array_equal(kr, kr2) and np.array_equal(vec, vec2)
assert rep.eig_residual == rep2.eig_residual
print("done")
""")


@pytest.mark.gpu
def test_read_backs_without_page_locked_slots():
    """Read-backs on both sides of every size rule come back by the runtime's own copy
    while their slots cannot be allocated, and through the slots later."""
    print("[gpu-case] read-backs without slots", flush=True)
    run("""
ctx = q.Context(0)
cases = [matrix(ctx, 18, 9, 0), matrix(ctx, 20, 10, 0), matrix(ctx, 25, 12, 0), matrix(ctx, 25, 12, 4)]
xs = [np.random.default_rng(i).normal(size=e.basis.n_rows * (2 if e.is_complex else 1)) for i, e in enumerate(cases)]
xs = [x.view(np.complex128) if e.is_complex else x for x, e in zip(xs, cases)]
w.fail_host(1 << 20, 1 << 40, 0, OOM, EVER)
got = [e.spmv(x) for e, x in zip(cases, xs)]
vec = q.lanczos(cases[1], want_eigvec=True)[3]
assert w.failed_host() >= 1
w.fail_host(1, 0, 0, 0, 0)
for e, x, y in zip(cases, xs, got):
    assert y.nbytes and np.array_equal(e.spmv(x), y)
assert np.array_equal(q.lanczos(cases[1], want_eigvec=True)[3], vec)
print("done")
""")


@pytest.mark.gpu
def test_uploads_without_page_locked_slots():
    """The tables of a basis and of a matrix reach the device while the slots of the
    uploads cannot be allocated, and through the slots later."""
    print("[gpu-case] uploads without slots", flush=True)
    run("""
want = matrix(q.Context(0), 16, 8, 0).export_reference()
ctx = q.Context(0)
lat, info = LM.chain(16, 1.0, 0.8, 0.0)
ge, _, ch = LM.translation_group(lat)
w.fail_host(1 << 16, 1 << 16, 0, OOM, 1)  # the first request of this size is the slots'
b = q.Basis(ctx, q.Group(ge, np.asarray(ch)[[0]]), 8, 0)
assert w.failed_host() == 1
t = q.Terms(16, LM.term_table(lat, info))
w.fail_host(1 << 16, 1 << 16, 0, OOM, EVER)
e = q.Ell(ctx, b, t)
assert w.failed_host() >= 1
w.fail_host(1, 0, 0, 0, 0)
for m in (e, q.Ell(ctx, b, t)):
    assert all(np.array_equal(a, c) for a, c in zip(m.export_reference(), want))
print("done")
""")


@pytest.mark.gpu
def test_context_after_a_failed_request_for_page_locked_memory():
    """A call that ends because its staging memory cannot grow leaves the context usable."""
    print("[gpu-case] staging memory that cannot grow", flush=True)
    run("""
ctx = q.Context(0)
e = matrix(ctx, 20, 10, 0)  # 9,252 rows: the start vector comes back through 74 KB
net = q.Mlp(ctx)
want, _ = net.start_vector(e.basis, 1.0, 0.0)
c2 = q.Context(0)
e2 = matrix(c2, 20, 10, 0)
net2 = q.Mlp(c2)
w.fail_host((1 << 16) + 1, 1 << 40, 0, OOM, 1)
try:
    net2.start_vector(e2.basis, 1.0, 0.0)
    raise SystemExit("nothing failed")
except q.QMBError as err:
    assert err.status == 3, err
e3 = matrix(c2, 16, 8, 0)
assert np.array_equal(net2.start_vector(e2.basis, 1.0, 0.0)[0], want)
assert all(np.array_equal(a, b) for a, b in zip(e3.export_reference(), matrix(ctx, 16, 8, 0).export_reference()))
print("done")
""")
