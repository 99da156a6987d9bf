"""Host code of the library without a GPU: which kernels a call launches, what
it leaves on its stream, and what it does where device memory runs short.  The
library runs in a process of its own on tests/host_runtime.cpp, whose kernels do
nothing and whose allocations can be limited."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "skema_amd", "libskema_mi355x.so")
pytestmark = pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")

# The binding is loaded by its path: the package would bring torch, and its own
# HIP runtime, into the process.
PRELUDE = r"""
import ctypes as C, importlib.util, os, sys
rt = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
rt.rt_used.restype = C.c_size_t
rt.rt_set_limit.argtypes = [C.c_size_t]
rt.rt_queued.restype, rt.rt_queued.argtypes = C.c_long, [C.c_void_p]
rt.rt_launches.restype = C.c_char_p
rt.rt_inspection.argtypes = [C.c_int64] * 3
spec = importlib.util.spec_from_file_location("binding", os.path.join(sys.argv[2], "skema_amd", "_lib.py"))
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
L.load()
MiB = 1 << 20

def device(count, item=8):
    p = C.c_void_p()
    assert rt.hipMalloc(C.byref(p), C.c_size_t(count * item)) == 0
    return p.value

def context():
    h = C.c_void_p()
    L.call("skema_ctx_create", 0, C.byref(h))
    return h

def dense_map(ctx, rows, cols):
    h = C.c_void_p()
    L.call("skema_map_gauss_seeded", ctx, rows, cols, 1, L.DIST_NORMAL, 0, C.byref(h))
    return h

def sign_map(ctx, rows, cols, zeta=8):
    h = C.c_void_p()
    L.call("skema_map_sparse_sign_seeded", ctx, rows, cols, 1, L.SSIGN_COLS, zeta, 0, C.byref(h))
    return h

def sketch(ctx, m, n, k, s, sign=False, **more):
    p = L.skema_params()
    L.load().skema_params_default(C.byref(p))
    p.m, p.n, p.rank, p.range, p.core, p.window = m, n, 2, k, s, m
    p.dim_redux = L.MAP_SPARSE_SIGN if sign else L.MAP_GAUSS
    for name, value in more.items():
        setattr(p, name, value)
    make = sign_map if sign else dense_map
    maps = [make(ctx, *shape) for shape in ((k, m), (k, n), (s, m), (s, n))]
    h = C.c_void_p()
    L.call("skema_sketch_create", ctx, C.byref(p), *maps, C.byref(h))
    return h

def launched():
    out = [line.rsplit(" ", 3) for line in rt.rt_launches().decode().splitlines()]
    rt.rt_forget()
    return [(name, tuple(map(int, grid))) for name, *grid in out]

def names():
    return [name for name, grid in launched()]

def refused(name, *args):
    try:
        L.call(name, *args)
    except L.SkemaError as e:
        return e.code
    return 0

rt.rt_forget()
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rt") / "libhostrt.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", out,
                    os.path.join(ROOT, "tests", "host_runtime.cpp")], check=True, timeout=120)
    return out


def run(runtime, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, runtime, ROOT], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


def test_refused_window_leaves_nothing_on_the_stream(runtime):
    """A refused window's call returns with its stream empty: the clearing of
    the inspection's flags has no successor that would wait for it, and the next
    call may come on another stream."""
    run(runtime, r"""
ctx = context()
m, n = 300, 40
sk = sketch(ctx, m, n, 9, 19)
rowptr, col, val = device(m + 1), device(1000, 4), device(1000)
stream = C.c_void_p(0x1000)
L.call("skema_ctx_set_stream", ctx, stream)
for flags in (1, 2, 3):
    rt.rt_inspection(0, 1000, flags)
    assert refused("skema_update_csr", sk, rowptr, col, val, 0, m) == 1
    assert rt.rt_queued(stream) == 0, (flags, launched())
rt.rt_inspection(0, 1000, 0)
L.call("skema_update_csr", sk, rowptr, col, val, 0, m)
""")


@pytest.mark.parametrize("transB", ["N", "T"])
@pytest.mark.parametrize("ld", [5000, (1 << 21) + 3, (1 << 25) + 3])
def test_large_products_take_the_wide_kernel_at_any_leading_dimension(runtime, transB, ld):
    """With 32-bit offsets where the operand's slices allow them (rows of the
    operand contiguous: up to 2^25), 64-bit ones past that."""
    run(runtime, rf"""
ctx = context()
M, N, K, ld, tb = 800, 4000, 1000, {ld}, {transB!r}
mp, out = dense_map(ctx, M, K), device(M * N)
rows, cols = (K, N) if tb == "N" else (N, K)
B = device(ld * (cols - 1) + rows)
rt.rt_forget()
L.call("skema_map_lmap", mp, 1.0, B, rows, cols, ld, 0.0, b"N", tb.encode(), 0, 0, out, M)
wide = [n for n in names() if "k_gemm_wide" in n]
far = ld > 1 << (25 if tb == "T" else 21)
assert len(wide) == 1 and ("ELb1EEEv" in wide[0]) == far, wide
""")


@pytest.mark.parametrize("M,N,K,kernel", [
    (694, 454, 32, "k_gemm_ksplitILi8E"),      # few tiles: their K loop's latency
    (1950, 449, 45, "k_gemm_ksplitILi2E"),     # many small ones: their rate
    (1601, 14345, 46, "k_gemm_wideILi1ELi1E"), # bound by its stores
    (100, 3000, 129, "k_gemm_ksplitILi8E"),    # past the short ones
])
def test_products_with_short_k_take_the_kernel_that_measured_fastest(runtime, M, N, K, kernel):
    run(runtime, rf"""
ctx = context()
M, N, K = {M}, {N}, {K}
mp, B, out = dense_map(ctx, M, K), device(K * N), device(M * N)
rt.rt_forget()
L.call("skema_map_lmap", mp, 1.0, B, K, N, K, 0.0, b"N", b"N", 0, 0, out, M)
got = names()
assert len(got) == 1 and {kernel!r} in got[0], got
""")


@pytest.mark.parametrize("rows,k,kernel,grid", [
    (64, 197, "ILi1ELi4ELi64E", (16, 4, 1)),      # too few blocks of 16 rows: 4 rows and 64 map rows a block
    (1000, 304, "ILi1ELi16ELi64E", (63, 5, 1)),   # 64 map rows a block are enough
    (20000, 304, "ILi5ELi16ELi64E", (1250, 1, 1)),
    (20000, 328, "ILi3ELi16ELi64E", (1250, 2, 1)),  # equal parts
    (20000, 9, "ILi1ELi16ELi16E", (1250, 1, 1)),    # four rows a wave
])
def test_csr_row_product_splits(runtime, rows, k, kernel, grid):
    run(runtime, rf"""
ctx = context()
m, rows, k = 30000, {rows}, {k}
p = L.skema_params()
L.load().skema_params_default(C.byref(p))
p.m, p.n, p.rank, p.range, p.window, p.issparse = m, m, 1, k, rows, 1
sp = C.c_void_p()
L.call("skema_spd_create", ctx, C.byref(p), dense_map(ctx, m, k), C.byref(sp))
rowptr, col, val = device(m + 1), device(1000, 4), device(1000)
rt.rt_forget()
L.call("skema_spd_update_csr", sp, rowptr, col, val, 0, rows)
got = [(n, g) for n, g in launched() if "k_csr_right_dense" in n]
assert len(got) == 1 and {kernel!r} in got[0][0] and got[0][1] == {grid!r}, got
""")


@pytest.mark.parametrize("m,k,products", [(5000, 5, False), (5000, 9, True), (300, 8, False), (1000, 5, True),
                                          (100000, 5, True)])
def test_a_few_columns_are_factored_one_by_one(runtime, m, k, products):
    run(runtime, rf"""
ctx = context()
m, k = {m}, {k}
sk = sketch(ctx, m, 200, k, 2 * k + 1)
U, S, V = device(2 * m), device(2), device(2 * 200)
rt.rt_forget()
L.call("skema_low_rank_approx_device", sk, U, m, S, V, 200)
used = [n for n in names() if "k_panel_mul" in n]
assert bool(used) == {products}, used
""")


def test_split_products_stay_within_their_scratch(runtime):
    """Partials of at most 512 MiB, fewer splits where that is not to be had, and
    none at all."""
    run(runtime, r"""
def product(M, N, K, room):
    ctx = context()
    mp, B, out = dense_map(ctx, M, K), device(K * N), device(M * N)
    rt.rt_forget()
    before = rt.rt_used()
    rt.rt_set_limit(before + room)
    L.call("skema_map_lmap", mp, 1.0, B, K, N, K, 0.0, b"N", b"N", 0, 0, out, M)
    rt.rt_set_limit(1 << 60)
    splits = [g[2] for n, g in launched() if "k_gemm_" in n]
    assert len(splits) == 1
    return splits[0], rt.rt_used() - before

splits, kept = product(4096, 1204, 16384, 1 << 60)
assert splits == 8 and kept <= 512 * MiB, (splits, kept)
splits, kept = product(4096, 1204, 16384, 200 * MiB)
assert 1 < splits < 8 and kept <= 200 * MiB, (splits, kept)
assert product(4096, 1204, 16384, 1 * MiB) == (1, 0)
splits, kept = product(66000, 604, 8192, 1 << 60)
assert kept <= 512 * MiB, (splits, kept)
""")


@pytest.mark.parametrize("room_windows,groups", [(1 << 20, [60]), (20, [15, 15, 15, 15]), (1, [])])
def test_grouped_windows_fit_the_memory_there_is(runtime, room_windows, groups):
    """60 windows whose G takes 30 KB each: one group, smaller ones, or the
    windows one by one."""
    run(runtime, rf"""
ctx = context()
m, n, w, k, s = 6000, 300, 100, 21, 43
sk, A = sketch(ctx, m, n, k, s, window=w), device(m * n)
rt.rt_forget()
rt.rt_set_limit(rt.rt_used() + {room_windows} * w * s * 8)
L.call("skema_linear_update_dense", sk, A, m)
got = launched()
series = [g[1] for name, g in got if "k_gemm_ksplit" in name and "Lb1EEEv" in name and g[1] > 1]
assert series == {groups!r}, got
""")


def test_sketch_without_room_for_its_joint_map_records(runtime):
    """The records (32 bytes a row) are an extra: a sketch that fits without them
    is made, and takes the pass that reads the maps' own tables."""
    run(runtime, r"""
ctx = context()
m, n, k, s, nnz = 20000, 400, 9, 19, 5000
rowptr, col, val = device(m + 1), device(nnz, 4), device(nnz)
rt.rt_inspection(0, nnz, 0)

def left_product(sk):
    rt.rt_forget()
    L.call("skema_linear_update_csr", sk, rowptr, col, val)
    return [n for n in names() if "k_left_" in n]

p = L.skema_params()
L.load().skema_params_default(C.byref(p))
p.m, p.n, p.rank, p.range, p.core, p.window, p.dim_redux, p.issparse = m, n, 2, k, s, m, L.MAP_SPARSE_SIGN, 1
maps = [sign_map(ctx, *shape) for shape in ((k, m), (k, n), (s, m), (s, n))]
roomy, tight = C.c_void_p(), C.c_void_p()
before = rt.rt_used()
L.call("skema_sketch_create", ctx, C.byref(p), *maps, C.byref(roomy))
takes = rt.rt_used() - before
rt.rt_set_limit(rt.rt_used() + takes - 32 * m)
L.call("skema_sketch_create", ctx, C.byref(p), *maps, C.byref(tight))
rt.rt_set_limit(1 << 60)
assert len(left_product(roomy)) == 1 and "k_left_tile" in left_product(roomy)[0]
assert len(left_product(tight)) == 1 and "k_left_fx" in left_product(tight)[0]
""")


@pytest.mark.parametrize("m,n,na,taken", [(200000, 20000, 304, True), (1_050_000_000, 512, 15, True),
                                          (1_200_000_000, 512, 15, True), (2_000_000_000, 512, 15, True),
                                          (1_200_000_000, 20000, 304, False), (1000, 100000, 304, False)])
def test_column_tiles_leave_countable_blocks(runtime, m, n, na, taken):
    """A count per tile and 256 rows, 2^31 of them at most: above a billion rows
    fewer and wider tiles, or the other form, which such a matrix always fitted."""
    run(runtime, rf"""
f = L.load()._ZN5skema14left_tile_colsElll
f.restype, f.argtypes = C.c_int64, [C.c_int64] * 3
tc = f({m}, {n}, {na})
assert (tc > 0) == {taken}, tc
if tc > 0:
    assert -(-{n} // tc) * -(-{m} // 256) < 1 << 31, tc
""")


def test_loss_and_gradient_hold_the_maps_once(runtime):
    """[B | OP^T | B] and the maps' copies in three times h n doubles, not four,
    beside Phi, the points and the least K rows."""
    run(runtime, r"""
ctx = context()
n, d, k, s = 20000, 16, 101, 203
h = k + s
maps = [dense_map(ctx, rows, n) for rows in (k, s, s)]
X, dX = device(n * d), device(n * d)
loss, dg = C.c_double(), C.c_double()
rt.rt_set_limit(rt.rt_used() + (3 * h * n + s * n + s * s + 2 * n) * 8 + 40 * MiB)
L.call("skema_rbf_sketch_loss_grad", ctx, X, n, d, n, 0.1, *maps, 4096, L.PREC_FP64, C.byref(loss), dX, n, C.byref(dg))
""")
