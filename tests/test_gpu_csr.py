"""GPU checks of the CSR kernels with dense maps at their tile edges, and of
the window inspection, against the oracle."""
import functools

import numpy as np
import pytest
import scipy.sparse as sp

from oracle import skema_oracle as O
from tests.gpu_helpers import TOL, gpu_maps, to_gpu_params

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import skema_amd

    skema_amd.load()
    return skema_amd


def _matrix(m, n, density, seed):
    A = sp.random(m, n, density=density, format="csr", random_state=seed)
    A.data = np.random.default_rng(seed).standard_normal(A.nnz)
    A.sort_indices()
    return A


# Rows a block (16), map rows a lane (64 to 320: k + s = 9 to 900), entries in
# flight (4) and their remainders, the row-blocked CSC build (256 rows and more)
# and the one with global counters, empty rows and columns.
@pytest.mark.parametrize("m,n,k,s,density,window", [(33, 20, 3, 6, 0.2, 17), (300, 150, 21, 43, 0.03, 260),
                                                    (700, 310, 100, 201, 0.02, 700), (900, 400, 130, 261, 0.05, 300),
                                                    (1000, 700, 299, 601, 0.004, 513)])
def test_csr_dense_maps(S, m, n, k, s, density, window):
    print(f"case csr dense maps {m}x{n} k={k} s={s} w={window}", flush=True)
    A = _matrix(m, n, density, m)
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=2, sketch_range=k, sketch_core=s, window=window, dim_redux="gauss",
                    issparse=True, sketch_nu=0.9, sketch_eta=1.2)
    osk = O.SketchySVD(p)
    osk.linear_update(A)
    maps = gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi, "Psi": osk.Psi})
    Ad = S.CrsMatrix.from_scipy(A)
    whole, parts = S.SketchySVD(to_gpu_params(p), maps=maps), S.SketchySVD(to_gpu_params(p), maps=maps)
    whole.linear_update(Ad)
    for r0 in range(0, m, window):
        parts.update(Ad, (r0, min(m, r0 + window)))
    for g in (whole, parts):
        for a, b in zip(g.state(), (osk.X, osk.Y, osk.Z)):
            assert O.rel_err(a, b) <= TOL


def test_inspection_after_a_bad_window(S):
    """A malformed window is refused before anything indexes with it, and the
    next call on the same context is judged anew."""
    print("case csr inspection", flush=True)
    m, n = 300, 40
    A = _matrix(m, n, 0.1, 5)
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=2, window=m, dim_redux="gauss", issparse=True)
    osk = O.SketchySVD(p)
    osk.linear_update(A)
    g = S.SketchySVD(to_gpu_params(p), maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi,
                                                      "Psi": osk.Psi}))
    good = S.CrsMatrix.from_scipy(A)
    for bad in ("col", "order", "short"):
        B = S.CrsMatrix.from_scipy(A)
        if bad == "col":
            B.col[A.nnz // 2] = n
        elif bad == "order":
            B.rowptr[7] = B.rowptr[8] + 1
        else:  # more entries than the arrays hold
            B.rowptr[-1] = 1 << 40
        with pytest.raises(S.SkemaError):
            g.linear_update(B)
        g.linear_update(good)
        for a, b in zip(g.state(), (osk.X, osk.Y, osk.Z)):
            assert O.rel_err(a, b) <= TOL


# Sparse-sign maps with fewer than 8 entries a column and with 8, columns with
# more nonzeros than a wave (256) or a tile's block (8192) keeps and with one,
# too many columns for 512 tiles, with k + s within a wave's 512 accumulators
# and past them, rows of Psi long enough (64) to be split over blocks with a
# remainder of the 8 loads in flight.
@pytest.mark.parametrize("m,n,k,s,density,window", [(60, 40, 3, 5, 0.1, 60), (900, 130, 21, 43, 0.4, 250),
                                                    (500, 1500, 60, 121, 0.004, 125), (400, 700, 200, 401, 0.02, 400),
                                                    (18100, 7, 9, 19, 0.5, 6000), (300, 14400, 150, 301, 0.003, 100),
                                                    (200, 11000, 200, 401, 0.004, 200)])
@pytest.mark.parametrize("conv", ["cols", "rows"])
def test_csr_sign_maps(S, m, n, k, s, density, window, conv):
    print(f"case csr sign maps {conv} {m}x{n} k={k} s={s} w={window}", flush=True)
    A = _matrix(m, n, density, n)
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=2, sketch_range=k, sketch_core=s, window=window,
                    dim_redux="sparse-sign", issparse=True, sketch_nu=0.9, sketch_eta=1.2)
    osk = O.SketchySVD(p, sparse_convention=conv)
    osk.linear_update(A)
    g = S.SketchySVD(to_gpu_params(p), maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi,
                                                      "Psi": osk.Psi}))
    g.linear_update(S.CrsMatrix.from_scipy(A))
    for a, b in zip(g.state(), (osk.X, osk.Y, osk.Z)):
        assert O.rel_err(a, b) <= TOL


@functools.lru_cache(maxsize=None)
def _shared_matrix(m, density):
    return _matrix(m, m, density, m)


# Map rows up to 16 and 32 (several rows a wave), 64 a block, one part of two to
# five times 64 and two equal parts; windows of a few rows, of a last ragged tile of
# 4, 8 and 16, and long enough for the wider blocks; entries in groups of four.
@pytest.mark.parametrize("k", [1, 16, 17, 32, 33, 64, 129, 320, 321, 390])
@pytest.mark.parametrize("m,rows,density", [(400, 3, 0.05), (1300, 1299, 0.01), (9000, 8501, 0.001)])
def test_csr_rows_times_dense_map(S, m, rows, density, k):
    print(f"case csr rows {rows} of {m} k={k}", flush=True)
    A = _shared_matrix(m, density)
    om = S.GaussDimRedux(m, k, seed=3, dist="normal")
    g = S.SketchySPD(S.AlgParams(matrix_m=m, matrix_n=m, rank=1, sketch_range=k, window=rows, issparse=True), omega=om)
    Ad = S.CrsMatrix.from_scipy(A)
    g.update(Ad, (m - rows, m))
    want = A[m - rows:] @ om.download()
    got = g.state()
    assert O.rel_err(got[m - rows:], want) <= TOL and not got[:m - rows].any()
