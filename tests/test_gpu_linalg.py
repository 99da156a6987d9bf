"""GPU checks of the factorisations inside low_rank_approx at the sizes where
their kernels change path, against the oracle's LAPACK."""
import numpy as np
import pytest

from oracle import skema_oracle as O
from tests.gpu_helpers import dev, gpu_maps, to_gpu_params

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import skema_amd

    skema_amd.load()
    return skema_amd


# The core solve multiplies rounding errors (eps ~ 1e-16) by the condition of
# two Gaussian (2k+1) x k factors (about 6 each) and the vectors by the inverse
# of the relative gap, about 1 / 0.035 at the sixth of a 0.7^i spectrum: 1e-12
# with some room for the orders (sqrt(k)) is 1e-10.
TOL = 1e-10


@pytest.mark.parametrize("m,n,k", [(60, 50, 9), (60, 50, 16), (90, 61, 17), (300, 150, 64), (300, 150, 65),
                                   (1500, 600, 130), (1300, 1100, 512), (1300, 1100, 515)])
def test_low_rank_approx_orders(S, m, n, k):
    """Core orders around the 8-column blocks and 64-row waves of the blocked
    Jacobi rounds (9 to 512) and beyond them (515: scalar rounds)."""
    print(f"case low_rank_approx {m}x{n} k={k}", flush=True)
    rng = np.random.default_rng(k)
    A = (rng.standard_normal((m, n)) / np.sqrt(m)) @ np.diag(0.7 ** np.arange(n)) @ rng.standard_normal((n, n))
    A += 1e-4 * rng.standard_normal((m, n))
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=6, sketch_range=k, sketch_core=2 * k + 1, window=m)
    osk = O.SketchySVD(p)
    osk.linear_update(A)
    Ur, Sr, Vr = osk.low_rank_approx()
    g = S.SketchySVD(to_gpu_params(p), maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi,
                                                      "Psi": osk.Psi}))
    g.linear_update(dev(A))
    U, Sv, V = g.low_rank_approx()
    assert np.abs(Sv - Sr).max() <= TOL * Sr[0]
    Ua, Va = O.align_signs(U, V, Ur, Vr)
    assert O.rel_err(Ua, Ur) <= TOL and O.rel_err(Va, Vr) <= TOL
    # every factor of the core's SVD, not the leading six only
    Q, P = g.checkpoint("Q"), g.checkpoint("P")
    sv = g.checkpoint("S")[:, 0]
    assert np.abs(sv - np.linalg.svd(g.checkpoint("C"), compute_uv=False)).max() <= 1e-13 * sv[0] * np.sqrt(k)
    for M in (Q, P):
        assert np.abs(M.T @ M - np.eye(k)).max() <= 1e-12


@pytest.mark.parametrize("m,n,k,decay,true_rank", [
    (2000, 700, 33, 0.9, 700),   # a last panel of one column
    (4100, 1030, 96, 0.9, 700),  # whole panels, a ragged last row tile
    (64, 64, 64, 0.98, 64),      # square factors: the last column has no row below it
    (900, 500, 40, 0.2, 500),    # columns dependent to 1e-16 within the first panel
    (900, 500, 70, 0.8, 6),      # exactly of rank 6, below the range
    (120, 100, 20, 0.9, 0),      # all zero
])
def test_thin_qr_panels(S, m, n, k, decay, true_rank):
    """Panels factored by products, and the matrices they give up on (columns
    too dependent), which are factored column by column: both have LAPACK's
    signs, so Q, P, T1 and T2 compare as they are."""
    print(f"case thin qr {m}x{n} k={k} decay={decay} rank={true_rank}", flush=True)
    rng = np.random.default_rng(m + k)
    A = (rng.standard_normal((m, n)) / np.sqrt(m)) @ np.diag(decay ** np.arange(n) * (np.arange(n) < true_rank))
    A = A @ rng.standard_normal((n, n)) / np.sqrt(n)
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=4, sketch_range=k, sketch_core=2 * k + 1, window=m)
    osk = O.SketchySVD(p)
    osk.linear_update(A)
    Ur, Sr, Vr = osk.low_rank_approx()
    g = S.SketchySVD(to_gpu_params(p), maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi,
                                                      "Psi": osk.Psi}))
    g.linear_update(dev(A))
    U, Sv, V = g.low_rank_approx()
    for name in ("Q", "P"):
        M = g.checkpoint(name)
        assert np.abs(M.T @ M - np.eye(k)).max() <= 1e-13 * np.sqrt(m), name
    if true_rank >= k and decay > 0.5:
        # forward error of a QR: eps (1e-16) times the condition of the k
        # sketched columns, at most about 1e5 here
        for name in ("Q", "P", "T1", "T2"):
            assert O.rel_err(g.checkpoint(name), osk.checkpoints[name]) <= TOL, name
    assert np.abs(Sv - Sr).max() <= TOL * max(Sr[0], 1e-300)
    if true_rank:
        Ua, Va = O.align_signs(U, V, Ur, Vr)
        assert O.rel_err(Ua * Sv, Ur * Sr) <= TOL and O.rel_err(Va * Sv, Vr * Sr) <= TOL


# Few columns: column by column up to 512 rows, above 1024 and up to 32768, by
# products between and beyond; the core's own factors have 2 k + 1 rows.
@pytest.mark.parametrize("k", [2, 5, 8])
@pytest.mark.parametrize("m,n", [(60, 50), (900, 520), (1500, 300), (33000, 40)])
def test_low_rank_approx_of_a_few_columns(S, m, n, k):
    print(f"case low_rank_approx {m}x{n} k={k}", flush=True)
    rng = np.random.default_rng(m + k)
    A = (rng.standard_normal((m, 30)) * 0.5 ** np.arange(30)) @ rng.standard_normal((30, n)) / np.sqrt(m)
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=2, sketch_range=k, sketch_core=2 * k + 1, window=m)
    osk = O.SketchySVD(p)
    osk.linear_update(A)
    Ur, Sr, Vr = osk.low_rank_approx()
    g = S.SketchySVD(to_gpu_params(p), maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi,
                                                      "Psi": osk.Psi}))
    g.linear_update(dev(A))
    U, Sv, V = g.low_rank_approx()
    for name in ("Q", "P", "T1", "T2"):
        assert O.rel_err(g.checkpoint(name), osk.checkpoints[name]) <= TOL, name
    assert np.abs(Sv - Sr).max() <= TOL * Sr[0]


@pytest.mark.parametrize("m,n", [(300, 200), (1500, 64)])
@pytest.mark.parametrize("form", ["triangular", "block", "diagonal"])
def test_thin_qr_of_columns_without_anything_below_the_diagonal(S, m, n, form):
    """dlarfg leaves such a column and its sign alone (tau = 0): Q and P as
    LAPACK's, from a state that holds one (block: the sixteenth column, once the
    fifteen before it are reduced)."""
    print(f"case thin qr {form} {m}x{n}", flush=True)
    k = 40
    rng = np.random.default_rng(m)

    def tall(rows):
        B = 0.1 * rng.standard_normal((rows, k))
        sign = np.where(rng.random(k) < 0.5, -1.0, 1.0)
        B[np.arange(k), np.arange(k)] += sign * (1.0 + rng.random(k))
        if form == "triangular":
            return np.triu(B)
        if form == "diagonal":
            return B * np.eye(rows, k)
        B[16:, :16] = 0.0
        return B

    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=4, sketch_range=k, sketch_core=2 * k + 1, window=m)
    osk = O.SketchySVD(p)
    osk.linear_update(np.zeros((m, n)))
    osk.X, osk.Y, osk.Z = tall(n).T.copy(), tall(m), rng.standard_normal((2 * k + 1, 2 * k + 1))
    osk.low_rank_approx()
    g = S.SketchySVD(to_gpu_params(p), maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi,
                                                      "Psi": osk.Psi}))
    g.set_state(osk.X, osk.Y, osk.Z)
    g.low_rank_approx()
    for name in ("Q", "P", "T1", "T2"):
        assert O.rel_err(g.checkpoint(name), osk.checkpoints[name]) <= TOL, name
