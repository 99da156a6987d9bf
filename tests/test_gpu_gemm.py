"""GPU checks of the FP64 product behind every dense step, through the Gauss
map's lmap (C = alpha op(map) op(B) + beta C), against numpy: the small kernel
(32 x 32 tiles, K dealt to eight waves) and the wide one (waves along M or N),
tile and slice remainders in every dimension, K split over blocks, odd leading
dimensions and every transposition."""
import numpy as np
import pytest

from tests.gpu_helpers import dev, host

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# One rounding per product and sum: the error of an inner product of length K
# is below K eps times the product of the norms, 5000 * 2.2e-16 = 1.1e-12 here
# at most, and its root-mean-square over a matrix about sqrt(K) eps, 2e-14.
TOL = 1e-12


@pytest.fixture(scope="module")
def S():
    import skema_amd

    skema_amd.load()
    return skema_amd


@pytest.mark.parametrize("tA", ["N", "T"])
@pytest.mark.parametrize("tB", ["N", "T"])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (33, 31, 7), (64, 98, 300), (17, 3000, 129), (401, 4111, 1000),
                                   (4111, 401, 1003), (97, 8300, 640), (8300, 97, 33), (2300, 1204, 15),
                                   (803, 803, 5000), (20, 40, 5000), (6000, 2500, 16), (270, 12000, 500)])
def test_products_of_every_shape(S, tA, tB, M, N, K):
    print(f"case gemm {M}x{N}x{K} {tA}{tB}", flush=True)
    rng = np.random.default_rng(M + N + K)
    D = rng.standard_normal((M, K) if tA == "N" else (K, M))
    B = rng.standard_normal((K, N) if tB == "N" else (N, K))
    C = rng.standard_normal((M, N))
    mp = S.GaussDimRedux(*D.shape, data=D)
    ref = (D if tA == "N" else D.T) @ (B if tB == "N" else B.T)
    for beta in (0.0, -0.5):
        # beta = 0 never reads C: NaN there must not come through
        out = dev(C if beta else np.full((M, N), np.nan))
        mp.lmap(1.5, dev(B), beta, tA, tB, C_out=out)
        want = 1.5 * ref + (beta * C if beta else 0.0)
        err = np.linalg.norm(host(out) - want) / np.linalg.norm(want)
        assert err <= TOL, (beta, err)


@pytest.mark.parametrize("n,d,window", [(300, 1, 300), (1000, 17, 129), (16500, 5, 16500)])
def test_rbf_rows_in_ranges(S, n, d, window):
    """K's rows formed in tiles with row and point remainders and feature
    counts off the slices of 16; at 16500 x 16500 in three ranges of points
    (1 GiB), whose products add up.  Against windows of 128 rows, and the small
    ones against K formed by torch."""
    print(f"case rbf rows n={n} d={d} w={window}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    X = torch.randn((d, n), dtype=torch.float64, device="cuda", generator=g).t()

    def state(w):
        p = S.AlgParams(matrix_m=n, matrix_n=n, rank=5, sketch_range=21, sketch_core=43, window=w,
                        kernel_func="gaussrbf", kernel_gamma=0.5 / d, nfeat=d)
        sk = S.SketchySVD(p, maps=S.make_maps(p, dist="normal"))
        sk.linear_update(X)
        return sk

    whole, parts = state(window), state(128)
    for a, b in zip(whole.state(), parts.state()):
        assert np.linalg.norm(a - b) <= TOL * np.linalg.norm(b)
    if n <= 1000:
        K = np.exp(-0.5 / d * torch.cdist(X.cpu(), X.cpu()).numpy() ** 2)
        om = whole.maps["Omega"].download()
        assert np.linalg.norm(whole.state()[1] - K @ om.T) <= TOL * np.linalg.norm(K @ om.T)


@pytest.mark.parametrize("m,n,w,k,s,nu", [(64, 33, 32, 3, 7, 1.0), (200, 129, 33, 21, 43, 0.7), (1000, 300, 64, 41, 83, 0.0),
                                          (960, 20000, 64, 5, 11, 0.9), (2049, 1000, 100, 41, 83, 1.0)])
def test_grouped_windows_equal_single_ones(S, m, n, w, k, s, nu):
    """linear_update takes small windows in groups of one launch per product:
    two windows, a shorter one after them, more than 128 MiB of rows (two
    groups), and nu = 0, where no output is read.  Bit for bit the windows' own
    updates."""
    print(f"case grouped windows {m}x{n} w={w} nu={nu}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m)
    A = torch.randn((n, m), dtype=torch.float64, device="cuda", generator=g).t()
    p = S.AlgParams(matrix_m=m, matrix_n=n, rank=2, sketch_range=k, sketch_core=s, window=w, sketch_nu=nu,
                    sketch_eta=1.3)
    maps = S.make_maps(p, dist="normal")
    whole, parts = S.SketchySVD(p, maps=maps), S.SketchySVD(p, maps=maps)
    whole.linear_update(A)
    for r0 in range(0, m, w):
        parts.update(A, (r0, min(m, r0 + w)))
    for a, b in zip(whole.state(), parts.state()):
        assert np.array_equal(a, b)


# Operand slices just within 4 GiB (32-bit offsets) and just past it (64-bit):
# 256 rows 2^21 apart where K is contiguous, 16 of K 2^25 apart where the rows are.
@pytest.mark.parametrize("side,trans,M,N,K,ld", [
    ("B", "N", 2000, 300, 1003, 1 << 21), ("B", "N", 2000, 300, 1003, (1 << 21) + 3),
    ("A", "T", 301, 3000, 1003, 1 << 21), ("A", "T", 301, 3000, 1003, (1 << 21) + 3),
    ("A", "N", 401, 3000, 43, 1 << 25), ("A", "N", 4001, 4003, 43, (1 << 25) + 3),
    ("B", "T", 401, 3000, 43, 1 << 25), ("B", "T", 4001, 4003, 43, (1 << 25) + 3)])
def test_leading_dimensions_around_32_bit_slices(S, side, trans, M, N, K, ld):
    print(f"case gemm ld={ld} {side}{trans} {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(K)
    A, B = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    far = A if side == "A" else B
    far = far if trans == "N" else far.T
    rows, cols = far.shape
    buf = torch.empty(ld * (cols - 1) + rows, dtype=torch.float64, device="cuda")
    X = buf.as_strided((rows, cols), (1, ld))
    X.copy_(torch.as_tensor(far, device="cuda"))
    out = dev(np.full((M, N), np.nan))
    if side == "A":
        S.GaussDimRedux(K, N, data=B).rmap(1.0, X, 0.0, trans, "N", C_out=out)
    else:
        S.GaussDimRedux(M, K, data=A).lmap(1.0, X, 0.0, "N", trans, C_out=out)
    want = A @ B
    assert np.linalg.norm(host(out) - want) <= TOL * np.linalg.norm(want)


@pytest.mark.parametrize("K", [1, 15, 16, 17, 32, 33, 65, 127, 128])
@pytest.mark.parametrize("trans", ["NN", "TN", "NT", "TT"])
def test_short_k(S, trans, K):
    """Enough 32 x 32 tiles for the blocks of two waves, whose K loop ends within
    either wave's first chunks, and the wide kernel's large outputs."""
    for M, N in ((1999, 1001), (4111, 3300)):
        print(f"case gemm short K {M}x{N}x{K} {trans}", flush=True)
        rng = np.random.default_rng(M + K)
        A, B = rng.standard_normal((M, K)), rng.standard_normal((K, N))
        mp = S.GaussDimRedux(*(A if trans[0] == "N" else A.T).shape, data=A if trans[0] == "N" else A.T)
        out = dev(np.full((M, N), np.nan))
        mp.lmap(1.0, dev(B if trans[1] == "N" else B.T), 0.0, trans[0], trans[1], C_out=out)
        want = A @ B
        assert np.linalg.norm(host(out) - want) <= TOL * np.linalg.norm(want)
