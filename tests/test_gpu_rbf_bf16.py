"""GPU checks of the BF16 RBF window products at their tile edges, column by
column, against the FP64 oracle."""
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


# Rounding K and a map (2^-9 each, relative) and the Gram (about 0.3% of K)
# moves each term of a sum by some 4e-3, independently: a column of X (k >= 101
# sums) or a row of Y by about as much of its norm.  Five times that.
BOUND = 2e-2


# Features padded to 32, 64 and 128; 256-point and 256-row blocks and one past
# them; 32-point steps with one, two and many in the last window and a
# remainder; 8, 13 and 2 x 13 map-row tiles; window starts off a multiple of 8;
# the points split over blocks, with windows off a multiple of 4 rows
@pytest.mark.parametrize("n,d,w,rank", [(257, 32, 128, 25), (512, 33, 129, 50), (300, 65, 136, 25), (641, 128, 256, 50),
                                        (513, 64, 168, 60), (1100, 100, 544, 51), (385, 20, 384, 50), (2101, 32, 131, 25)])
def test_rbf_bf16_products_by_column(S, n, d, w, rank):
    print(f"case rbf bf16 columns n={n} d={d} w={w} r={rank}", flush=True)
    rng = np.random.default_rng(n * d)
    X = rng.standard_normal((n, d)) + 2.0 * rng.standard_normal((10, d))[rng.integers(0, 10, n)]
    p = O.AlgParams(matrix_m=n, matrix_n=n, rank=rank, window=w, kernel_func="gaussrbf", kernel_gamma=1.0 / d,
                    sketch_nu=0.9, sketch_eta=1.1)
    osk = O.SketchySVD(p)
    osk.linear_update(X)
    maps = {"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi, "Psi": osk.Psi}
    g = S.SketchySVD(to_gpu_params(p, nfeat=d, precision="bf16"), maps=gpu_maps(maps))
    g.linear_update(dev(X))
    Xg, Yg, _ = (np.asarray(t.cpu()) if hasattr(t, "cpu") else np.asarray(t) for t in g.state())
    ex = np.linalg.norm(Xg - osk.X, axis=0) / np.linalg.norm(osk.X, axis=0)
    ey = np.linalg.norm(Yg - osk.Y, axis=1) / np.linalg.norm(osk.Y, axis=1)
    assert ex.max() <= BOUND, (int(ex.argmax()), ex.max())
    assert ey.max() <= BOUND, (int(ey.argmax()), ey.max())
