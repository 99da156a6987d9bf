"""GPU checks of the split-BF16 products whose K is no multiple of 64, on data
that both planes hold exactly."""
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


# One operand holds {-2 .. 2} + {-1, 0, 1} / 512 (a hi and a lo plane), the
# other whole numbers (no lo plane): the dropped lo.lo product is zero and
# every partial sum a multiple of 1 / 512 below 4.01 K <= 2^15, exact in FP32.
# X and Y then equal the oracle's up to its own FP64 sums; Z's right operand
# is rounded to 16 bits (2^-17 relative, well below 2e-5).
#
# K of one and two steps, a remainder of one and of 31, two K splits of which
# the first ends inside a 64-element step; row tiles of 64, 96 and 128 and one
# past them; windows whose last is 8 rows or 1; the long right product's plan.
@pytest.mark.parametrize("lo", ["input", "maps"])
@pytest.mark.parametrize("m,n,w,rank", [(25, 33, 8, 2), (200, 37, 96, 2), (321, 65, 64, 5), (700, 1031, 256, 31),
                                        (520, 4099, 264, 50), (1153, 607, 1152, 10), (2056, 8203, 2048, 20)])
def test_split_bf16_ragged_k(S, m, n, w, rank, lo):
    print(f"case split bf16 {m}x{n} w={w} r={rank} lo={lo}", flush=True)
    rng = np.random.default_rng(m + n)

    def whole(shape):
        return rng.integers(-2, 3, size=shape).astype(np.float64)

    def split(shape):
        return whole(shape) + rng.integers(-1, 2, size=shape) / 512.0

    A = (split if lo == "input" else whole)((m, n))
    p = O.AlgParams(matrix_m=m, matrix_n=n, rank=rank, window=w, sketch_nu=0.5, sketch_eta=1.0)
    maps = O.make_maps(p)
    for mp in maps.values():
        mp.data = (split if lo == "maps" else whole)(mp.data.shape)
    osk = O.SketchySVD(p, maps=maps)
    osk.linear_update(A)
    g = S.SketchySVD(to_gpu_params(p, precision="bf16x3"),
                     maps=gpu_maps({"Upsilon": osk.Upsilon, "Omega": osk.Omega, "Phi": osk.Phi, "Psi": osk.Psi}))
    g.linear_update(dev(A))
    X, Y, Z = g.state()
    ex, ey, ez = np.abs(X - osk.X).max(), np.abs(Y - osk.Y).max(), O.rel_err(Z, osk.Z)
    print(f"max err X {ex:.3e} Y {ey:.3e}, rel err Z {ez:.3e}", flush=True)
    assert ex <= 1e-9 and ey <= 1e-9 and ez <= 2e-5, (ex, ey, ez)
