"""Timed cases of skema_amd: the calls a user's program makes, at the sizes it makes them.

A case is a dict of plain values.  Its "kind" names the call sequence:

  stream    reset, then update() for every row window of a dense matrix as it arrives
  update    linear_update() of a resident dense matrix (every precision form)
  sketch    linear_update(), low_rank_approx() and compute_residuals(): a whole small job
  finalize  low_rank_approx() of a sketch that holds its state
  csr       linear_update() of a CSR matrix, Gauss or sparse-sign maps
  csrstream reset, then update() for every row window of a CSR matrix
  rbf       linear_update() of the Gaussian RBF matrix of a point set
  adjoint   rbf_sketch_loss_grad(): the loss and its gradients (forward and backward)
  spd       SketchySPD: linear_update() and low_rank_approx() of an RBF or dense PSD matrix

Sketch sizes follow the library's defaults: range k = 4 r + 1, core s = 2 k + 1.
"""
import ctypes
import math
import random

import torch

import skema_amd as S
from skema_amd import _lib as L

F64 = torch.float64


# ---- sizes --------------------------------------------------------------------
def _ks(case):
    k = 4 * case["rank"] + 1
    return k, 2 * k + 1


def listed():
    return [
        # Smallest call: a few-hundred-row matrix streamed window by window (the
        # smoke test's sizes): launch and call latency.
        dict(name="stream-fp64-400x300", kind="stream", m=400, n=300, rank=8, window=64, form="fp64", nu=1.0),
        # Ordinary small job, start to end: the 2000x1000 workload of the benchmark.
        dict(name="sketch-fp64-2000x1000", kind="sketch", m=2000, n=1000, rank=10, window=100, form="fp64", nu=1.0),
        # The benchmark's matrix in the plain form, and its fastest accepted form.
        dict(name="update-fp64-65536x16384", kind="update", m=65536, n=16384, rank=100, window=4096, form="fp64",
             nu=1.0),
        dict(name="update-fp8-65536x16384", kind="update", m=65536, n=16384, rank=100, window=4096, form="fp8",
             nu=1.0),
        # Odd sizes, a last window that is short, and forgetting (nu < 1): windows one by one.
        dict(name="update-bf16x3-30011x5003", kind="update", m=30011, n=5003, rank=50, window=2048, form="bf16x3",
             nu=0.98),
        # The factors of the benchmark's sketch.
        dict(name="finalize-65536x16384", kind="finalize", m=65536, n=16384, rank=100, window=4096, form="fp64",
             nu=1.0),
        # The benchmark's sparse matrix, sparse-sign maps.
        dict(name="csr-sign-200000x20000", kind="csr", m=200000, n=20000, rank=25, window=10000, density=1e-3,
             maps="sparse-sign", nu=1.0),
        # CSR windows as they arrive, Gauss maps, odd sizes.
        dict(name="csrstream-gauss-30007x3001", kind="csrstream", m=30007, n=3001, rank=25, window=4096, density=5e-3,
             maps="gauss", nu=1.0),
        # Kernel matrix, FP64: odd point count, a short last window.
        dict(name="rbf-fp64-20011x64", kind="rbf", m=20011, d=64, rank=50, window=2048, form="fp64"),
        # The benchmark's kernel matrix in its fast form.
        dict(name="rbf-bf16-100000x128", kind="rbf", m=100000, d=128, rank=50, window=2048, form="bf16"),
        # Forward and backward of the kernel sketch's loss.
        dict(name="adjoint-fp64-12288x64", kind="adjoint", m=12288, d=64, rank=50, window=4096, form="fp64"),
        # The route kernel input takes by default: Nystrom sketch and eigenpairs.
        dict(name="spd-rbf-16384x32", kind="spd", m=16384, d=32, rank=20, window=2048, form="fp64"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm, odd or even alike."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["stream", "update", "update", "update", "sketch", "finalize", "csr", "csrstream", "rbf", "rbf",
                       "adjoint", "spd"])
    if kind in ("stream", "update"):
        m, n = _log(rng, 400, 65536), _log(rng, 300, 16384)
        rank = _log(rng, 4, min(100, (min(m, n) - 1) // 4))
        window = _log(rng, 64, 4096) if kind == "update" else max(_log(rng, 64, 4096), m // 40)
        return dict(kind=kind, m=m, n=n, rank=rank, window=min(m, window),
                    form=rng.choice(["fp64", "fp64", "fp32", "bf16x3", "bf16", "fp8"]),
                    nu=rng.choice([1.0, 1.0, 0.98]))
    if kind == "sketch":
        m, n = _log(rng, 400, 10000), _log(rng, 300, 4000)
        return dict(kind=kind, m=m, n=n, rank=_log(rng, 4, 20), window=_log(rng, 64, min(m, 2048)), form="fp64",
                    nu=1.0)
    if kind == "finalize":
        m, n = _log(rng, 800, 65536), _log(rng, 800, 16384)
        return dict(kind=kind, m=m, n=n, rank=_log(rng, 5, 100), window=min(m, 4096), form="fp64", nu=1.0)
    if kind in ("csr", "csrstream"):
        m, n = _log(rng, 1000, 200000), _log(rng, 300, 20000)
        nnz = min(4_000_000, 0.05 * m * n)
        return dict(kind=kind, m=m, n=n, rank=_log(rng, 4, 25), window=max(_log(rng, 500, 10000), m // 30),
                    density=min(0.05, max(1e-3, nnz / (m * n) * rng.uniform(0.05, 1.0))) if m * n < 4e9 else 1e-3,
                    maps=rng.choice(["gauss", "sparse-sign"]), nu=rng.choice([1.0, 0.9]))
    if kind == "rbf":
        form = rng.choice(["fp64", "bf16"])
        m = _log(rng, 500, 25000 if form == "fp64" else 60000)
        return dict(kind=kind, m=m, d=_log(rng, 3, 128), rank=_log(rng, 4, 50), window=_log(rng, 256, 4096), form=form)
    if kind == "adjoint":
        return dict(kind=kind, m=_log(rng, 300, 16384), d=_log(rng, 3, 128), rank=_log(rng, 5, 50),
                    window=_log(rng, 256, 4096), form="fp64")
    return dict(kind=kind, m=_log(rng, 500, 16384), d=_log(rng, 24, 128), rank=_log(rng, 4, 25),
                window=_log(rng, 256, 4096), form="fp64")


# ---- inputs -------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * int(seed) + salt)
    return g


def _cm(rows, cols, g, scale=1.0):
    """Column-major rows x cols N(0, scale^2)."""
    return torch.randn((cols, rows), dtype=F64, device="cuda", generator=g).mul_(scale).t()


def _dense(case, seed):
    """Decaying spectrum plus noise, column-major, built in place."""
    m, n = case["m"], case["n"]
    g = _gen(seed, 1)
    p = min(4 * case["rank"], m, n)
    decay = 0.95 if case["rank"] > 20 else 0.8
    sig = decay ** torch.arange(p, dtype=F64, device="cuda")
    At = _cm(m, n, g, 1e-6).t()
    U = _cm(m, p, g, 1.0 / math.sqrt(m)) * sig
    V = _cm(n, p, g, 1.0 / math.sqrt(n))
    At.addmm_(V, U.t())
    return At.t()


def _points(case, seed):
    """Mixture of ten Gaussians (means N(0, 4 I), unit covariance), single precision widened."""
    g = _gen(seed, 2)
    n, d = case["m"], case["d"]
    means = 2.0 * torch.randn((10, d), dtype=torch.float32, device="cuda", generator=g)
    which = torch.randint(0, 10, (n,), device="cuda", generator=g)
    X = means[which] + torch.randn((n, d), dtype=torch.float32, device="cuda", generator=g)
    return X.t().double().contiguous().t()


def _csr(case, seed):
    """Uniform positions, duplicates merged, N(0, 1) values: (rowptr, col, val) on the GPU."""
    g = _gen(seed, 3)
    m, n = case["m"], case["n"]
    want = max(1, int(case["density"] * m * n))
    key = torch.unique(torch.randint(0, m * n, (want,), dtype=torch.int64, device="cuda", generator=g))
    row = torch.div(key, n, rounding_mode="floor")
    rowptr = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.bincount(row, minlength=m).cumsum(0)
    val = torch.randn(key.numel(), dtype=F64, device="cuda", generator=g)
    return rowptr, (key - row * n).to(torch.int32), val


def _params(case):
    rbf, csr = "d" in case, "density" in case
    return S.AlgParams(matrix_m=case["m"], matrix_n=case["m"] if rbf else case["n"], rank=case["rank"],
                       window=case["window"], sketch_nu=case.get("nu", 1.0),
                       dim_redux="gauss" if case.get("maps", "gauss") == "gauss" else "sparse-sign", issparse=csr,
                       kernel_func="gaussrbf" if rbf else "none", kernel_gamma=_gamma(case) if rbf else 1.0,
                       nfeat=case.get("d", 0), precision=case.get("form", "fp64"))


def _gamma(case):
    return 1.0 / case["d"]


def _dense_map(data, transposed):
    """GaussDimRedux holding a device matrix (column-major), as a program with its own maps makes it."""
    ctx = S.default_context()
    rows, cols = data.shape
    h = ctypes.c_void_p()
    L.call("skema_map_dense_device", ctx.h, rows, cols, data.data_ptr(), rows, int(transposed), ctypes.byref(h))
    m = S.GaussDimRedux.__new__(S.GaussDimRedux)
    super(S.GaussDimRedux, m).__init__(ctx, h, rows, cols, transposed)
    return m


def _gauss_data(p, seed):
    """Stored N(0, 1) matrices of the four maps and whether each is stored transposed."""
    return {name: (_cm(r, c, _gen(seed, 10 + i)), t)
            for i, (name, ((r, c), t)) in enumerate(S.map_shapes(p).items())}


_ZETA = 8


def _sign_data(rows, cols, seed, salt):
    """Logical rows x cols sparse-sign map: per column zeta distinct rows, +-1/sqrt(zeta); (row, col, val)."""
    g = _gen(seed, salt)
    z = min(_ZETA, rows)
    r = torch.rand((cols, rows), device="cuda", generator=g).topk(z, dim=1).indices.reshape(-1)
    c = torch.arange(cols, device="cuda").repeat_interleave(z)
    v = (torch.randint(0, 2, (cols * z,), device="cuda", generator=g) * 2 - 1).double() / math.sqrt(z)
    return r, c, v


def _sign_map(rows, cols, data, transposed):
    r, c, v = data
    if transposed:
        r, c, rows, cols = c, r, cols, rows
    key, order = torch.sort(r * cols + c)
    rp = torch.zeros(rows + 1, dtype=torch.int64)
    rp[1:] = torch.bincount(r, minlength=rows).cumsum(0).cpu()
    return S.SparseSignDimRedux(rows, cols, init_transposed=transposed,
                                csr=(rp.numpy(), (key % cols).to(torch.int32).cpu().numpy(), v[order].cpu().numpy()))


def _logical_shapes(p):
    return {name: ((c, r) if t else (r, c), t) for name, ((r, c), t) in S.map_shapes(p).items()}


def _maps(case, p, seed):
    if p.dim_redux == "gauss":
        return {name: _dense_map(d, t) for name, (d, t) in _gauss_data(p, seed).items()}
    return {name: _sign_map(r, c, _sign_data(r, c, seed, 20 + i), t)
            for i, (name, ((r, c), t)) in enumerate(_logical_shapes(p).items())}


def _input(case, seed):
    if "d" in case:
        return _points(case, seed)
    if "density" in case:
        return S.CrsMatrix(case["m"], case["n"], *_csr(case, seed))
    return _dense(case, seed)


class _Device:
    """A device buffer of the library as seen by torch (the array interface); a
    tensor made from it holds this object, and so the sketch that owns the buffer."""

    def __init__(self, owner, ptr, rows, cols):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(rows, cols), strides=(8, 8 * rows), typestr="<f8",
                                             data=(ptr, False), version=2)


def _state(sk):
    """The sketch's X, Y and Z where they lie in device memory."""
    ptr = [ctypes.c_void_p() for _ in range(3)]
    L.call("skema_state_device", sk.h, *[ctypes.byref(q) for q in ptr])
    shapes = [(sk.range, sk.ncol), (sk.nrow, sk.range), (sk.core, sk.core)]
    return [torch.as_tensor(_Device(sk, q.value, r, c), device="cuda") for q, (r, c) in zip(ptr, shapes)]


def prepare(case, seed):
    p = _params(case)
    A = _input(case, seed)
    if case["kind"] == "adjoint":
        n, (k, s) = case["m"], _ks(case)
        om, ph, ps = (_dense_map(_cm(r, n, _gen(seed, 10 + i)), False) for i, r in enumerate((k, s, s)))
        return dict(case=case, A=A, om=om, ph=ph, ps=ps, gamma=0.5 / case["d"])
    if case["kind"] == "spd":
        k, _ = _ks(case)
        sk = S.SketchySPD(p, omega=_dense_map(_cm(case["m"], k, _gen(seed, 10)), False))
        return dict(case=case, A=A, sk=sk)
    sk = S.SketchySVD(p, maps=_maps(case, p, seed))
    if case["kind"] == "finalize":
        sk.linear_update(A)
        A = None
    return dict(case=case, A=A, sk=sk, state=_state(sk))


def run(state):
    case, A = state["case"], state["A"]
    kind = case["kind"]
    if kind == "adjoint":
        loss, dX, dgamma = S.rbf_sketch_loss_grad(A, state["gamma"], state["om"], state["ph"], state["ps"],
                                                  window=case["window"], precision=case["form"])
        return dict(loss=loss, dX=dX, dgamma=dgamma)
    sk = state["sk"]
    if kind == "spd":
        sk.linear_update(A)
        U, lam = sk.low_rank_approx(device=True)
        return dict(U=U, lam=lam)
    if kind == "finalize":
        U, sv, V = sk.low_rank_approx(device=True)
        return dict(U=U, S=sv, V=V)
    if kind in ("stream", "csrstream"):
        sk.reset()
        m, w = case["m"], case["window"]
        for r0 in range(0, m, w):
            sk.update(A, (r0, min(m, r0 + w)))
    else:
        sk.linear_update(A)
    X, Y, Z = state["state"]
    if kind == "sketch":
        U, sv, V = sk.low_rank_approx(device=True)
        return dict(X=X, Y=Y, Z=Z, U=U, S=sv, V=V, rnrms=sk.compute_residuals(A, U, sv, V))
    return dict(X=X, Y=Y, Z=Z)


# ---- what a pass cannot do without ---------------------------------------------
def work(case):
    k, s = _ks(case)
    m, kind = case["m"], case["kind"]
    n = case.get("n", m)
    state = 8.0 * (k * n + m * k + s * s)
    factor = 8.0 * ((k + s) * (m + n))
    fin = 4.0 * (m + n) * k * k + 2.0 * s * k * (m + n) + 16.0 * s * k * k + 20.0 * k ** 3 \
        + 2.0 * case["rank"] * k * (m + n)
    fin_bytes = state + 8.0 * s * (m + n) + 8.0 * case["rank"] * (m + n)
    if "d" in case:
        d = case["d"]
        gram = 2.0 * m * m * d
        if kind == "adjoint":
            return dict(bytes=8.0 * m * (2 * d + k + 2 * s), flops=3 * gram + m * m * (2.0 * (k + s) + 4.0 * (k + s)))
        if kind == "spd":
            return dict(bytes=8.0 * m * (d + 4 * k), flops=gram + 2.0 * m * m * k + 10.0 * m * k * k + 40.0 * k ** 3)
        return dict(bytes=8.0 * m * d + factor + state, flops=gram + 2.0 * m * m * (2 * k + s) + 2.0 * s * s * m)
    if "density" in case:
        nnz = case["density"] * m * n
        per = 2 * k + s if case["maps"] == "gauss" else 2 * _ZETA + 2 * _ZETA
        maps = factor if case["maps"] == "gauss" else 4.0 * _ZETA * 2 * (m + n)
        return dict(bytes=12.0 * nnz + 8.0 * m + maps + state, flops=2.0 * nnz * per + (
            2.0 * s * s * m if case["maps"] == "gauss" else 2.0 * _ZETA * s * n))
    if kind == "finalize":
        return dict(bytes=fin_bytes, flops=fin)
    flops = 2.0 * m * n * (2 * k + s) + 2.0 * s * s * m
    bytes_ = 8.0 * m * n + factor + state
    if kind == "sketch":
        flops += fin + 4.0 * m * n * case["rank"]
        bytes_ += fin_bytes
    return dict(bytes=bytes_, flops=flops)


# ---- the same in 64 bits with torch alone ----------------------------------------
def _logical(case, p, seed):
    if p.dim_redux == "gauss":
        return {name: (d.t() if t else d) for name, (d, t) in _gauss_data(p, seed).items()}
    out = {}
    for i, (name, ((r, c), _)) in enumerate(_logical_shapes(p).items()):
        row, col, v = _sign_data(r, c, seed, 20 + i)
        M = torch.zeros((c, r), dtype=F64, device="cuda")
        M[col, row] = v
        out[name] = M.t()
    return out


def _rows(case, A, r0, r1):
    """Rows [r0, r1) of the input as a dense matrix."""
    if "d" in case:
        sq = (A * A).sum(1)
        D = (sq[r0:r1, None] + sq[None, :]).addmm_(A[r0:r1], A.t(), alpha=-2.0)
        K = D.clamp_(min=0.0).mul_(-_gamma(case)).exp_()
        K[torch.arange(r1 - r0, device="cuda"), torch.arange(r0, r1, device="cuda")] = 1.0
        return K
    if "density" in case:
        rp, ci, v = A
        e0, e1 = int(rp[r0]), int(rp[r1])
        H = torch.zeros((r1 - r0, case["n"]), dtype=F64, device="cuda")
        row = torch.repeat_interleave(torch.arange(r1 - r0, device="cuda"), rp[r0 + 1:r1 + 1] - rp[r0:r1])
        H[row, ci[e0:e1].long()] = v[e0:e1]
        return H
    return A[r0:r1]


def _exact_state(case, seed):
    p = _params(case)
    A = _csr(case, seed) if "density" in case else _input(case, seed)
    maps = _logical(case, p, seed)
    m, w, (k, s) = case["m"], min(case["window"], case["m"]), _ks(case)
    n = case.get("n", m)
    X = torch.zeros((k, n), dtype=F64, device="cuda")
    Y = torch.zeros((m, k), dtype=F64, device="cuda")
    Z = torch.zeros((s, s), dtype=F64, device="cuda")
    nu = case.get("nu", 1.0)
    step = w if nu != 1.0 else max(256, min(m, 400_000_000 // n))
    for r0 in range(0, m, step):
        r1 = min(m, r0 + step)
        H = _rows(case, A, r0, r1)
        X.mul_(nu).addmm_(maps["Upsilon"][:, r0:r1], H)
        Y[r0:r1] = H @ maps["Omega"].t()
        Z.mul_(nu).addmm_(maps["Phi"][:, r0:r1], H @ maps["Psi"].t())
        del H
    return A, maps, X, Y, Z


def _exact_values(maps, X, Y, Z):
    """Singular values of the core of the three-sketch approximation, with LAPACK."""
    P = torch.linalg.qr(X.t().cpu())[0]
    Q = torch.linalg.qr(Y.cpu())[0]
    U1, T1 = torch.linalg.qr(maps["Phi"].cpu() @ Q)
    U2, T2 = torch.linalg.qr(maps["Psi"].cpu() @ P)
    C = torch.linalg.solve_triangular(T1, U1.t() @ Z.cpu() @ U2, upper=True)
    C = torch.linalg.solve_triangular(T2, C.t().contiguous(), upper=True).t()
    return torch.linalg.svdvals(C.contiguous())


def exact(case, seed):
    kind, rank = case["kind"], case["rank"]
    k, s = _ks(case)
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    if kind == "spd":
        A = _points(case, seed)
        n = case["m"]
        Om = _cm(n, k, _gen(seed, 10))
        Y = torch.empty((n, k), dtype=F64, device="cuda")
        for r0 in range(0, n, 4096):
            Y[r0:r0 + 4096] = _rows(case, A, r0, min(n, r0 + 4096)) @ Om
        Y, Om = Y.cpu(), Om.cpu()
        shift = torch.finfo(F64).eps * float(torch.linalg.matrix_norm(Y, 2))
        B = Om.t() @ (Y + shift * Om)
        R = torch.linalg.cholesky(0.5 * (B + B.t()), upper=True)
        E = torch.linalg.solve_triangular(R, Y, upper=True, left=False)
        lam = (torch.linalg.svdvals(E)[:rank] ** 2 - shift).clamp(min=0.0)
        return dict(U=None, lam=lam)  # eigenvectors: each up to its sign
    A, maps, X, Y, Z = _exact_state(case, seed)
    if kind in ("finalize", "sketch"):
        sv = _exact_values(maps, X, Y, Z)[:rank]
        if kind == "finalize":
            return dict(U=None, S=sv, V=None)  # singular vectors: each pair up to its sign
        return dict(X=X, Y=Y, Z=Z, U=None, S=sv, V=None, rnrms=None)
    return dict(X=X, Y=Y, Z=Z)


def _exact_adjoint(case, seed):
    """Loss, dL/dX and dL/dgamma from their closed forms, rows of K at a time."""
    X = _points(case, seed)
    n, (k, s), gamma = case["m"], _ks(case), 0.5 / case["d"]
    Om, Ph, Ps = (_cm(r, n, _gen(seed, 10 + i)) for i, r in enumerate((k, s, s)))
    OP = torch.cat([Om, Ps])
    sq = (X * X).sum(1)
    step = max(256, min(n, 200_000_000 // n))

    def rows(r0, r1):
        D = (sq[r0:r1, None] + sq[None, :]).addmm_(X[r0:r1], X.t(), alpha=-2.0).clamp_(min=0.0)
        D[torch.arange(r1 - r0, device="cuda"), torch.arange(r0, r1, device="cuda")] = 0.0
        return D, torch.exp(-gamma * D)

    YG = torch.empty((n, k + s), dtype=F64, device="cuda")
    for r0 in range(0, n, step):
        r1 = min(n, r0 + step)
        YG[r0:r1] = rows(r0, r1)[1] @ OP.t()
    W = Ph @ YG[:, k:]
    loss = float((YG[:, :k] ** 2).sum() + (W ** 2).sum())
    B = torch.cat([YG[:, :k], Ph.t() @ W], dim=1)  # dL/dK = 2 B OP
    dX = torch.empty((n, case["d"]), dtype=F64, device="cuda")
    dgamma = 0.0
    for r0 in range(0, n, step):
        r1 = min(n, r0 + step)
        D, K = rows(r0, r1)
        H = (B[r0:r1] @ OP).addmm_(OP[:, r0:r1].t(), B.t()).mul_(2.0).mul_(K)  # (G + G^T) o K
        dX[r0:r1] = -2.0 * gamma * (H.sum(1, keepdim=True) * X[r0:r1] - H @ X)
        dgamma -= 0.5 * float((H * D).sum())
    return dict(loss=loss, dX=dX, dgamma=dgamma)
