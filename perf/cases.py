"""The work this framework is measured on: matrix-vector products, Krylov
solves, the ILU(0) preconditioner, the batched solver and the training step of
the learned preconditioner, each through the public entry points of tnl_amd,
from the smallest calls (launch latency) to the largest (HBM bandwidth).

listed() are the cases, draw() gives further ones of the same ranges,
prepare() makes what a program holds before the call, run() is one pass,
work() the bytes and operations a pass cannot do without, tolerance() how far
two correct implementations may lie apart, and exact() the 64-bit answer in
plain torch."""
import math

import numpy as np
import torch

import tnl_amd
from tnl_amd import batched, solvers, spai

FORMATS = {"CSR": (tnl_amd.CSR, 0), "Ellpack": (tnl_amd.ELLPACK, 0), "SlicedEllpack32": (tnl_amd.SLICED_ELLPACK, 32),
           "SlicedEllpack64": (tnl_amd.SLICED_ELLPACK, 64)}
DTYPES = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one product with a small stencil matrix: the call and its launch are most of the time
        {"name": "spmv_laplace512_csr_f64", "kind": "spmv", "matrix": "laplace", "nx": 512, "ny": 512, "nz": 1,
         "format": "CSR", "dtype": "f64"},
        # one product with a large graph-like matrix (power-law rows, random columns): y = A x where x misses the caches
        {"name": "spmv_zipf4m_csr_f64", "kind": "spmv", "matrix": "zipf", "n": 4194304, "format": "CSR",
         "dtype": "f64"},
        # one single-precision product with a 3D stencil of odd sides in the GPU's usual sliced format
        {"name": "spmv_grid3d_sliced_f32", "kind": "spmv", "matrix": "laplace", "nx": 149, "ny": 151, "nz": 157,
         "format": "SlicedEllpack32", "dtype": "f32"},
        # a small variable-coefficient diffusion solve: hundreds of iterations of tiny kernels
        {"name": "cg_diffusion2d_120x97", "kind": "cg", "solver": "cg", "coefficients": "variable", "nx": 120,
         "ny": 97, "nz": 1, "format": "CSR"},
        # the large Poisson solve, in FP64 throughout
        {"name": "cg_poisson256_f64", "kind": "cg", "solver": "cg", "coefficients": "constant", "nx": 256, "ny": 256,
         "nz": 256, "format": "CSR"},
        # the same solve with BF16 matrix values and FP32 iterations inside FP64 residual replacement
        {"name": "cg_poisson256_reliable_bf16", "kind": "cg", "solver": "reliable_bf16", "coefficients": "constant",
         "nx": 256, "ny": 256, "nz": 256, "format": "Ellpack"},
        # GMRES as the solver class sets it up by default (MGSR, restart 10), on a middle-sized problem
        {"name": "gmres_mgsr10_convdiff200", "kind": "gmres", "variant": "MGSR", "restart": 10, "iterations": 200,
         "m": 200},
        # GMRES(30) with the blocked orthogonalisation on a large problem
        {"name": "gmres_cgsr30_convdiff1024", "kind": "gmres", "variant": "CGSR", "restart": 30, "iterations": 300,
         "m": 1024},
        # one implicit time step of convection-diffusion
        {"name": "bicgstab_step_convdiff1024", "kind": "bicgstab", "m": 1024, "shift": 0.02},
        # one application of the ILU(0) preconditioner (forward and backward triangular solve)
        {"name": "ilu0_apply_convdiff1024", "kind": "ilu0", "matrix": "convdiff", "nx": 1024, "ny": 1024, "nz": 1},
        # many small independent solves in one launch
        {"name": "batched_cg_1024", "kind": "batched", "systems": 1024, "smin": 16, "smax": 128, "block": 1024,
         "lanes": 1, "format": "CSR"},
        # one training step's forward and backward pass of the learned sparse approximate inverse
        {"name": "spai_train_256", "kind": "spai", "m": 256, "probes": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "cg", "cg", "gmres", "bicgstab", "ilu0", "batched", "spai"])
    if kind == "spmv":
        if rng.random() < 0.35:
            return {"kind": "spmv", "matrix": "zipf", "n": _log(rng, 20000, 4194304), "format": "CSR",
                    "dtype": rng.choice(["f64", "f32"])}
        case = {"kind": "spmv", "matrix": "laplace", "format": rng.choice(sorted(FORMATS)),
                "dtype": rng.choice(["f64", "f32"])}
        if rng.random() < 0.5:
            return dict(case, nx=_log(rng, 60, 3000), ny=_log(rng, 60, 3000), nz=1)
        return dict(case, nx=_log(rng, 24, 256), ny=_log(rng, 24, 256), nz=_log(rng, 24, 256))
    if kind == "cg":
        coefficients = rng.choice(["constant", "variable"])
        solver = rng.choice(["cg", "reliable"])
        if solver == "reliable":  # BF16 holds the constant stencil's values exactly; varying ones need FP32
            solver = "reliable_bf16" if coefficients == "constant" else "reliable_f32"
        case = {"kind": "cg", "solver": solver, "coefficients": coefficients, "format": rng.choice(["CSR", "Ellpack"])}
        if rng.random() < 0.5:
            return dict(case, nx=_log(rng, 40, 500), ny=_log(rng, 40, 500), nz=1)
        top = 230 if coefficients == "constant" else 150
        return dict(case, nx=_log(rng, 20, top), ny=_log(rng, 20, top), nz=_log(rng, 20, top))
    if kind == "gmres":
        return {"kind": "gmres", "variant": rng.choice(["MGSR", "CGSR", "MGS", "CGS"]),
                "restart": rng.choice([10, 20, 30]), "iterations": 60 * rng.randint(1, 5), "m": _log(rng, 64, 1024)}
    if kind == "bicgstab":
        return {"kind": "bicgstab", "m": _log(rng, 100, 1024), "shift": rng.choice([0.01, 0.02, 0.05])}
    if kind == "ilu0":
        if rng.random() < 0.5:
            m = _log(rng, 90, 1024)
            return {"kind": "ilu0", "matrix": "convdiff", "nx": m, "ny": m, "nz": 1}
        if rng.random() < 0.5:
            return {"kind": "ilu0", "matrix": "diffusion", "nx": _log(rng, 80, 1024), "ny": _log(rng, 80, 1024),
                    "nz": 1}
        return {"kind": "ilu0", "matrix": "diffusion", "nx": _log(rng, 16, 80), "ny": _log(rng, 16, 80),
                "nz": _log(rng, 16, 80)}
    if kind == "batched":
        return {"kind": "batched", "systems": _log(rng, 64, 1024), "smin": rng.choice([8, 12, 16]),
                "smax": rng.choice([48, 64, 96, 128]), "block": rng.choice([256, 512, 1024]),
                "lanes": rng.choice([1, 2]), "format": rng.choice(["CSR", "SlicedEllpack32"])}
    return {"kind": "spai", "m": _log(rng, 48, 300), "probes": rng.choice([2, 4])}


# ---------------------------------------------------------------- matrices
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _normal(n, g):
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float64)


class Grid:
    """A 5- or 7-point matrix on an nx x ny x nz grid: coefficient k of row i multiplies x[i + shift[k]] (0 where
    the grid ends)."""

    def __init__(self, nx, ny, nz, coefficients, mask):
        self.n = nx * ny * nz
        self.dims = (nx, ny, nz)
        self.shift = [-nx * ny, -nx, -1, 0, 1, nx, nx * ny]
        self.c = coefficients  # 7 x n
        self.mask = mask       # 7 x n, the stored entries

    def csr(self):
        keep = self.mask.t()
        shift = torch.tensor(self.shift, device="cuda", dtype=torch.int32)
        cols = (torch.arange(self.n, device="cuda", dtype=torch.int32)[:, None] + shift)[keep]
        off = torch.zeros(self.n + 1, dtype=torch.int32, device="cuda")
        off[1:] = self.mask.sum(0).cumsum(0)
        return off, cols, self.c.t()[keep]

    def times(self, x):
        y = self.c[3] * x
        for k, s in enumerate(self.shift):
            if s > 0 and s < self.n:
                y[:-s] += self.c[k, :-s] * x[s:]
            elif s < 0 and -s < self.n:
                y[-s:] += self.c[k, -s:] * x[:s]
        return y


def _mask(nx, ny, nz):
    m = torch.ones(7, nz, ny, nx, dtype=torch.bool, device="cuda")
    m[0, 0], m[6, -1] = False, False
    m[1, :, 0], m[5, :, -1] = False, False
    m[2, :, :, 0], m[4, :, :, -1] = False, False
    return m.reshape(7, -1)


def _laplace(nx, ny, nz):
    mask = _mask(nx, ny, nz)
    c = -mask.double()
    c[3] = 4.0 if nz == 1 else 6.0
    return Grid(nx, ny, nz, c, mask)


def _diffusion(nx, ny, nz, g):
    """Log-normal face coefficients, Dirichlet boundary faces included."""
    c = torch.zeros(7, nz, ny, nx, dtype=torch.float64, device="cuda")
    for axis, (lo, hi) in enumerate([(0, 6), (1, 5), (2, 4)]):
        if axis == 0 and nz == 1:
            continue
        shape = [nz, ny, nx]
        shape[axis] += 1
        face = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64).exp()
        low, high = face.narrow(axis, 0, shape[axis] - 1), face.narrow(axis, 1, shape[axis] - 1)
        c[3] += low + high
        c[lo] -= low
        c[hi] -= high
    mask = _mask(nx, ny, nz)
    c = c.reshape(7, -1)
    c[~mask] = 0.0
    return Grid(nx, ny, nz, c, mask)


def _convdiff(m, g, shift=0.0):
    """Upwind convection-diffusion on an m x m grid with a divergence-free velocity of eight random modes, plus
    shift on the diagonal (an implicit time step)."""
    h = 1.0 / (m + 1)
    x = torch.arange(1, m + 1, device="cuda", dtype=torch.float64) * (h * math.pi)
    amp, k = _normal(8, g), torch.randint(1, 5, (2, 8), generator=g, device="cuda")
    sx, cx = torch.sin(k[0][:, None] * x), torch.cos(k[0][:, None] * x)
    sy, cy = torch.sin(k[1][:, None] * x), torch.cos(k[1][:, None] * x)
    amp = (amp / (k[0] ** 2 + k[1] ** 2).double().sqrt())[:, None]
    vx = ((amp * k[1][:, None] * cy).t() @ sx).reshape(-1)
    vy = -((amp * sy).t() @ (k[0][:, None] * cx)).reshape(-1)
    scale = h * (1.0 + 99.0 * torch.rand(1, generator=g, device="cuda", dtype=torch.float64))
    scale = scale / (vx * vx + vy * vy).max().sqrt()
    vx, vy = vx * scale, vy * scale
    c = torch.zeros(7, m * m, dtype=torch.float64, device="cuda")
    c[1], c[2] = -1.0 - vy.clamp(min=0.0), -1.0 - vx.clamp(min=0.0)
    c[3] = 4.0 + shift + vx.abs() + vy.abs()
    c[4], c[5] = -1.0 - (-vx).clamp(min=0.0), -1.0 - (-vy).clamp(min=0.0)
    mask = _mask(m, m, 1)
    c[~mask] = 0.0
    return Grid(m, m, 1, c, mask)


def _zipf(n, g):
    """Power-law row lengths (exponent 2, at most 4096, 16 on average), distinct uniform columns, normal values."""
    p = torch.arange(1, 4097, device="cuda", dtype=torch.float64) ** -2
    k = torch.searchsorted((p / p.sum()).cumsum(0), torch.rand(n, generator=g, device="cuda", dtype=torch.float64))
    k = (k + 1).clamp(max=4096).double()
    lo, hi = 1.0, 64.0
    for _ in range(40):
        a = 0.5 * (lo + hi)
        if float((k * a).round().clamp(1, 4096).mean()) > 16.0:
            hi = a
        else:
            lo = a
    size = (k * lo).round().clamp(1, min(4096, n)).long()
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), size)
    key = row * n + torch.randint(0, n, (row.numel(),), generator=g, device="cuda")
    del row
    key = torch.unique_consecutive(key.sort()[0])
    off = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    off[1:] = torch.bincount(key // n, minlength=n).cumsum(0)
    return off, (key % n).int(), _normal(key.numel(), g)


def _batch(case, g):
    """Independent 2D diffusion systems as one block-diagonal CSR matrix, and each system's first row: sides spread
    evenly over the logarithm of [smin, smax] in a mixed order, log-normal face coefficients."""
    k = torch.arange(case["systems"], dtype=torch.float64)
    sides = (case["smin"] * (case["smax"] / case["smin"]) ** (k * 0.6180339887498949 % 1.0)).round().long()
    rows = torch.zeros(len(sides) + 1, dtype=torch.int64)
    rows[1:] = (sides * sides).cumsum(0)
    n = int(rows[-1])
    system = torch.repeat_interleave(torch.arange(len(sides), device="cuda"), (sides * sides).cuda())
    s, i = sides.cuda()[system], torch.arange(n, device="cuda")
    local = i - rows.cuda()[system]
    ix, iy = local % s, local // s
    east, north, west_end, south_end = (_normal(n, g).exp() for _ in range(4))
    west = torch.where(ix > 0, east[(i - 1).clamp(min=0)], west_end)
    south = torch.where(iy > 0, north[(i - s).clamp(min=0)], south_end)
    vals = torch.stack([-south, -west, east + north + west + south, -east, -north], 1)
    cols = torch.stack([i - s, i - 1, i, i + 1, i + s], 1)
    keep = torch.stack([iy > 0, ix > 0, ix >= 0, ix < s - 1, iy < s - 1], 1)
    off = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    off[1:] = keep.sum(1).cumsum(0)
    return (off, cols[keep].int(), vals[keep]), rows.numpy()


def _grid(case, g):
    kind = case.get("matrix") or case.get("coefficients")
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if kind in ("laplace", "constant"):
        return _laplace(nx, ny, nz)
    return _convdiff(nx, g) if kind == "convdiff" else _diffusion(nx, ny, nz, g)


def _matrix(csr, fmt="CSR", dtype=torch.float64):
    off, cols, vals = csr
    n = off.numel() - 1
    f, param = FORMATS[fmt]
    return tnl_amd.SparseMatrix.from_csr(n, n, off, cols, vals, fmt=f, param=param, value_dtype=dtype)


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    """(matrix, right-hand side or vector) of a case, in 64 bits: a Grid or CSR arrays, and a tensor."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "spmv" and case["matrix"] == "zipf":
        csr = _zipf(case["n"], g)
        return csr, _normal(case["n"], g)
    if kind in ("spmv", "cg", "ilu0"):
        grid = _grid(case, g)
    else:
        grid = _convdiff(case["m"], g, case.get("shift", 0.0))
    return grid, _normal(grid.n, g)


def _spai_inputs(case, seed):
    g = _generator(seed)
    grid = _convdiff(case["m"], g)
    p = spai.init_parameters(seed % 100000)
    rng = np.random.default_rng(seed % 100000 + 1)  # a decoder under training (the initial one is zero)
    p[-65:] = 0.02 * rng.standard_normal(65)
    Z = torch.randint(0, 2, (case["probes"], grid.n), generator=g, device="cuda").double() * 2.0 - 1.0
    return grid, p, Z


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batched":
        g = _generator(seed)
        csr, sys_rows = _batch(case, g)
        A = _matrix(csr, case["format"])
        solver = batched.BatchedCG(A, sys_rows, block_size=case["block"], lanes_per_row=case["lanes"])
        b = _normal(A.rows, g)
        return {"kind": kind, "A": A, "solver": solver, "b": b, "x": torch.zeros_like(b)}
    if kind == "spai":
        grid, p, Z = _spai_inputs(case, seed)
        return {"kind": kind, "A": _matrix(grid.csr()), "net": spai.Network(p), "Z": Z}
    source, v = _inputs(case, seed)
    csr = source.csr() if isinstance(source, Grid) else source
    if kind == "spmv":
        dtype = DTYPES[case["dtype"]]
        A = _matrix(csr, case["format"], dtype)
        x = v.to(dtype)
        return {"kind": kind, "A": A, "x": x, "y": torch.zeros_like(x)}
    A = _matrix(csr, case.get("format", "CSR"))
    state = {"kind": kind, "A": A, "b": v, "x": torch.zeros_like(v)}
    if kind == "ilu0":
        state["preconditioner"] = solvers.ILU0(A)
        return state
    if kind == "cg" and case["solver"] != "cg":
        s = solvers.ReliableMixedCG()
        state["A_lo"] = tnl_amd.SparseMatrix(A.rows, A.columns, A.segments,
                                             A.values.to(DTYPES[case["solver"].split("_")[1]]), A.column_indexes)
        s.setInnerMatrix(state["A_lo"])
    else:
        s = {"cg": solvers.CG, "gmres": solvers.GMRES, "bicgstab": solvers.BICGStab}[kind]()
        state["preconditioner"] = solvers.Diagonal(A)
        s.setPreconditioner(state["preconditioner"])
    s.setMatrix(A)
    s.setConvergenceResidue(1e-10)
    if kind == "gmres":
        # a budget of iterations (the reference counts one more than the limit), as inside an outer iteration
        s.setup(case["variant"], case["restart"], case["restart"])
        s.setConvergenceResidue(0.0)
        s.setMaxIterations(case["iterations"] - 1)
    state["solver"] = s
    return state


def run(state):
    kind = state["kind"]
    if kind == "spmv":
        return state["A"].vectorProduct(state["x"], state["y"])
    if kind == "spai":
        loss, M = state["net"].loss_grad(state["A"], state["Z"])
        return {"loss": loss, "M": M, "gradients": state["net"].gradients()}
    if kind == "ilu0":
        return state["preconditioner"].solve(state["b"], state["x"])
    state["x"].zero_()  # the initial guess
    if kind == "batched":
        state["solver"].solve(state["b"], state["x"])
    else:
        state["solver"].solve(state["b"], state["x"])
    return state["x"]


# ---------------------------------------------------------------- work
def work(case):
    """Each input read once and each output written once per pass, and for an iterative solve per iteration: the
    matrix once (12 bytes per FP64 entry), and each vector the iteration's recurrences read or write once.  Numbers of
    iterations are those these problems are known to take."""
    kind = case["kind"]
    if kind == "spmv":
        sv = 8 if case["dtype"] == "f64" else 4
        if case["matrix"] == "zipf":
            n, nnz = case["n"], 16 * case["n"]
        else:
            n, nnz = _grid_size(case)
        return {"bytes": (sv + 4) * nnz + 4 * (n + 1) + 2 * sv * n, "flops": 2 * nnz}
    if kind == "cg":
        n, nnz = _grid_size(case)
        side = max(case["nx"], case["ny"], case["nz"])
        its = side * (4.1 if case["coefficients"] == "constant" else 6.0)
        entry, vec = (12, 8) if case["solver"] == "cg" else (6, 4) if case["solver"] == "reliable_bf16" else (8, 4)
        return {"bytes": its * (entry * nnz + 11 * vec * n), "flops": its * (2 * nnz + 10 * n)}
    if kind == "spai":
        e, n = 5 * case["m"] ** 2, case["m"] ** 2
        # three layers, forward and backward, of BF16 edge and node activations of width 64 written and read, and
        # their five 64 x 64 products (one per edge, four per node) with two more of each size in the backward pass
        return {"bytes": 3 * 2 * 2 * 128 * (e + n) + 40 * e, "flops": 3 * 3 * 2 * 64 * 64 * (e + 4 * n)}
    if kind == "batched":
        # sides uniform in the logarithm: the mean of s^2; a system of side s takes about 6.5 s iterations
        a, b = case["smin"], case["smax"]
        span = math.log(b / a)
        rows, its_rows = (b * b - a * a) / (2 * span), 6.5 * (b ** 3 - a ** 3) / (3 * span)
        k = case["systems"]
        return {"bytes": k * rows * (5 * 12 + 24), "flops": k * its_rows * (10 + 10)}
    if kind == "ilu0":
        n, nnz = _grid_size(case)
        return {"bytes": 12 * nnz + 32 * n, "flops": 2 * nnz}
    n = case["m"] ** 2
    nnz = 5 * n
    if kind == "gmres":
        passes = 2 if case["variant"].endswith("R") else 1
        mean = (case["restart"] + 1) / 2
        per = 12 * nnz + 8 * n * (4 + passes * mean)
        return {"bytes": case["iterations"] * per,
                "flops": case["iterations"] * (2 * nnz + 4 * n * passes * mean)}
    its = 10 / math.sqrt(case["shift"])
    return {"bytes": its * (24 * nnz + 16 * 8 * n), "flops": its * (4 * nnz + 20 * n)}


def _grid_size(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    return n, n + 2 * (n - ny * nz) + 2 * (n - nx * nz) + 2 * (n - nx * ny)


def tolerance(case):
    kind = case["kind"]
    if kind == "spmv":  # the products of a row in another order
        return {"rel": 5e-15, "max": 1e-12} if case["dtype"] == "f64" else {"rel": 1e-6, "max": 1e-3}
    if kind == "ilu0":  # rounding along the chain of a triangular solve
        return {"rel": 1e-14, "max": 1e-12}
    if kind == "gmres":  # rounding over restart cycles
        return {"rel": 1e-10, "max": 1e-8}
    if kind in ("cg", "batched", "bicgstab"):
        # both answers meet ||b - A x|| <= 1e-10 ||b|| (in the solver's norm); x is off by up to the condition number
        return {"rel": 2e-8, "max": 1e-6}
    return {"rel": 2e-2, "max": 0.5}  # BF16 activations: ties and signs near zero fall either way


# ---------------------------------------------------------------- 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind == "spai":
        return _spai_exact(*_spai_inputs(case, seed))
    if kind == "batched":
        return _batched_exact(case, seed)
    source, v = _inputs(case, seed)
    if kind == "spmv":
        dtype = DTYPES[case["dtype"]]
        x = v.to(dtype).double()
        if isinstance(source, Grid):
            return source.times(x)
        off, cols, vals = source
        row = torch.repeat_interleave(torch.arange(x.numel(), device="cuda"), (off[1:] - off[:-1]).long())
        return torch.zeros_like(x).index_add_(0, row, vals.to(dtype).double() * x[cols])
    if kind == "cg":
        return _pcg(source.times, source.c[3], v, lambda t: t.sum())
    if kind == "ilu0":
        return _ilu0_exact(source, v)
    if kind == "gmres":
        return _gmres(source, v, case["restart"], case["iterations"], 0.0)
    return _gmres(source, v, 30, 3000, 1e-15)


def _pcg(times, diag, b, total, rounds=6000):
    """Jacobi-CG to the accuracy of 64 bits; total sums a vector's entries (per system)."""
    x = torch.zeros_like(b)
    r = b.clone()
    p = r / diag
    rz = total(r * p)
    target = rz * 1e-28
    for i in range(rounds):
        q = times(p)
        alpha = torch.where(rz > target, rz / total(p * q), torch.zeros_like(rz))  # (a system that is done rests)
        x += _spread(alpha, total) * p
        r -= _spread(alpha, total) * q
        z = r / diag
        new = total(r * z)
        if i % 20 == 19 and bool((new <= target).all()):
            break
        p = z + _spread(torch.where(rz > target, new / rz, torch.zeros_like(rz)), total) * p
        rz = new
    return x


def _spread(s, total):
    return total.spread(s) if hasattr(total, "spread") else s


class _PerSystem:
    """Sums over the rows of each system of a batch."""

    def __init__(self, sys_rows):
        self.lengths = torch.as_tensor(np.diff(sys_rows), device="cuda")

    def __call__(self, v):
        return torch.segment_reduce(v, "sum", lengths=self.lengths)

    def spread(self, s):
        return torch.repeat_interleave(s, self.lengths)


def _batched_exact(case, seed):
    g = _generator(seed)
    (off, cols, vals), sys_rows = _batch(case, g)
    n = int(sys_rows[-1])
    b = _normal(n, g)
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), (off[1:] - off[:-1]).long())
    diag = torch.zeros_like(b)
    diag[row[row == cols]] = vals[row == cols]
    A = torch.sparse_csr_tensor(off, cols, vals, (n, n))
    return _pcg(lambda p: A @ p, diag, b, _PerSystem(sys_rows))


def _gmres(grid, b, restart, iterations, target):
    """Left Jacobi-preconditioned GMRES(restart) from zero."""
    diag = grid.c[3]
    x = torch.zeros_like(b)
    norm = (b / diag).norm()
    done = 0
    while done < iterations:
        r = (b - grid.times(x)) / diag
        beta = r.norm()
        if float(beta) <= target * float(norm):
            break
        steps = min(restart, iterations - done)
        V = torch.zeros(steps + 1, b.numel(), dtype=torch.float64, device="cuda")
        H = torch.zeros(steps + 1, steps, dtype=torch.float64, device="cuda")
        V[0] = r / beta
        for j in range(steps):
            w = grid.times(V[j]) / diag
            for _ in range(2):
                h = V[: j + 1] @ w
                w = w - h @ V[: j + 1]
                H[: j + 1, j] += h
            H[j + 1, j] = w.norm()
            V[j + 1] = w / H[j + 1, j]
        e = torch.zeros(steps + 1, 1, dtype=torch.float64)
        e[0] = float(beta)
        y = torch.linalg.lstsq(H.cpu(), e).solution[:, 0].cuda()
        x = x + y @ V[:steps]
        done += steps
    return x


def _ilu0_exact(grid, b):
    """The 5/7-point stencil's ILU(0) (its pattern has no triangles, so only the diagonal changes), along the planes
    x + y + z = const."""
    nx, ny, nz = grid.dims
    i = torch.arange(grid.n, device="cuda")
    level = i % nx + (i // nx) % ny + i // (nx * ny)
    order = torch.argsort(level, stable=True)
    planes = torch.split(order, torch.bincount(level).tolist())
    ks = [k for k, s in enumerate(grid.shift) if abs(s) < grid.n and s != 0]
    low, high = [k for k in ks if k < 3], [k for k in ks if k > 3]
    c, shift = grid.c, grid.shift
    d, y, x = c[3].clone(), b.clone(), torch.zeros_like(b)

    def at(v, rows, k):
        return v[(rows + shift[k]).clamp(0, grid.n - 1)]
    for rows in planes:
        for k in low:
            ratio = c[k, rows] / at(d, rows, k)
            d[rows] -= ratio * at(c[6 - k], rows, k)
            y[rows] -= ratio * at(y, rows, k)
    for rows in reversed(planes):
        t = y[rows]
        for k in high:
            t = t - c[k, rows] * at(x, rows, k)
        x[rows] = t / d[rows]
    return x


def _spai_exact(grid, flat, Z):
    """Forward pass, probe loss and gradients of the network in 64 bits."""
    off, col, vals = grid.csr()
    n, col = grid.n, col.long()
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), (off[1:] - off[:-1]).long())
    p, k = {}, 0
    for name, shape in spai.layout():
        size = int(np.prod(shape))
        p[name] = torch.tensor(flat[k:k + size], dtype=torch.float64, device="cuda").reshape(shape).requires_grad_()
        k += size

    def by_row(e, index=row):
        return torch.zeros((n,) + e.shape[1:], dtype=torch.float64, device="cuda").index_add(0, index, e)
    on_diagonal = (row == col).double()
    diag, deg = by_row(vals * on_diagonal), by_row(torch.ones_like(vals))
    xe = torch.stack([vals / diag[row], vals / diag[col], on_diagonal, vals.abs() / diag[row]], 1)
    xn = torch.stack([by_row(vals.abs() * (1 - on_diagonal)) / diag, by_row(vals) / diag, deg / 5, torch.ones_like(diag)], 1)
    E, H = (xe @ p["Ae"] + p["ae"]).relu(), (xn @ p["An"] + p["an"]).relu()
    for layer in range(spai.LAYERS):
        w = {name: p[f"{name}{layer}"] for name in ("We", "Wu", "Wv", "Wh", "Wg", "be", "bh")}
        E = (E @ w["We"] + (H @ w["Wu"])[col] + (H @ w["Wv"])[row] + w["be"]).relu()
        H = (H @ w["Wh"] + (by_row(E) / deg[:, None]) @ w["Wg"] + w["bh"]).relu()
    M = (on_diagonal + E @ p["wo"] + p["bo"]) / diag[row]
    loss = 0.0
    for z in Z:
        y = by_row(vals * z[col])
        loss = loss + (z - by_row(M * y[col])).square().sum()
    loss = loss / Z.numel()
    loss.backward()
    grads = torch.cat([(torch.zeros_like(t) if t.grad is None else t.grad).reshape(-1) for t in p.values()])
    return {"loss": float(loss.detach()), "M": M.detach(), "gradients": grads}
