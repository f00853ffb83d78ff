"""Performance cases: the calls that a user of this package makes, over the range they make them in.

Every case runs through the public binding (smaxkernels_amd.capi) on device-resident operands.  Matrices are
made on the GPU: the heavy-tailed band matrix of the benchmark (Lomax(1.5) row lengths, mean 16,
cap 2000, one column in each of L equal strata of a band of +-N/8, so that a row's columns are distinct and
ascending), 5-point and 27-point stencils, and a 7-point adjacency of dense b x b blocks.

Kinds of work:
  powers     `steps` successive products y_{i+1} = A y_i (steps = 1: one SpMV), SELL-C-sigma handle or CRS arrays
  convert    CRS -> SELL-C-sigma of a new matrix (the handle a solver or a training loop then keeps)
  transpose  CRS -> SELL-C-sigma layout of A^T (what the adjoint product needs), for a new pattern
  train      one step of training the values of a sparse layer: new values into both layouts, Y = A X,
             dX = A^T G, dvals = SDDMM(G, X)
  spmm       CRS SpMM with the reference's default column-major operands
  cg         a whole solve: FP64 CG, or FP64 refinement of a CG on BF16 / FP32 values
  bcrs_train the training step on block matrices (values of the transpose refreshed, forward, adjoint, SDDMM)
  newton     a new block Jacobian: CRS -> BCRS, then `steps` successive products with it
"""
import math

import torch

from smaxkernels_amd import capi

DEV = "cuda"
VT = {"f64": capi.F64, "f32": capi.F32, "bf16": capi.BF16}
VAL = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
VEC = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.float32}
VB = {"f64": 8, "f32": 4, "bf16": 2}
XB = {"f64": 8, "f32": 4, "bf16": 4}
LOMAX_LAMBDA, LOMAX_CAP, LOMAX_MEAN = 8.3, 2000, 16.03
CG_TOL = 1e-12


def listed():
    return [
        # four terms of a Krylov basis on a small grid: launch latency, everything in cache
        {"name": "powers_poisson64_sell_f64", "kind": "powers", "matrix": "poisson", "n": 64, "format": "sell",
         "C": 64, "sigma": 1, "dtype": "f64", "steps": 4},
        # one FP64 SpMV of the benchmark's largest matrix in its headline layout
        {"name": "spmv_lomax4m_sell_f64", "kind": "powers", "matrix": "lomax", "n": 4000000, "format": "sell",
         "C": 64, "sigma": 4096, "dtype": "f64", "steps": 1},
        # one SpMV on the registered CRS arrays (no conversion), BF16 values, an odd number of rows
        {"name": "spmv_lomax300k_crs_bf16", "kind": "powers", "matrix": "lomax", "n": 300007, "format": "crs",
         "C": 64, "sigma": 1, "dtype": "bf16", "steps": 1},
        # a matrix assembled anew enters the solver's layout
        {"name": "convert_lomax2m_f64", "kind": "convert", "matrix": "lomax", "n": 2000003, "C": 64, "sigma": 4096,
         "dtype": "f64"},
        # a new sparsity pattern needs the layout of its transpose for the backward pass
        {"name": "transpose_lomax500k_f32", "kind": "transpose", "matrix": "lomax", "n": 500009, "C": 64,
         "sigma": 65536, "dtype": "f32"},
        # the benchmark's differentiation workload as a training step
        {"name": "train_lomax1m_f32_k32", "kind": "train", "matrix": "lomax", "n": 1000000, "C": 64, "sigma": 65536,
         "dtype": "f32", "k": 32},
        # the same step on a small graph with BF16 weights and a feature count that is no power of two
        {"name": "train_lomax40k_bf16_k20", "kind": "train", "matrix": "lomax", "n": 40013, "C": 64, "sigma": 4096,
         "dtype": "bf16", "k": 20},
        # block of right-hand sides in the reference's default layout (column-major), a handful of columns
        {"name": "spmm_lomax200k_f64_k10", "kind": "spmm", "matrix": "lomax", "n": 200003, "dtype": "f64", "k": 10},
        # a small FP64 solve: many short, dependent iterations
        {"name": "cg_poisson96_f64", "kind": "cg", "matrix": "poisson", "n": 96, "inner": "f64"},
        # a large solve by BF16-value CG under FP64 refinement
        {"name": "ircg_stencil128_bf16", "kind": "cg", "matrix": "stencil", "n": 128, "inner": "bf16"},
        # the benchmark's block matrix, all three products of a training step
        {"name": "bcrs_train_96_bf16_k8", "kind": "bcrs_train", "n": 96, "b": 4, "dtype": "bf16", "k": 8},
        # 3 x 3 FP64 blocks (displacements in three dimensions): a new Jacobian and the products of a short solve
        {"name": "newton_48_f64_b3", "kind": "newton", "n": 48, "b": 3, "dtype": "f64", "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["powers", "powers", "convert", "transpose", "train", "train", "spmm", "cg", "bcrs_train",
                       "newton"])
    dtype = rng.choice(["f64", "f32", "bf16"])
    if kind == "powers":
        matrix = rng.choice(["poisson", "lomax", "stencil"])
        n = {"poisson": lambda: _log_int(rng, 32, 1024), "lomax": lambda: _log_int(rng, 5000, 4000000),
             "stencil": lambda: _log_int(rng, 14, 128)}[matrix]()
        return {"kind": kind, "matrix": matrix, "n": n, "format": rng.choice(["sell", "sell", "crs"]),
                "C": rng.choice([32, 64]), "sigma": 1 if matrix != "lomax" else rng.choice([64, 4096, 65536]),
                "dtype": dtype, "steps": 1 if matrix == "lomax" or n > 300 else rng.randint(1, 8)}
    if kind == "convert":
        return {"kind": kind, "matrix": "lomax", "n": _log_int(rng, 20000, 2000000), "C": rng.choice([32, 64]),
                "sigma": rng.choice([256, 1024, 4096, 65536, 1 << 30]), "dtype": dtype}
    if kind == "transpose":
        return {"kind": kind, "matrix": "lomax", "n": _log_int(rng, 20000, 1000000), "C": rng.choice([32, 64]),
                "sigma": rng.choice([1024, 4096, 65536]), "dtype": dtype}
    if kind == "train":
        k = rng.choice([1, 4, 8, 16, 32, 64, rng.randint(2, 48)])
        return {"kind": kind, "matrix": "lomax", "n": _log_int(rng, 10000, 1000000 if k <= 32 else 300000), "C": 64,
                "sigma": rng.choice([4096, 65536]), "dtype": dtype, "k": k}
    if kind == "spmm":
        return {"kind": kind, "matrix": "lomax", "n": _log_int(rng, 10000, 400000), "dtype": dtype,
                "k": rng.choice([2, 4, 8, 16, 32, rng.randint(2, 32)])}
    if kind == "cg":
        matrix = rng.choice(["poisson", "stencil"])
        return {"kind": kind, "matrix": matrix,
                "n": _log_int(rng, 24, 160) if matrix == "poisson" else _log_int(rng, 16, 128),
                "inner": rng.choice(["f64", "f32", "bf16"])}
    if kind == "bcrs_train":
        return {"kind": kind, "n": _log_int(rng, 12, 64), "b": rng.choice([2, 3, 4]), "dtype": dtype,
                "k": rng.choice([4, 8, 16, rng.randint(2, 24)])}
    return {"kind": kind, "n": _log_int(rng, 12, 64), "b": rng.randint(2, 6), "dtype": dtype,
            "steps": rng.randint(2, 10)}


# ---------------------------------------------------------------- matrices
def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(seed * 64 + salt)


def _uniform(g, n, dtype):
    return (torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * 2 - 1).to(dtype)


def _lomax(n, seed, fixed_columns=False):
    """CRS row pointers and columns of the band matrix.  Row lengths depend on n alone (every seed's arrays have
    the same sizes), columns on the seed too, unless the sizes follow from the columns."""
    g = _gen(n, 0)
    half = max(n // 8, 1)
    i = torch.arange(n, device=DEV)
    lo = (i - half).clamp_(min=0)
    width = (i + half).clamp_(max=n - 1) - lo + 1
    u = 1.0 - torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    length = (1 + (LOMAX_LAMBDA * (u.pow(-2.0 / 3.0) - 1)).floor()).clamp_(max=LOMAX_CAP).long()
    length = torch.minimum(length, width)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(length, 0, out=ptr[1:])
    nnz = int(ptr[-1])
    row = torch.repeat_interleave(i, length, output_size=nnz)
    j = torch.arange(nnz, device=DEV) - ptr[row]
    first = j * width[row] // length[row]
    last = (j + 1) * width[row] // length[row]
    span = last - first
    g = g if fixed_columns else _gen(seed, 1)
    off = (torch.rand(nnz, generator=g, device=DEV) * span).long()
    col = lo[row] + first + torch.minimum(off, span - 1)
    return ptr.int(), col.int()


def _grid(n, dims):
    """Coordinates of the n^dims grid points, slowest first."""
    i = torch.arange(n ** dims, device=DEV)
    return [(i // n ** (dims - 1 - d)) % n for d in range(dims)]


def _stencil(n, offsets, dims):
    """CRS of a stencil with the given offsets (in column order) on an n^dims grid."""
    x = _grid(n, dims)
    cols, inside = [], []
    for off in offsets:
        ok, c = torch.ones_like(x[0], dtype=torch.bool), torch.zeros_like(x[0])
        for d in range(dims):
            y = x[d] + off[d]
            ok &= (y >= 0) & (y < n)
            c = c * n + y
        cols.append(c)
        inside.append(ok)
    inside, cols = torch.stack(inside, 1), torch.stack(cols, 1)
    ptr = torch.zeros(n ** dims + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(inside.sum(1), 0, out=ptr[1:])
    return ptr.int(), cols[inside].int()


def _rows(ptr):
    return torch.repeat_interleave(torch.arange(ptr.numel() - 1, device=DEV), (ptr[1:] - ptr[:-1]).long())


POISSON = [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)]
CUBE27 = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
CROSS7 = [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0)]


def _matrix(case, seed):
    """(n_rows, row_ptr, col, val) of a scalar CRS matrix on the GPU."""
    n, dtype = case["n"], VAL[case.get("dtype", "f64")]
    if case["matrix"] == "lomax":
        ptr, col = _lomax(n, seed, fixed_columns=case["kind"] == "transpose")
        return n, ptr, col, _uniform(_gen(seed, 2), col.numel(), dtype)
    offsets, dims, diag = (POISSON, 2, 4.0) if case["matrix"] == "poisson" else (CUBE27, 3, 26.01)
    ptr, col = _stencil(n, offsets, dims)
    val = (_rows(ptr) == col).double() * (diag + 1) - 1
    return n ** dims, ptr, col, val.to(dtype)


def _block_matrix(case, seed):
    """Scalar CRS of the 7-point adjacency of dense b x b blocks on an n^3 grid, diagonal blocks shifted by 8 I."""
    n, b = case["n"], case["b"]
    bptr, bcol = _stencil(n, CROSS7, 3)
    nb = n ** 3
    per_row = ((bptr[1:] - bptr[:-1]).long() * b).repeat_interleave(b)
    ptr = torch.zeros(nb * b + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(per_row, 0, out=ptr[1:])
    nnz = int(ptr[-1])
    row = torch.repeat_interleave(torch.arange(nb * b, device=DEV), per_row, output_size=nnz)
    j = torch.arange(nnz, device=DEV) - ptr[row]
    col = bcol[bptr[row // b].long() + j // b].long() * b + j % b
    val = _uniform(_gen(seed, 2), nnz, torch.float32)
    val += 8.0 * (row == col)
    return nb * b, ptr.int(), col.int(), val.to(VAL[case["dtype"]])


# ---------------------------------------------------------------- the program's state
_context = None


def _ctx():
    global _context
    if _context is None:
        _context = capi.Context(0)
    return _context


class Owned:
    """A matrix handle, destroyed with the last reference to it."""

    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        self.handle.destroy()


class State:
    """What a program holds between calls."""

    def __init__(self, case):
        self.case, self.ctx, self.owned, self.plan = case, _ctx(), [], None

    def keep(self, handle):
        self.owned.append(Owned(handle))
        return handle

    def __del__(self):
        if self.plan:
            self.ctx.crs_plan_destroy(self.plan)


class _Device:
    """Device memory of a handle as an array that torch can view; it holds the handle."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(owner, ptr, n, typestr="<i4"):
    t = torch.as_tensor(_Device(owner, ptr, n, typestr), device=DEV)
    t.owner = owner  # the handle's memory lives as long as a result that shows it
    return t


# BF16 arrays of a handle are returned as their bit patterns
TYPESTR = {8: "<f8", 4: "<f4", 2: "<i2"}


def _sell_arrays(owner):
    i = owner.handle.info
    parts = {"chunk_ptr": (i.chunk_ptr, i.n_chunks + 1), "chunk_lengths": (i.chunk_lengths, i.n_chunks),
             "col": (i.col, i.n_elements), "val": (i.val, i.n_elements, TYPESTR[i.val_bytes]),
             "perm": (i.perm, i.n_rows), "src_index": (i.src_index, i.n_elements)}
    return {name: _view(owner, *part) for name, part in parts.items()}


def prepare(case, seed):
    s, c, kind = State(case), _ctx(), case["kind"]
    dtype = case.get("dtype", "f64")
    vec = VEC[dtype]
    g = _gen(seed, 3)
    if kind in ("bcrs_train", "newton"):
        s.n, s.ptr, s.col, s.val = _block_matrix(case, seed)
    else:
        s.n, s.ptr, s.col, s.val = _matrix(case, seed)
    s.nnz, n = s.col.numel(), s.n
    crs = (n, n, s.nnz, s.ptr, s.col, s.val, VB[dtype])
    torch.cuda.synchronize()  # the context works on a stream of its own
    if kind == "powers":
        s.ys = [_uniform(g, n, vec)] + [torch.zeros(n, dtype=vec, device=DEV) for _ in range(case["steps"])]
        if case["format"] == "sell":
            s.A = s.keep(c.scs_from_crs(*crs, case["C"], case["sigma"]))
        else:
            s.plan = c.crs_plan(n, s.nnz, s.ptr)
    elif kind == "train":
        k = case["k"]
        s.X, s.G = _uniform(g, n * k, vec), _uniform(g, n * k, vec)
        s.new_val = _uniform(g, s.nnz, VAL[dtype])
        s.Y, s.dX, s.dv = torch.zeros_like(s.X), torch.zeros_like(s.X), torch.zeros(s.nnz, dtype=vec, device=DEV)
        s.A = s.keep(c.scs_from_crs(*crs, case["C"], case["sigma"]))
        s.AT = s.keep(c.scs_transpose_from_crs(*crs, case["C"], case["sigma"]))
    elif kind == "spmm":
        s.X = _uniform(g, n * case["k"], vec)
        s.Y = torch.zeros_like(s.X)
        s.plan = c.crs_plan(n, s.nnz, s.ptr)
    elif kind == "cg":
        s.b, s.x = _uniform(g, n, torch.float64), torch.zeros(n, dtype=torch.float64, device=DEV)
        s.A = s.keep(c.scs_from_crs(*crs, 64, 1))
        s.params = capi.CgParams(rel_tol=CG_TOL, max_iters=20000, check_every=25, inner_rel_tol=0.1, max_inner=5000,
                                 inner_value_type=VT[case["inner"]], keep_diag_f32=1)
    elif kind == "bcrs_train":
        k, b = case["k"], case["b"]
        s.X, s.G = _uniform(g, n * k, vec), _uniform(g, n * k, vec)
        s.Y, s.dX, s.dv = torch.zeros_like(s.X), torch.zeros_like(s.X), torch.zeros(s.nnz, dtype=vec, device=DEV)
        s.A = s.keep(c.bcrs_from_crs(*crs, b, b, b, b, 0))
        s.AT = s.keep(s.A.transpose())
        s.ptr = s.col = s.val = None  # the program goes on with the block arrays
    elif kind == "newton":
        s.ys = [_uniform(g, n, vec)] + [torch.zeros(n, dtype=vec, device=DEV) for _ in range(case["steps"])]
    torch.cuda.synchronize()
    return s


def run(s):
    case, c = s.case, s.ctx
    kind, vt = case["kind"], VT[case.get("dtype", "f64")]
    if kind == "powers":
        for x, y in zip(s.ys, s.ys[1:]):
            if s.plan:
                c.crs_spmv(vt, s.n, s.n, s.nnz, s.ptr, s.col, s.val, x, y, s.plan)
            else:
                s.A.apply(vt, x, y, unpermuted=True)
        return s.ys[1:]
    if kind in ("convert", "transpose"):
        s.owned = []  # the last matrix's layout
        build = c.scs_from_crs if kind == "convert" else c.scs_transpose_from_crs
        s.keep(build(s.n, s.n, s.nnz, s.ptr, s.col, s.val, VB[case["dtype"]], case["C"], case["sigma"]))
        return _sell_arrays(s.owned[-1])
    if kind == "train":
        k = case["k"]
        s.A.refresh_values(s.new_val)
        s.AT.refresh_values(s.new_val)
        s.A.apply_spmm(vt, k, s.X, s.Y)
        s.AT.apply_spmm(vt, k, s.G, s.dX)
        s.A.sddmm(vt, k, s.G, s.X, s.dv)
        return [s.Y, s.dX, s.dv]
    if kind == "spmm":
        c.crs_spmm(vt, s.n, s.n, s.nnz, s.ptr, s.col, s.val, case["k"], False, s.X, s.n, s.Y, s.n, s.plan)
        return s.Y
    if kind == "cg":
        c._check(c.lib.smax_hip_zero(c.handle, s.x.data_ptr(), 8 * s.n))  # start from x = 0
        c.cg(s.A, s.b, s.x, s.params, case["inner"] != "f64")
        return s.x
    if kind == "bcrs_train":
        k = case["k"]
        s.AT.refresh_values(s.A.info.val)
        s.A.spmm(vt, k, s.X, s.Y)
        s.AT.spmm(vt, k, s.G, s.dX)
        s.A.sddmm(vt, k, s.G, s.X, s.dv)
        return [s.Y, s.dX, s.dv]
    s.owned = []  # the last Jacobian
    b = case["b"]
    A = s.keep(c.bcrs_from_crs(s.n, s.n, s.nnz, s.ptr, s.col, s.val, VB[case["dtype"]], b, b, b, b, 0))
    for x, y in zip(s.ys, s.ys[1:]):
        A.spmv(vt, x, y)
    i, owner = A.info, s.owned[-1]
    return {"col": _view(owner, i.col, i.n_blocks), "row_ptr": _view(owner, i.row_ptr, i.n_block_rows + 1),
            "y": s.ys[1:]}


# ---------------------------------------------------------------- compulsory work
def _nnz(case):
    n = case["n"]
    if "b" in case:
        return (7 * n ** 3 - 6 * n ** 2) * case["b"] ** 2
    if case["matrix"] == "lomax":
        return int(LOMAX_MEAN * n)
    return 5 * n * n - 4 * n if case["matrix"] == "poisson" else (3 * n - 2) ** 3


def _iterations(case):
    """CG iterations to CG_TOL: about half of what the condition number's bound sqrt(kappa) / 2 ln(2 / tol) allows."""
    t = 2 * math.cos(math.pi / (case["n"] + 1))
    kappa = (4 + 2 * t) / (4 - 2 * t) if case["matrix"] == "poisson" else 36.01 / (27.01 - (1 + t) ** 3)
    return 0.25 * math.sqrt(kappa) * math.log(2 / CG_TOL)


def work(case):
    kind, nnz = case["kind"], _nnz(case)
    dtype = case.get("dtype", "f64")
    vb, xb = VB[dtype], XB[dtype]
    if "b" in case:
        b, n = case["b"], case["n"] ** 3 * case["b"]
        blocks = nnz // b ** 2
        matrix = nnz * vb + 4 * blocks + 4 * (n // b + 1)
    else:
        n = case["n"] ** {"lomax": 1, "poisson": 2, "stencil": 3}[case["matrix"]]
        matrix = nnz * (vb + 4) + 4 * (n + 1)
    if kind == "powers":  # a matrix that stays in the caches is read once from memory
        return {"bytes": matrix + (1 + case["steps"]) * n * xb, "flops": 2 * nnz * case["steps"]}
    if kind in ("convert", "transpose"):  # CRS in; columns, values, positions and permutations out
        return {"bytes": matrix + nnz * (vb + 8) + 12 * n, "flops": 0}
    if kind == "train":  # values in, both layouts' columns and values, X and G in, three results out
        k = case["k"]
        return {"bytes": nnz * (vb + 2 * (vb + 4) + xb) + 4 * n * k * xb, "flops": 6 * nnz * k}
    if kind == "spmm":
        return {"bytes": matrix + 2 * n * case["k"] * xb, "flops": 2 * nnz * case["k"]}
    if kind == "cg":  # per iteration the values and one-byte columns, and ten vector passes
        lo = case["inner"]
        return {"bytes": _iterations(case) * (nnz * (VB[lo] + 1) + 10 * n * XB[lo]),
                "flops": _iterations(case) * (2 * nnz + 10 * n)}
    if kind == "bcrs_train":
        k = case["k"]
        return {"bytes": 2 * matrix + 4 * n * k * xb + nnz * xb, "flops": 6 * nnz * k}
    crs = nnz * (vb + 4) + 4 * (n + 1)
    return {"bytes": crs + matrix + (1 + case["steps"]) * n * xb, "flops": 2 * nnz * case["steps"]}


# ---------------------------------------------------------------- results in 64 bits
def _product(row, col, val, X, n_out, part=1 << 22):
    """sum over entries of val * X[col] into the rows `row`, in binary64 (X: rows x k)."""
    Y = torch.zeros(n_out, X.shape[1], dtype=torch.float64, device=DEV)
    for a in range(0, col.numel(), part):
        p = slice(a, a + part)
        Y.index_add_(0, row[p], val[p].double()[:, None] * X[col[p]])
    return Y


def _dots(row, col, G, X, part=1 << 22):
    """sum_v G[row, v] X[col, v] of every entry, in binary64."""
    return torch.cat([(G[row[a:a + part]] * X[col[a:a + part]]).sum(1) for a in range(0, col.numel(), part)])


def _sine(n):
    """Orthonormal sine basis (eigenvectors of the 1-D stencils) and its angles' cosines."""
    i = torch.arange(1, n + 1, dtype=torch.float64, device=DEV)
    a = math.pi / (n + 1)
    return math.sqrt(2 / (n + 1)) * torch.sin(a * i[:, None] * i[None, :]), torch.cos(a * i)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("convert", "transpose"):
        return None  # positions and copied values: they stay equal bit for bit
    s = State(case)
    vec = VEC[case.get("dtype", "f64")]
    g = _gen(seed, 3)
    if kind == "cg":  # closed form: both stencils are diagonal in the sine basis
        n = case["n"]
        S, c = _sine(n)
        if case["matrix"] == "poisson":
            B = _uniform(g, n * n, torch.float64).view(n, n)
            lam = 4 - 2 * c[:, None] - 2 * c[None, :]
            return (S @ ((S @ B @ S) / lam) @ S).reshape(-1)
        B = _uniform(g, n ** 3, torch.float64).view(n, n, n)
        t = 1 + 2 * c

        def transform(V):
            for _ in range(3):
                V = (S @ V.reshape(n, n * n)).reshape(n, n, n).permute(1, 2, 0).contiguous()
            return V

        return transform(transform(B) / (27.01 - t[:, None, None] * t[None, :, None] * t[None, None, :])).reshape(-1)
    n, ptr, col, val = (_block_matrix if "b" in case else _matrix)(case, seed)
    row, col = _rows(ptr), col.long()
    if kind in ("powers", "newton"):
        ys = [_uniform(g, n, vec).double()[:, None]]
        for _ in range(case["steps"]):
            ys.append(_product(row, col, val, ys[-1], n))
        ys = [y[:, 0] for y in ys[1:]]
        return ys if kind == "powers" else {"col": None, "row_ptr": None, "y": ys}
    k = case["k"]
    if kind == "spmm":
        X = _uniform(g, n * k, vec).double().view(k, n).T.contiguous()
        return _product(row, col, val, X, n).T.contiguous().reshape(-1)
    X, G = _uniform(g, n * k, vec).double().view(n, k), _uniform(g, n * k, vec).double().view(n, k)
    if kind == "train":
        val = _uniform(g, col.numel(), VAL[case["dtype"]])
    dv = _dots(row, col, G, X)
    if kind == "bcrs_train":  # entries in block order: block, row in block, column in block
        b = case["b"]
        per_row = (ptr[1:] - ptr[:-1]).long()
        j = torch.arange(col.numel(), device=DEV) - ptr[row].long()
        at = ptr[(row // b) * b].long() + (j // b) * b * b + (row % b) * b + j % b
        assert int(per_row.min()) > 0
        dv = torch.zeros_like(dv).index_copy_(0, at, dv)
    return [_product(row, col, val, X, n).reshape(-1), _product(col, row, val, G, n).reshape(-1), dv]
