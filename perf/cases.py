"""Performance cases of the sparse operators: CSR SpMV / SpMM and their COO forms.

A case names an entry point (`call`), a sparsity pattern and its sizes, the value and
index types, the op, and for SpMM the dense width.  `prepare` makes the operands on the
GPU from the seed, plus the prepared matrix where a program keeps one; `run` is one
operator call; `exact` is the same product in 64 bits in plain torch.

Entry points (`call`):
  spmv_kept   flagsparse_spmv_csr on a matrix prepared once: the iterative solver's or
              PageRank's inner step
  spmv        flagsparse_spmv_csr on the CSR arrays: one product with a new matrix, its
              structure checked by the call
  spmm_kept   flagsparse_spmm_csr_run on a prepared route: graph-network layers, block
              solvers
  spmm        flagsparse_spmm_csr on the CSR arrays
  coo_spmv    flagsparse_spmv_coo on unsorted COO arrays
  coo_spmm    flagsparse_spmm_coo on unsorted COO arrays

Patterns:
  uniform     equal rows, columns spread over the whole width
  ragged      row lengths between 0 and twice the mean, columns as above
  powerlaw    heavy-tailed row lengths (up to 50,000), columns as above
  rmat        R-MAT graph (0.57, 0.19, 0.19, 0.05), parallel edges kept: hub rows, hub
              columns and empty rows
  stencil     27-point stencil on a box, truncated at the boundary
  scattered   COO entries at uniformly random places, in random order
"""

import math

import numpy as np
import torch

import flagsparse_amd as fs

_DTYPES = {
    "f16": torch.float16,
    "bf16": torch.bfloat16,
    "f32": torch.float32,
    "f64": torch.float64,
    "c64": torch.complex64,
    "c128": torch.complex128,
}
_INDEX = {"i32": torch.int32, "i64": torch.int64}
_VALUE_BYTES = {"f16": 2, "bf16": 2, "f32": 4, "f64": 8, "c64": 8, "c128": 16}
_INDEX_BYTES = {"i32": 4, "i64": 8}


def listed():
    return [
        # a small system's product in a solver loop: the launch and the call are what counts
        dict(name="spmv_kept_4096_f32", call="spmv_kept", pattern="uniform", rows=4096, cols=4096, per_row=16,
             dtype="f32", index="i32", op="non"),
        # a small rectangular matrix used once, int64 indices as scipy / torch make them
        dict(name="spmv_ragged_3001_f64", call="spmv", pattern="ragged", rows=3001, cols=2503, per_row=11,
             dtype="f64", index="i64", op="non"),
        # a 3D PDE operator in an iterative solver, double precision
        dict(name="spmv_kept_stencil128_f64", call="spmv_kept", pattern="stencil", nx=128, ny=128, nz=128,
             dtype="f64", index="i32", op="non"),
        # a graph-sized matrix with heavy-tailed rows in a fixed-point iteration
        dict(name="spmv_kept_powerlaw4M_f32", call="spmv_kept", pattern="powerlaw", rows=4194304, cols=4194304,
             per_row=16, dtype="f32", index="i32", op="non"),
        # a gradient step's A^T r with a matrix that was just assembled
        dict(name="spmv_trans_uniform1M_f32", call="spmv", pattern="uniform", rows=1048576, cols=1048576, per_row=32,
             dtype="f32", index="i32", op="trans"),
        # a few right-hand sides on a small matrix, odd width
        dict(name="spmm_ragged_2047_f32_n17", call="spmm", pattern="ragged", rows=2047, cols=1531, per_row=9,
             dtype="f32", index="i32", op="non", n=17),
        # a graph layer's feature aggregation, 64 features
        dict(name="spmm_kept_uniform1M_f32_n64", call="spmm_kept", pattern="uniform", rows=1048576, cols=1048576,
             per_row=32, dtype="f32", index="i32", op="non", n=64),
        # a graph with hubs and wide features: the largest case
        dict(name="spmm_kept_rmat21_f32_n256", call="spmm_kept", pattern="rmat", scale=21, edges=16, dtype="f32",
             index="i64", op="non", n=256),
        # the adjoint on a complex block of vectors, the matrix new to the call
        dict(name="spmm_conj_rmat21_c64_n32", call="spmm", pattern="rmat", scale=21, edges=16, dtype="c64",
             index="i64", op="conj", n=32),
        # aggregation in the 16-bit type that networks train in
        dict(name="spmm_kept_ragged250k_bf16_n128", call="spmm_kept", pattern="ragged", rows=250007, cols=250007,
             per_row=24, dtype="bf16", index="i32", op="non", n=128),
        # a matrix as an assembly loop leaves it: unsorted triplets, one product
        dict(name="coo_spmv_400k_f64", call="coo_spmv", pattern="scattered", rows=400009, cols=400009, per_row=10,
             dtype="f64", index="i64", op="non"),
        # edge list times features, without a conversion by the caller
        dict(name="coo_spmm_300k_f32_n32", call="coo_spmm", pattern="scattered", rows=300007, cols=300007, per_row=20,
             dtype="f32", index="i64", op="non", n=32),
    ]


_MAX_NNZ = 1 << 26
_MAX_SPMM_WORK = 1 << 32  # nnz * n, half of the largest listed case


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["spmv_kept", "spmv", "spmm_kept", "spmm", "coo_spmv", "coo_spmm"])
    coo = call.startswith("coo")
    spmm = "spmm" in call
    pattern = "scattered" if coo else rng.choice(["uniform", "ragged", "powerlaw", "rmat", "stencil"])
    dtype = rng.choice(["f32", "f32", "f64", "f64", "c64", "c128", "bf16", "f16"])
    case = dict(call=call, pattern=pattern, dtype=dtype, index=rng.choice(["i32", "i64"]), op="non")
    if spmm:
        case["n"] = _log_int(rng, 1, 256)
    if call != "coo_spmm" and call != "spmm_kept":
        case["op"] = rng.choice(["non", "non", "trans", "conj"])
    limit = _MAX_NNZ // max(1, _VALUE_BYTES[dtype] // 4)
    if spmm:
        limit = min(limit, _MAX_SPMM_WORK // (case["n"] * max(1, _VALUE_BYTES[dtype] // 4)))
    if coo:
        limit = min(limit, 1 << 24)
    if pattern == "rmat":
        case["edges"] = rng.randint(4, 24)
        case["scale"] = rng.randint(10, min(21, int(math.log2(limit / case["edges"]))))
    elif pattern == "stencil":
        top = min(128, int((limit / 27) ** (1 / 3)))
        for axis in ("nx", "ny", "nz"):
            case[axis] = _log_int(rng, 10, top)
    else:
        case["per_row"] = _log_int(rng, 4, 64)
        case["rows"] = _log_int(rng, 1000, min(4000000, limit // case["per_row"]))
        case["cols"] = max(200, int(case["rows"] * math.exp(rng.uniform(-1.0, 1.0))))
        if spmm:  # the dense operands stay within a few GB
            case["rows"] = min(case["rows"], (1 << 29) // case["n"])
            case["cols"] = min(case["cols"], (1 << 29) // case["n"])
    return case


# -- sizes -----------------------------------------------------------------------------


def _shape_nnz(case):
    if case["pattern"] == "rmat":
        n = 1 << case["scale"]
        return n, n, case["edges"] * n
    if case["pattern"] == "stencil":
        dims = [case[a] for a in ("nx", "ny", "nz")]
        n = dims[0] * dims[1] * dims[2]
        return n, n, math.prod(3 * d - 2 for d in dims)
    return case["rows"], case["cols"], case["rows"] * case["per_row"]


def work(case):
    """A, the dense operand and the result once each; a complex multiply-add is 8 flops."""
    m, k, nnz = _shape_nnz(case)
    n = case.get("n", 1)
    value, index = _VALUE_BYTES[case["dtype"]], _INDEX_BYTES[case["index"]]
    places = 2 * nnz if case["pattern"] == "scattered" else nnz + m + 1
    return {
        "bytes": nnz * value + places * index + (m + k) * n * value,
        "flops": (8 if case["dtype"] in ("c64", "c128") else 2) * nnz * n,
    }


# -- inputs ----------------------------------------------------------------------------


def _rand(shape, dtype, g):
    """Uniform in (-1, 1), both parts of a complex value."""
    if dtype.is_complex:
        real = torch.float32 if dtype == torch.complex64 else torch.float64
        return torch.complex(_rand(shape, real, g), _rand(shape, real, g))
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    return (torch.rand(shape, dtype=wide, device="cuda", generator=g) * 2 - 1).to(dtype)


def _row_pointer(case, rows, cols, nnz, g):
    """int64 row pointer of exactly nnz entries with the pattern's row lengths, none longer than a row."""
    if case["pattern"] == "uniform":
        return torch.arange(rows + 1, device="cuda") * (nnz // rows)
    u = torch.rand(rows, dtype=torch.float64, device="cuda", generator=g)
    if case["pattern"] == "ragged":
        weight = (u * 256).to(torch.int64)
    else:  # Pareto tail with exponent 2 over a floor, clipped
        weight = ((8 + 1 / (1 - u)).clamp(max=50000) * 64).to(torch.int64)
    total = torch.cumsum(weight, 0)
    ptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = (total.double() * (nnz / float(total[-1]))).round().to(torch.int64)
    ptr[-1] = nnz
    return ptr


def _csr(case, g):
    """(indices, indptr) in int64: columns ascending within each row."""
    rows, cols, nnz = _shape_nnz(case)
    if case["pattern"] == "rmat":
        row = torch.zeros(nnz, dtype=torch.int64, device="cuda")
        col = torch.zeros(nnz, dtype=torch.int64, device="cuda")
        for _ in range(case["scale"]):
            u = torch.rand(nnz, device="cuda", generator=g)
            row = row * 2 + (u >= 0.76)
            col = col * 2 + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
        key = torch.sort(row * cols + col)[0]
        starts = torch.arange(rows + 1, device="cuda") * cols
        return key % cols, torch.searchsorted(key, starts)
    if case["pattern"] == "stencil":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        r = torch.arange(rows, device="cuda")
        x, y, z = r // (ny * nz), r // nz % ny, r % nz
        offsets = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
        inside = torch.stack([(x + a >= 0) & (x + a < nx) & (y + b >= 0) & (y + b < ny) & (z + c >= 0) & (z + c < nz)
                              for a, b, c in offsets], 1)
        place = torch.stack([r + (a * ny + b) * nz + c for a, b, c in offsets], 1)
        ptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
        ptr[1:] = torch.cumsum(inside.sum(1), 0)
        return place[inside], ptr
    # one column in each of the row's equal strips of the width: distinct and ascending
    # (rows longer than the width repeat columns)
    ptr = _row_pointer(case, rows, cols, nnz, g)
    length = ptr[1:] - ptr[:-1]
    row = torch.repeat_interleave(torch.arange(rows, device="cuda"), length, output_size=nnz)
    slot = torch.arange(nnz, device="cuda") - ptr[row]
    u = torch.rand(nnz, dtype=torch.float64, device="cuda", generator=g)
    return ((slot + u) * (cols / length[row])).to(torch.int64).clamp_(max=cols - 1), ptr


def _operands(case, seed):
    """The call's own arguments: values, places and the dense operand."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    m, k, nnz = _shape_nnz(case)
    dtype, index = _DTYPES[case["dtype"]], _INDEX[case["index"]]
    if case["pattern"] == "scattered":
        places = (torch.randint(0, m, (nnz,), device="cuda", generator=g).to(index),
                  torch.randint(0, k, (nnz,), device="cuda", generator=g).to(index))
    else:
        indices, indptr = _csr(case, g)
        places = (indices.to(index), indptr.to(index))
    data = _rand((nnz,), dtype, g)
    inner = k if case["op"] == "non" else m
    dense = _rand((inner, case["n"]) if "n" in case else (inner,), dtype, g)
    return data, places, dense, (m, k)


def prepare(case, seed):
    data, places, dense, shape = _operands(case, seed)
    state = dict(call=case["call"], op=case["op"], dense=dense)
    if case["call"] == "spmv_kept":
        state["kept"] = fs.prepare_spmv_csr(data, *places, shape, op=case["op"])
    elif case["call"] == "spmm_kept":
        state["kept"] = fs.prepare_spmm_csr_route(data, *places, shape, op=case["op"])
    else:
        state.update(data=data, places=places, shape=shape)
    return state


def run(state):
    call, dense, op = state["call"], state["dense"], state["op"]
    if call == "spmv_kept":
        return fs.flagsparse_spmv_csr(x=dense, prepared=state["kept"])
    if call == "spmm_kept":
        return fs.flagsparse_spmm_csr_run(state["kept"], dense)
    data, (first, second), shape = state["data"], state["places"], state["shape"]
    if call == "spmv":
        return fs.flagsparse_spmv_csr(data, first, second, dense, shape, op=op)
    if call == "spmm":
        return fs.flagsparse_spmm_csr(data, first, second, dense, shape, op=op)
    if call == "coo_spmv":
        return fs.flagsparse_spmv_coo(data, first, second, dense, shape, op=op)
    return fs.flagsparse_spmm_coo(data, first, second, dense, shape)


# -- reference -------------------------------------------------------------------------

_CHUNK = 1 << 28  # gathered values at a time: 2 GB of float64


def exact(case, seed):
    """op(A) @ dense in float64 / complex128: entries sorted by result row, rows summed in
    segments.  The inputs are taken as they are, 16-bit values included."""
    data, places, dense, (m, k) = _operands(case, seed)
    if case["pattern"] == "scattered":
        row, col = places[0].long(), places[1].long()
    else:
        indptr = places[1].long()
        row = torch.repeat_interleave(torch.arange(m, device="cuda"), indptr[1:] - indptr[:-1])
        col = places[0].long()
    wide = torch.complex128 if data.dtype.is_complex else torch.float64
    data, dense = data.to(wide), dense.to(wide)
    rows = m
    if case["op"] != "non":
        row, col, rows = col, row, k
        if case["op"] == "conj":
            data = data.conj().resolve_conj()
    row, order = torch.sort(row, stable=True)
    col, data = col[order], data[order]
    vector = dense.ndim == 1
    if vector:
        dense = dense[:, None]
    n = dense.shape[1]
    parts = 2 if wide.is_complex else 1
    lengths = torch.bincount(row, minlength=rows)
    ends = torch.cumsum(lengths, 0).cpu().numpy()
    out = torch.zeros((rows, n), dtype=wide, device="cuda")
    step = max(1, _CHUNK // (n * parts))
    r0 = e0 = 0
    while r0 < rows:
        r1 = max(r0 + 1, int(np.searchsorted(ends, e0 + step, side="right")))
        r1, e1 = min(r1, rows), int(ends[min(r1, rows) - 1])
        if e1 > e0:
            term = data[e0:e1, None] * dense[col[e0:e1]]
            if parts == 2:
                term = torch.view_as_real(term).reshape(e1 - e0, 2 * n)
            total = torch.segment_reduce(term, "sum", lengths=lengths[r0:r1], axis=0, unsafe=True, initial=0)
            out[r0:r1] = torch.view_as_complex(total.reshape(r1 - r0, n, 2)) if parts == 2 else total
        r0, e0 = r1, e1
    return out[:, 0] if vector else out


def tolerance(case):
    """float32 / complex64 products are summed in float64 and rounded once (half an ulp:
    3e-8 of the result); float64 / complex128 sums carry a few rounding errors of their
    own; 16-bit results are rounded from float32 once."""
    return {
        "f16": {"rel": 8e-4, "max": 3e-3},
        "bf16": {"rel": 7e-3, "max": 2.5e-2},
        "f32": {"rel": 1.2e-7, "max": 4e-7},
        "c64": {"rel": 1.2e-7, "max": 4e-7},
        "f64": {"rel": 1e-15, "max": 1e-13},
        "c128": {"rel": 1e-15, "max": 1e-13},
    }[case["dtype"]]
