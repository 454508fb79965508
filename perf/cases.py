"""Measured cases of the VCSR-MC SpMM library: what its users have it do, through the public
Python entry points, over the range of sizes and options they use.

A case is a dict of plain values.  Its "path" is one of

  multiply   C += A.B or C = A.B with a format that is already built, the call a solver or a
             graph network repeats: DeviceFormat.launcher, bound once to B and C
  build      a new matrix on the device: DeviceFormat.from_device_csr, one multiply, close
  dropin     the reference's sequence on host arrays: csr_to_vcsr_mc, upload_vcsr_mc_device,
             run_vcsr_mc_spmm_gpu, destroy_vcsr_mc_device
  reorder    rcm_order_device, then apply_column_permutation_device on a copy of A, with B

Matrices are made on the GPU from the seed, of the structure classes of the library's benchmark
and corpus: "uniform" (Poisson row lengths, uniform columns), "powerlaw" (configuration model on
Zipf(2.1) degrees, symmetric), "stencil" (27-point grid), "grid" (2D 5-point grid), "block"
(32 x 32 dense blocks) and "rmat" ((0.57, 0.19, 0.19, 0.05), 16 edges per vertex).
"""
import math

import torch

import vcsr_mc_amd as vm

DEV = "cuda:0"


# ---- matrices -------------------------------------------------------------------------------
def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 8 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _from_pairs(r, c, M, N):
    """(row_ptr, col) of the distinct pairs, in row-major order."""
    key = torch.unique(r.to(torch.int64) * N + c)
    rows = key // N
    col = (key - rows * N).to(torch.int32)
    return _row_ptr(torch.bincount(rows, minlength=M)), col


def _row_ptr(counts):
    rp = torch.zeros(counts.numel() + 1, dtype=torch.int32, device=DEV)
    rp[1:] = torch.cumsum(counts, 0)
    return rp


def _uniform(case, g):
    M, N = case["rows"], case["cols"]
    k = torch.poisson(torch.full((M,), float(case["per_row"]), device=DEV), generator=g).long()
    r = torch.repeat_interleave(torch.arange(M, device=DEV), k)
    c = torch.randint(0, N, (r.numel(),), device=DEV, generator=g)
    return _from_pairs(r, c, M, N)


def _powerlaw(case, g):
    n, per_row, dmax = case["rows"], case["per_row"], 1383
    p = torch.arange(1, dmax + 1, device=DEV, dtype=torch.float64) ** -2.1
    z = 1 + torch.searchsorted(torch.cumsum(p, 0) / p.sum(),
                               torch.rand(n, device=DEV, generator=g, dtype=torch.float64))
    z = z.clamp(max=dmax).double()
    d = (z * (per_row * n / z.sum())).round().clamp(1, dmax).long()
    stubs = torch.repeat_interleave(torch.arange(n, device=DEV), d)
    stubs = stubs[torch.randperm(stubs.numel(), device=DEV, generator=g)]
    h = stubs.numel() // 2
    a, b = stubs[:h], stubs[h:2 * h]
    keep = a != b
    a, b = a[keep], b[keep]
    return _from_pairs(torch.cat([a, b]), torch.cat([b, a]), n, n)


def _offsets(side, steps):
    """(row_ptr, col) of a grid of sides `side` whose points are joined along `steps`."""
    n = math.prod(side)
    idx = torch.arange(n, device=DEV)
    at, rest = [], idx
    for s in reversed(side):
        at.insert(0, rest % s)
        rest = rest // s
    col = torch.empty((n, len(steps)), dtype=torch.int32, device=DEV)
    ok = torch.ones((n, len(steps)), dtype=torch.bool, device=DEV)
    for j, step in enumerate(steps):
        off = 0
        for a, s, d in zip(at, side, step):
            ok[:, j] &= (a + d >= 0) & (a + d < s)
            off = off * s + d
        col[:, j] = (idx + off).to(torch.int32)
    return _row_ptr(ok.sum(1)), col[ok]


def _stencil(case, g):
    steps = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
    return _offsets((case["side"],) * 3, steps)


def _grid(case, g):
    return _offsets((case["side"],) * 2, [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)])


def _block(case, g):
    # four blocks in each block row, one in each quarter of the block columns
    nb = case["block_rows"]
    n, q = 32 * nb, nb // 4
    start = torch.arange(4, device=DEV) * q
    bc = start + torch.randint(0, q, (nb, 4), device=DEV, generator=g)
    cols = (32 * bc[:, :, None] + torch.arange(32, device=DEV)).reshape(nb, 1, 128)
    col = cols.expand(nb, 32, 128).reshape(-1).to(torch.int32)
    return torch.arange(n + 1, device=DEV, dtype=torch.int32) * 128, col


def _rmat(case, g):
    n = 1 << case["scale"]
    r = torch.zeros(16 * n, dtype=torch.int64, device=DEV)
    c = torch.zeros_like(r)
    for _ in range(case["scale"]):
        u = torch.rand(r.numel(), device=DEV, generator=g)
        r = 2 * r + (u >= 0.76)
        c = 2 * c + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    return _from_pairs(r, c, n, n)


_MAKE = {"uniform": _uniform, "powerlaw": _powerlaw, "stencil": _stencil, "grid": _grid,
         "block": _block, "rmat": _rmat}


def _shape(case):
    """(M, N, about how many nonzeros, rows with nonzeros, columns with nonzeros)."""
    kind = case["matrix"]
    if kind == "uniform":
        M, N, k = case["rows"], case["cols"], case["per_row"]
        nnz = M * k
        return M, N, nnz, M * (1 - math.exp(-k)), N * (1 - math.exp(-nnz / N))
    if kind == "powerlaw":
        n = case["rows"]
        return n, n, n * case["per_row"], n, n
    if kind == "stencil":
        s = case["side"]
        return s ** 3, s ** 3, (3 * s - 2) ** 3, s ** 3, s ** 3
    if kind == "grid":
        s = case["side"]
        return s * s, s * s, 5 * s * s - 4 * s, s * s, s * s
    if kind == "block":
        n = 32 * case["block_rows"]
        return n, n, 128 * n, n, n * (1 - math.exp(-4))
    # duplicates take 19% (scale 12) down to 3% (scale 22) of the edges, and 0.72 down to 0.48 of
    # the vertices keep a nonzero
    s = case["scale"]
    n = 1 << s
    t = min(1.0, max(0.0, (s - 12) / 10))
    used = n * (0.72 - 0.24 * t)
    return n, n, int(16 * n * (0.81 + 0.16 * t)), used, used


def _matrix(case, seed):
    M, N = _shape(case)[:2]
    g = _gen(seed, 0)
    rp, col = _MAKE[case["matrix"]](case, g)
    if case["path"] == "reorder" and case["matrix"] in ("uniform", "powerlaw", "rmat"):
        # a number of entries that the case fixes, so that outputs have one size for every seed
        row = torch.repeat_interleave(torch.arange(M, device=DEV), (rp[1:] - rp[:-1]).long())
        at = torch.randperm(col.numel(), device=DEV, generator=g)[:int(0.8 * _shape(case)[2])]
        rp, col = _from_pairs(row[at], col[at].long(), M, N)
    elif case["path"] == "reorder" and case["matrix"] in ("stencil", "grid"):
        # a mesh as a mesher numbers it: its points in an order of their own
        new = torch.randperm(N, device=DEV, generator=g)
        row = torch.repeat_interleave(torch.arange(M, device=DEV), (rp[1:] - rp[:-1]).long())
        rp, col = _from_pairs(new[row], new[col.long()], M, N)
    val = torch.randn(col.numel(), device=DEV, generator=g)
    return M, N, rp, col, val


def _operands(case, M, N, seed):
    g = _gen(seed, 1)
    O = case["width"]
    B = torch.randn((N, O), device=DEV, generator=g)
    if case["operand"] == "half":
        B = B.half()
    return B, torch.randn((M, O), device=DEV, generator=g)


# ---- cases ----------------------------------------------------------------------------------
def _case(name, path, width, format="half", operand="half", add=True, segment=32, tile=128,
          **matrix):
    return dict(name=name, path=path, width=width, format=format, operand=operand, add=add,
                segment=segment, tile=tile, **matrix)


def listed():
    return [
        # The smallest benchmark workload: one launch of a few microseconds.
        _case("multiply uniform f32", "multiply", 128, "single", "single",
              matrix="uniform", rows=4096, cols=4096, per_row=16),
        # The headline workload: a mid-size graph, features in binary16.
        _case("multiply powerlaw f16", "multiply", 128,
              matrix="powerlaw", rows=36692, per_row=10),
        # The same graph as the reference's driver calls it: binary16 A, B still in float.
        _case("multiply powerlaw f16 B f32", "multiply", 128, "half", "single",
              matrix="powerlaw", rows=36692, per_row=10),
        # A feature width that is no multiple of a vector: rows of 200 bytes.
        _case("multiply powerlaw f16 ragged", "multiply", 100, add=False,
              matrix="powerlaw", rows=100000, per_row=12),
        # A narrow output (classes of a graph network), in float.
        _case("multiply rmat f32 narrow", "multiply", 16, "single", "single", add=False,
              matrix="rmat", scale=18),
        # A block of solver vectors on a 3D mesh.
        _case("multiply stencil f32", "multiply", 128, "single", "single",
              matrix="stencil", side=100),
        # Block-sparse weights, binary16 and float.
        _case("multiply block f16", "multiply", 256, add=False, matrix="block", block_rows=8192),
        _case("multiply block f32", "multiply", 256, "single", "single",
              matrix="block", block_rows=8192),
        # The largest benchmark workload: a graph whose B is far beyond every cache.
        _case("multiply rmat f16", "multiply", 128, matrix="rmat", scale=22),
        # The reference's own sequence on host arrays.
        _case("dropin powerlaw f16", "dropin", 128, "half", "single",
              matrix="powerlaw", rows=36692, per_row=10),
        # A new large matrix on the device, used once.
        _case("build stencil f32", "build", 128, "single", "single", add=False,
              matrix="stencil", side=100),
        # A mesh in a mesher's numbering, brought to a narrow band before the format is built.
        _case("reorder mesh", "reorder", 64, "single", "single", matrix="stencil", side=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_matrix(rng, small):
    """A matrix of the classes above; `small`: for paths that cost more per nonzero."""
    kind = rng.choice(("uniform", "powerlaw", "stencil", "grid", "block", "rmat"))
    if kind == "uniform":
        rows = _log_int(rng, 2000, 60000 if small else 130000)
        cols = rows if rng.random() < 0.5 else _log_int(rng, 2000, 130000)
        return dict(matrix=kind, rows=rows, cols=cols, per_row=rng.randint(3, 32))
    if kind == "powerlaw":
        return dict(matrix=kind, rows=_log_int(rng, 4000, 100000 if small else 200000),
                    per_row=rng.randint(6, 20))
    if kind == "stencil":
        return dict(matrix=kind, side=_log_int(rng, 16, 56 if small else 96))
    if kind == "grid":
        return dict(matrix=kind, side=_log_int(rng, 100, 300 if small else 1000))
    if kind == "block":
        return dict(matrix=kind, block_rows=_log_int(rng, 96, 1500 if small else 8000))
    return dict(matrix=kind, scale=rng.randint(12, 16 if small else 19))


def draw(rng):
    path = rng.choice(("multiply",) * 8 + ("build", "build", "dropin", "reorder"))
    format, operand = rng.choice((("single", "single"), ("half", "half"), ("half", "single")))
    if path == "dropin":
        operand = "single"
    if path == "reorder":
        format = operand = "single"
    width = rng.choice((32, 64, 128, 128, 256)) if rng.random() < 0.4 else _log_int(rng, 7, 256)
    case = _case(None, path, width, format, operand, add=path == "dropin" or rng.random() < 0.5,
                 segment=rng.choice((16, 32, 48, 64)), tile=rng.choice((64, 128, 128)),
                 **_draw_matrix(rng, path in ("dropin", "reorder")))
    del case["name"]
    return case


# ---- one pass -------------------------------------------------------------------------------
def prepare(case, seed):
    M, N, rp, col, val = _matrix(case, seed)
    state = {"case": case, "M": M, "N": N}
    if case["path"] == "reorder":
        B = _operands(case, M, N, seed)[0]
        state.update(rp=rp, col=col, val=val, B=B, B_out=torch.empty_like(B),
                     position=torch.empty(N, dtype=torch.int32, device=DEV))
        return state
    B, C = _operands(case, M, N, seed)
    state.update(B=B, C=C)
    if case["path"] == "dropin":
        state["csr"] = vm.CSR.from_arrays(rp.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy(),
                                          M, N)
    elif case["path"] == "build":
        state.update(rp=rp, col=col, val=val)
    else:
        fmt = vm.DeviceFormat.from_device_csr(rp, col, val, M, N, case["format"] == "single",
                                              case["segment"])
        state["format"] = fmt
        state["launch"] = fmt.launcher(B, C, tileK=case["tile"], overwrite=not case["add"])
    return state


def run(state):
    case = state["case"]
    if case["path"] == "multiply":
        state["launch"]()
        return {"C": state["C"]}
    if case["path"] == "build":
        fmt = vm.DeviceFormat.from_device_csr(state["rp"], state["col"], state["val"], state["M"],
                                              state["N"], case["format"] == "single",
                                              case["segment"])
        fmt.spmm(state["B"], state["C"], tileK=case["tile"], overwrite=not case["add"])
        fmt.close()
        return {"C": state["C"]}
    if case["path"] == "dropin":
        V = vm.csr_to_vcsr_mc(state["csr"], case["format"] == "single", case["segment"])
        vm.upload_vcsr_mc_device(V)
        vm.run_vcsr_mc_spmm_gpu(V, state["B"], case["width"], case["tile"], state["C"])
        vm.destroy_vcsr_mc_device()
        return {"C": state["C"]}
    vm.rcm_order_device(state["rp"], state["col"], state["M"], state["N"], state["position"])
    col, val = state["col"].clone(), state["val"].clone()
    vm.apply_column_permutation_device(state["rp"], col, val, state["M"], state["N"],
                                       state["position"], state["B"], state["B_out"],
                                       case["width"])
    return {"position": state["position"], "col": col, "val": val, "B": state["B_out"]}


def work(case):
    M, N, nnz, rows, cols = _shape(case)
    O = case["width"]
    if case["path"] == "reorder":
        # A read, its columns and values written again, the order, B moved
        return {"bytes": 16 * nnz + 4 * (M + 1) + 4 * N + 8 * N * O, "flops": 0}
    # the format keeps binary16 or float values; what is built from a float CSR reads float
    value = 4 if case["format"] == "single" or case["path"] != "multiply" else 2
    passes = 2 if case["add"] else 1  # C += A.B reads C too
    b = (value + 4) * nnz + 4 * (M + 1)
    b += cols * O * (2 if case["operand"] == "half" else 4) + passes * 4 * rows * O
    if case["path"] == "dropin":
        b += 8 * nnz  # the format's columns and values written for the caller
    return {"bytes": int(b), "flops": 2 * nnz * O}


def tolerance(case):
    if case["path"] == "reorder":
        return "exact"  # an order, and values moved
    # float: sums of products in another order.  binary16: A and B rounded to 11 bits
    return {"rel": 1e-6} if case["format"] == "single" else {"rel": 1e-3}


# ---- in 64 bits -----------------------------------------------------------------------------
def _product(rp, col, val, M, N, B, C0, add):
    """C0 + A.B (rows that A does not touch keep C0), a block of columns at a time."""
    A = torch.sparse_csr_tensor(rp.long(), col.long(), val.double(), size=(M, N))
    R = C0.double()
    untouched = (rp[1:] == rp[:-1])[:, None]
    for k in range(0, B.shape[1], 32):
        P = A @ B[:, k:k + 32].double()
        R[:, k:k + 32] = R[:, k:k + 32] + P if add else torch.where(untouched, R[:, k:k + 32], P)
    return R


def exact(case, seed):
    if case["path"] == "reorder":
        return None  # positions, and values that only move
    M, N, rp, col, val = _matrix(case, seed)
    B, C = _operands(case, M, N, seed)
    R = _product(rp, col, val, M, N, B, C, case["add"] or case["path"] == "dropin")
    return {"C": R}
