"""Performance cases of the SpMV engine.

Each case is one pass through a public entry point on a matrix that is
already resident on the GPU: single-vector SpMV in the storage formats
(y += A x), multi-vector SpMV, block SpMM on 16-bit values, a Cocktail pass
over a partitioned matrix, and a burst of requests through the serving loop.

Matrices come from the families that the engine's benchmark and tests use:
the 5-point Laplacian, the 27-point stencil, power-law rows (Zipf(1.8)
clipped to [1, 5000], random columns, optionally united with a band), dense
4x4 blocks at 12 block-column offsets, and a mesh-like matrix with 8..40
neighbours per row near the diagonal.  They are generated on the GPU from
the seed, converted with the library's own host conversions and uploaded.
"""

import ctypes
import math

import numpy as np
import torch

import clspmv_mic_amd as cs

DEV = "cuda"
DTYPES = {"f32": cs.DT_F32, "bf16": cs.DT_BF16, "f16": cs.DT_F16}
TORCH16 = {"bf16": torch.bfloat16, "f16": torch.float16}
BLOCK_OFFSETS = (0, 1, -1, 32, -32, 33, -33, 4096, -4096, 4097, -4097, 31)
BAND = (0, 1, -1, 1000, -1000)
ZIPF_S, ZIPF_MAX = 1.8, 5000
_context = None


def context():
    """The one context (device and stream) such a program has."""
    global _context
    if _context is None:
        _context = cs.Context(0)
    return _context


class Buffer:
    """A torch tensor as a device operand of the library (address, sizes)."""

    def __init__(self, t):
        self.t, self.p = t, ctypes.c_void_p(t.data_ptr())
        self.n, self.nbytes = t.numel(), t.numel() * t.element_size()


class _Raw:
    """The y of a Cocktail runtime as torch sees it (no copy): the tensor made
    from it keeps the runtime, which owns the memory."""

    def __init__(self, rt, n):
        self.rt, address = rt, cs.lib.clspmv_cocktail_gpu_res(rt.g)
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (address, False), "version": 2}


# ---- the cases -----------------------------------------------------------

def listed():
    return [
        # The reference's own flow (partition, upload, tune, do_spmv) on the
        # benchmark's small grid problem: launch latency is what it costs.
        dict(name="cocktail-laplace2d-256", op="cocktail", format="cocktail", matrix="laplace2d", n=256,
             values="f32"),
        # CSR on an ordinary 3-D discretisation with an odd number of rows.
        dict(name="csr-stencil27-77", op="spmv", format="csr", matrix="stencil27", n=77, values="f32"),
        # CSR as a caller uploads a graph: skewed rows, columns without locality.
        dict(name="csr-powerlaw-1M", op="spmv", format="csr", matrix="powerlaw", n=1_000_000, values="f32"),
        # The benchmark's stencil in the format the partitioner gives it.
        dict(name="dia-stencil27-128", op="spmv", format="dia", matrix="stencil27", n=128, values="f32"),
        # Diagonals in 16-bit storage, a ragged grid.
        dict(name="dia-bf16-stencil27-101", op="spmv", format="dia", matrix="stencil27", n=101, values="bf16"),
        # An unstructured mesh in slices.
        dict(name="sell-mesh-500009", op="spmv", format="sell", matrix="mesh", n=500_009, values="f32"),
        # Dense 4x4 blocks (several unknowns per node).
        dict(name="bcsr-block4x4-131072", op="spmv", format="bcsr", matrix="block", n=131_072, values="f32"),
        # The same flow on the benchmark's graph with a band.
        dict(name="cocktail-powerlaw-1M", op="cocktail", format="cocktail", matrix="powerlaw_band", n=1_000_000,
             values="f32"),
        # A block of right-hand sides on a stencil (block solvers, serving).
        dict(name="multi-dia-stencil27-96-k16", op="multi", format="dia", matrix="stencil27", n=96, values="f32",
             k=16),
        # A block of right-hand sides on a graph with 16-bit values.
        dict(name="multi-csr-bf16-powerlaw-600k-k8", op="multi", format="csr", matrix="powerlaw", n=600_011,
             values="bf16", k=8),
        # Mixed-precision block SpMM, the widest of the benchmark's blocks.
        dict(name="spmm-bf16-block4x4-k32", op="spmm", format="bspmm", matrix="block", n=262_144, values="bf16",
             k=32, layout="tiled", accumulate=False),
        # A burst of requests against resident matrices of mixed kinds.
        dict(name="serve-8x48", op="serve", format="mix", matrix="mix", n=400_000, matrices=8, requests=48,
             values="mix"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grid", "grid", "graph", "mesh", "mesh", "block", "multi", "multi", "spmm", "spmm", "cocktail",
                       "serve"])
    if kind == "grid":  # the formats a regular grid goes into
        matrix = rng.choice(["laplace2d", "stencil27"])
        n = _log_int(rng, 500, 1400) if matrix == "laplace2d" else _log_int(rng, 50, 110)
        fmt = rng.choice(["csr", "ell", "sell", "dia", "bdia"])
        values = rng.choice(["f32", "f32", "bf16", "f16"]) if fmt == "dia" else "f32"
        return dict(op="spmv", format=fmt, matrix=matrix, n=n, values=values)
    if kind == "graph":
        fmt = rng.choice(["csr", "coo"])
        values = rng.choice(["f32", "f32", "bf16", "f16"])
        return dict(op="spmv", format=fmt, matrix=rng.choice(["powerlaw", "powerlaw_band"]),
                    n=_log_int(rng, 30_000, 1_000_000), values=values)
    if kind == "mesh":
        return dict(op="spmv", format=rng.choice(["csr", "coo", "ell", "sell"]), matrix="mesh",
                    n=_log_int(rng, 20_000, 700_000), values="f32")
    if kind == "block":
        return dict(op="spmv", format=rng.choice(["bcsr", "bell", "sbell"]), matrix="block",
                    n=_log_int(rng, 20_000, 131_072), values="f32")
    if kind == "multi":
        values, k = rng.choice(["f32", "f32", "bf16", "f16"]), rng.randint(1, 16)
        matrix = rng.choice(["stencil27", "laplace2d", "powerlaw", "mesh"])
        if matrix in ("stencil27", "laplace2d"):
            n = _log_int(rng, 32, 96) if matrix == "stencil27" else _log_int(rng, 200, 900)
            return dict(op="multi", format=rng.choice(["dia", "dia", "csr"]), matrix=matrix, n=n, values=values, k=k)
        return dict(op="multi", format="csr", matrix=matrix, n=_log_int(rng, 10_000, 500_000), values=values, k=k)
    if kind == "spmm":
        return dict(op="spmm", format="bspmm", matrix="block", n=_log_int(rng, 9_000, 131_072),
                    values=rng.choice(["bf16", "f16"]), k=rng.randint(1, 32), layout=rng.choice(["tiled", "columns"]),
                    accumulate=rng.choice([True, False]))
    if kind == "cocktail":
        matrix = rng.choice(["powerlaw_band", "stencil27", "laplace2d", "block", "mesh"])
        n = {"powerlaw_band": _log_int(rng, 20_000, 400_000), "stencil27": _log_int(rng, 20, 90),
             "laplace2d": _log_int(rng, 100, 1000), "block": _log_int(rng, 9_000, 60_000),
             "mesh": _log_int(rng, 10_000, 200_000)}[matrix]
        return dict(op="cocktail", format="cocktail", matrix=matrix, n=n, values="f32")
    return dict(op="serve", format="mix", matrix="mix", n=_log_int(rng, 20_000, 300_000),
                matrices=rng.randint(3, 8), requests=rng.randint(12, 48), values="mix")


# ---- matrices, on the GPU ------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _unique(key, width):
    key = torch.unique(key)  # sorted: row-major order
    return (key // width), key % width


def _grid(n, dims, reach):
    """Rows and columns of the stencil of `reach` offsets on an n^dims grid,
    in (row, column) order."""
    m = n ** dims
    r = torch.arange(m, device=DEV)
    at = [(r // n ** d) % n for d in range(dims)]
    cols, ok = [], []
    for off in reach:  # ascending column offsets
        good = torch.ones(m, dtype=torch.bool, device=DEV)
        for d in range(dims):
            good &= (at[d] + off[d] >= 0) & (at[d] + off[d] < n)
        cols.append(r + sum(off[d] * n ** d for d in range(dims)))
        ok.append(good)
    ok = torch.stack(ok, 1)
    return r[:, None].expand(m, len(reach))[ok], torch.stack(cols, 1)[ok], m


def _zipf_cdf():
    k = np.arange(1, ZIPF_MAX, dtype=np.float64)
    return np.cumsum(k ** -ZIPF_S) / 1.8822296181028220  # zeta(1.8)


def make_matrix(kind, n, values, g):
    """(rows, cols, FP32 values, height, width), sorted by row and column;
    with 16-bit `values` the values are ones that the type holds."""
    if kind == "laplace2d":
        rows, cols, m = _grid(n, 2, [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)])
        vals = torch.where(rows == cols, 4.0, -1.0).float()
        return rows, cols, vals, m, m
    if kind == "stencil27":
        reach = [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
        rows, cols, m = _grid(n, 3, reach)
        vals = torch.randn(rows.numel(), generator=g, device=DEV)
        vals = torch.where(rows == cols, vals.abs() + 22.0, vals)  # dominant centre
    elif kind == "block":
        m = 4 * n
        br = torch.arange(n, device=DEV)
        bcol = (br[:, None] + torch.tensor(BLOCK_OFFSETS, device=DEV)[None, :]) % n
        bcol = torch.sort(bcol, 1).values
        e = torch.arange(4, device=DEV)
        rows = (4 * br[:, None, None, None] + e[None, :, None, None]).expand(n, 4, len(BLOCK_OFFSETS), 4)
        cols = (4 * bcol[:, None, :, None] + e[None, None, None, :]).expand(n, 4, len(BLOCK_OFFSETS), 4)
        rows, cols = rows.reshape(-1), cols.reshape(-1)
        vals = torch.randn(rows.numel(), generator=g, device=DEV)
    else:
        m = n
        if kind == "mesh":
            lens = torch.randint(8, 41, (m,), generator=g, device=DEV)
            near = int(3 * math.sqrt(m))
            rows = torch.repeat_interleave(torch.arange(m, device=DEV), lens)
            cols = (rows + torch.randint(-near, near + 1, (rows.numel(),), generator=g, device=DEV)).clamp_(0, m - 1)
            band = (0,)
        else:
            cdf = torch.from_numpy(_zipf_cdf()).to(DEV)
            u = torch.rand(m, generator=g, device=DEV, dtype=torch.float64)
            lens = torch.searchsorted(cdf, u).add_(1).clamp_(max=min(m, ZIPF_MAX))
            rows = torch.repeat_interleave(torch.arange(m, device=DEV), lens)
            cols = torch.randint(0, m, (rows.numel(),), generator=g, device=DEV)
            band = BAND if kind == "powerlaw_band" else ()
        keys = [rows * m + cols]
        for off in band:
            r = torch.arange(max(0, -off), min(m, m - off), device=DEV)
            keys.append(r * m + r + off)
        rows, cols = _unique(torch.cat(keys), m)
        vals = torch.randn(rows.numel(), generator=g, device=DEV)
    if values in TORCH16:
        vals = vals.to(TORCH16[values]).float()
    return rows, cols, vals, m, m


def _to_coo(rows, cols, vals, height, width):
    return cs.Coo(rows.int().cpu().numpy(), cols.int().cpu().numpy(), vals.cpu().numpy(), height, width)


def upload(coo, fmt, values):
    """The device matrix in `fmt`, as the library's conversions give it."""
    ctx, dt = context(), DTYPES[values]
    kw = {} if values == "f32" else {"dtype": dt}
    if fmt == "csr":  # the caller's own arrays, as clspmv_upload_csr keeps them
        return cs.DeviceMatrix(ctx, cs.coo2csr(coo), panel=0, **kw) if kw else cs.DeviceMatrix(ctx, cs.coo2csr(coo))
    if fmt == "coo":
        return cs.DeviceMatrix(ctx, coo, **kw)
    if fmt == "dia":
        return cs.DeviceMatrix(ctx, cs.coo2dia(coo), **kw)
    convert = {"ell": cs.coo2ell, "sell": cs.coo2sell, "bdia": cs.coo2bdia}.get(fmt)
    if convert:
        return cs.DeviceMatrix(ctx, convert(coo))
    if fmt == "sbell":
        return cs.DeviceMatrix(ctx, cs.coo2sbell(coo, 4, 4, cap=False))
    blocked = cs.coo2b4csr if fmt == "bcsr" else cs.coo2b4ell
    return cs.DeviceMatrix(ctx, blocked(coo, 4, 4, cap=False))


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV) * 2 - 1


def _round4(n):
    return (n + 3) // 4 * 4


def _vectors(case, g, height, width):
    """The dense operands of a case: X and the preloaded Y (a block SpMM's
    columns start at multiples of 4)."""
    if case["op"] == "multi":
        return _uniform(g, width, case["k"]), _uniform(g, case["k"], height)
    if case["op"] == "spmm":
        X = _uniform(g, case["k"], _round4(width)).to(TORCH16[case["values"]])
        X[:, width:] = 0
        return X, _uniform(g, case["k"], _round4(height))
    return _uniform(g, width), _uniform(g, height)


def _mix(case, seed):
    """Matrices and requests of a serving case: [(format, values, matrix)],
    [(matrix index, x)]; sizes log-uniform up to n rows, half stencils, half
    power-law, FP32 and BF16 in turn, 1..16 right-hand sides a request."""
    g = _generator(seed)
    shape = np.random.default_rng([case["n"], case["matrices"], case["requests"]])  # the mix itself: by the case
    mats = []
    for i in range(case["matrices"]):
        m = int(math.exp(shape.uniform(math.log(10_000), math.log(case["n"]))))
        values = "bf16" if (i // 2) % 2 else "f32"
        if i % 2:
            mats.append(("csr", values, make_matrix("powerlaw", m, values, g)))
        elif i % 4 == 0:
            mats.append(("dia", values, make_matrix("stencil27", max(4, round(m ** (1 / 3))), values, g)))
        else:
            mats.append(("dia", values, make_matrix("laplace2d", max(8, round(m ** 0.5)), values, g)))
    reqs = []
    for _ in range(case["requests"]):
        i, k = int(shape.integers(0, len(mats))), int(shape.integers(1, 17))
        reqs.append((i, _uniform(g, k, mats[i][2][4])))
    return mats, reqs


# ---- state, pass, work, exact values -------------------------------------

def prepare(case, seed):
    g = _generator(seed)
    if case["op"] == "serve":
        mats, reqs = _mix(case, seed)
        server = cs.Server(streams=4, max_batch=64, hbm_budget=1 << 30)
        ids = []
        for fmt, values, M in mats:
            coo = _to_coo(*M)
            dm = (cs.DeviceMatrix(context(), cs.coo2csr(coo), panel=cs.PANEL_BOTH, dtype=DTYPES[values])
                  if fmt == "csr" else upload(coo, fmt, values))
            ids.append(server.add(dm, kmax=16))
        todo = [(ids[i], x.shape[0], Buffer(x), Buffer(torch.zeros(x.shape[0], mats[i][2][3], device=DEV)))
                for i, x in reqs]
        torch.cuda.synchronize()
        return {"op": "serve", "server": server, "todo": todo, "out": [y.t for _, _, _, y in todo]}
    rows, cols, vals, height, width = make_matrix(case["matrix"], case["n"], case["values"], g)
    coo = _to_coo(rows, cols, vals, height, width)
    del rows, cols, vals
    X, Y = _vectors(case, g, height, width)
    state = {"op": case["op"]}
    if case["op"] == "cocktail":
        rt = cs.CocktailRuntime(cs.analyze_matrix(coo, cs.TABLES_DIR), X.cpu().numpy(), Y.cpu().numpy())
        rt.tune()
        rt.set_y(Y.cpu().numpy())  # tuning runs passes of its own
        state.update(rt=rt, out=torch.as_tensor(_Raw(rt, height), device=DEV))
    elif case["op"] == "spmm":
        state.update(A=cs.BlockSpmm(context(), cs.coo2bcsr(coo, 4, 4), DTYPES[case["values"]]), k=case["k"],
                     layout=case["layout"], accumulate=case["accumulate"], ldx=X.shape[1], ldy=Y.shape[1])
        if case["layout"] == "tiled":  # 4-row tiles: values of rows 4c..4c+3 of one column together
            X = X.reshape(case["k"], -1, 4).permute(1, 0, 2).contiguous()
        state.update(X=Buffer(X), Y=Buffer(Y), out=Y)
    else:
        state.update(A=upload(coo, case["format"], case["values"]), k=case.get("k", 1), ldy=height, X=Buffer(X),
                     Y=Buffer(Y), out=Y)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return state


def run(state):
    op = state["op"]
    if op == "spmv":
        state["A"].spmv(state["X"], state["Y"])
    elif op == "multi":
        state["A"].spmv_multi(state["k"], state["X"], state["Y"], state["ldy"])
    elif op == "spmm":
        if state["layout"] == "tiled":
            state["A"].spmm_tiled(state["k"], state["X"], state["Y"], state["ldy"], state["accumulate"])
        else:
            state["A"].spmm(state["k"], state["X"], state["ldx"], state["Y"], state["ldy"])
    elif op == "cocktail":
        state["rt"].do_spmv(1)
    else:
        server = state["server"]
        tickets = [server.submit(i, k, 0, x=x, device_y=y) for i, k, x, y in state["todo"]]
        for t in tickets:
            server.wait(t)
    return state["out"]


def _mean_zipf():
    k = np.arange(1, ZIPF_MAX, dtype=np.float64)
    p = k ** -ZIPF_S / 1.8822296181028220
    return float((k * p).sum() + ZIPF_MAX * (1 - p.sum()))


def _size(kind, n):
    """(rows, expected nonzeros) of a matrix."""
    if kind == "laplace2d":
        return n * n, 5 * n * n - 4 * n
    if kind == "stencil27":
        return n ** 3, (3 * n - 2) ** 3
    if kind == "block":
        return 4 * n, 16 * len(BLOCK_OFFSETS) * n
    if kind == "mesh":
        return n, 25 * n
    return n, int(_mean_zipf() * n) + (5 * n if kind == "powerlaw_band" else 0)


def _matrix_bytes(fmt, kind, n, value_bytes):
    m, nnz = _size(kind, n)
    if fmt in ("dia", "bdia"):
        return value_bytes * nnz
    if fmt in ("bcsr", "bell", "sbell", "bspmm") or (fmt == "cocktail" and kind == "block"):
        return value_bytes * nnz + 4 * (nnz // 16) + 4 * (n + 1)
    if fmt == "cocktail" and kind in ("stencil27", "laplace2d"):
        return 4 * nnz
    if fmt == "cocktail" and kind == "powerlaw_band":  # the band as diagonals
        return 8 * (nnz - 5 * n) + 4 * 5 * n + 4 * (m + 1)
    return (4 + value_bytes) * nnz + 4 * (m + 1)


def work(case):
    if case["op"] == "serve":
        shape = np.random.default_rng([case["n"], case["matrices"], case["requests"]])
        size = []
        for i in range(case["matrices"]):
            m = int(math.exp(shape.uniform(math.log(10_000), math.log(case["n"]))))
            kind = "powerlaw" if i % 2 else "stencil27" if i % 4 == 0 else "laplace2d"
            n = m if i % 2 else max(4, round(m ** (1 / 3))) if i % 4 == 0 else max(8, round(m ** 0.5))
            size.append((*_size(kind, n), _matrix_bytes("csr" if i % 2 else "dia", kind, n, 2 if (i // 2) % 2 else 4)))
        nbytes, flops, used = 0, 0, set()
        for _ in range(case["requests"]):
            i, k = int(shape.integers(0, len(size))), int(shape.integers(1, 17))
            used.add(i)
            nbytes += 8 * size[i][0] * k
            flops += 2 * size[i][1] * k
        return {"bytes": nbytes + sum(size[i][2] for i in used), "flops": flops}
    m, nnz = _size(case["matrix"], case["n"])
    k = case.get("k", 1)
    vb = 4 if case["values"] == "f32" else 2
    nbytes = _matrix_bytes(case["format"], case["matrix"], case["n"], vb)
    if case["op"] == "spmm":
        y = 4 if case["layout"] == "tiled" and not case["accumulate"] else 8
        nbytes += m * k * (2 + y)
    else:
        nbytes += m * k * (4 + 8)  # x read, y read and written
    return {"bytes": nbytes, "flops": 2 * nnz * k}


def _product64(rows, cols, vals, X, Y):
    """Y + A X in 64 bits, one column at a time: X (k, width), Y (k, height)."""
    v = vals.double()
    out = Y.double().clone()
    for q in range(out.shape[0]):
        out[q, :].index_add_(0, rows, v * X[q].double()[cols])
    return out


def exact(case, seed):
    if case["op"] == "serve":
        mats, reqs = _mix(case, seed)
        return [_product64(*mats[i][2][:3], x, torch.zeros(x.shape[0], mats[i][2][3], device=DEV)) for i, x in reqs]
    g = _generator(seed)
    rows, cols, vals, height, width = make_matrix(case["matrix"], case["n"], case["values"], g)
    X, Y = _vectors(case, g, height, width)
    if case["op"] == "multi":
        return _product64(rows, cols, vals, X.t(), Y)
    if case["op"] == "spmm":
        if case["layout"] == "tiled" and not case["accumulate"]:
            Y[:, :height] = 0
        return _product64(rows, cols, vals, X, Y)
    return _product64(rows, cols, vals, X[None], Y[None])[0]
