"""GPU parity of every storage format and kernel variant against the oracle.

Bar: |y_i - y64_i| <= 1e-5 * (|y0_i| + sum_j |a_ij x_j|) against the FP64
oracle, and bit-exact equality on dyadic inputs,
where every FP32 partial sum is exact so the summation order cannot matter.
All calls go through the C-ABI (libclspmv.so).
"""

import numpy as np
import pytest

import clspmv_mic_amd as cs
from clspmv_mic_amd import matrices

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _cases():
    return {
        "rand_small": matrices.random_sparse(300, 257, 0.03, seed=1),
        "rand_dyadic": matrices.random_sparse(513, 700, 0.02, seed=2, dyadic=True),
        "rand_empty_rows": matrices.random_sparse(1000, 1000, 0.01, seed=3, empty_rows=0.3),
        "rand_long_rows": matrices.random_sparse(2000, 3000, 0.002, seed=4, long_rows=5,
                                                 long_len=2500),
        "rand_long_dyadic": matrices.random_sparse(1500, 1500, 0.003, seed=5, dyadic=True,
                                                   long_rows=3, long_len=1400),
        # rows of up to ~1000 entries inside the short-row blocks (spanning
        # many stream chunks), empty rows, dyadic values
        "rand_mid_dyadic": matrices.random_sparse(3000, 2000, 0.002, seed=14, dyadic=True,
                                                  empty_rows=0.2, long_rows=6, long_len=1000),
        "lap2d_256": matrices.laplacian_2d(256),
        "stencil27_16": matrices.stencil_27pt(16, seed=3),
        "stencil27_dyadic": matrices.stencil_27pt(12, seed=5, dyadic=True),
        "block_small": matrices.block_stencil(700, 4, 4, seed=6, offsets=(0, 1, -1, 32, -33, 5)),
        "tall": matrices.random_sparse(3001, 97, 0.05, seed=7),
        "wide": matrices.random_sparse(97, 3001, 0.05, seed=8),
        "banded": matrices.banded(5000, (0, 1, -1, 2, 3, -7, 300, -300, 301, 302), seed=9),
        "banded_dyadic": matrices.banded(4099, (-2, -1, 0, 1, 5, 6, 7, 8, 1000), seed=10,
                                         dyadic=True),
    }


CASES = _cases()


def _is_dyadic(a: np.ndarray) -> bool:
    return bool(np.all(a * 64 == np.round(a * 64)))


def _run(ctx, oracle, A: cs.Coo, owned, method, panel=None, x_offset=0, dtype=None):
    dyadic = _is_dyadic(A.val)
    if dyadic:
        x = matrices.dyadic_vector(A.width, seed=11)
        y0 = matrices.dyadic_vector(A.height, seed=12)
    else:
        x = matrices.uniform_vector(A.width, seed=11)
        y0 = matrices.uniform_vector(A.height, seed=12)
    dA = cs.DeviceMatrix(ctx, owned, panel=panel, dtype=dtype)
    if panel is not None and panel > 0:
        assert dA.info.panel_width == panel and dA.info.panel_active == 1 and dA.info.plain == 0
    vals = A.val
    if dtype not in (None, cs.DT_F32):
        # The reference for 16-bit storage: the FP64 product of the values
        # as stored.
        assert dA.info.dtype == dtype
        vals = cs.convert_to_f32(cs.convert_from_f32(A.val, dtype), dtype)
    if x_offset:
        # x starting x_offset floats into its buffer: unaligned for 128-bit loads
        dx = cs.DeviceVector(ctx, A.width + x_offset, np.concatenate([np.zeros(x_offset, np.float32), x]))
        dx = dx.view(x_offset)
    else:
        dx = cs.DeviceVector(ctx, A.width, x)
    dy = cs.DeviceVector(ctx, A.height, y0)
    dA.spmv(dx, dy, method)
    ctx.sync()
    y = dy.download()
    y64, bound = oracle.spmv_f64(A.row, A.col, vals, x, A.height, y0)
    err, worst = oracle.scaled_error(y, y64, bound)
    assert err <= TOL, f"scaled error {err:.3e} at row {worst}: got {y[worst]} want {y64[worst]}"
    if dyadic:
        np.testing.assert_array_equal(y, y64.astype(np.float32))
    return y


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("method", [0, 1])
def test_csr(ctx, oracle, name, method):
    A = CASES[name]
    _run(ctx, oracle, A, cs.coo2csr(A.copy()), method)


@pytest.mark.parametrize("name", list(CASES))
def test_coo(ctx, oracle, name):
    A = CASES[name]
    _run(ctx, oracle, A, A.copy(), 0)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("method", [0, 1])
def test_ell(ctx, oracle, name, method):
    A = CASES[name]
    if name.startswith("rand_long"):
        pytest.skip("ELL of a matrix with 2500-entry rows is all padding")
    _run(ctx, oracle, A, cs.coo2ell(A.copy()), method)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("slice_height", [32, 128])
def test_sell(ctx, oracle, name, slice_height):
    A = CASES[name]
    for method in (0, 1):
        _run(ctx, oracle, A, cs.coo2sell(A, slice_height), method)


DIA_CASES = ["lap2d_256", "stencil27_16", "stencil27_dyadic", "block_small", "banded",
             "banded_dyadic"]


@pytest.mark.parametrize("name", DIA_CASES)
@pytest.mark.parametrize("method", [0, 1, 2, 3])
def test_dia(ctx, oracle, name, method):
    A = CASES[name]
    d = cs.coo2dia(A)
    if d is None:
        pytest.skip("DIA refused: padded size >= 2*nnz (include/matrix_storage.h:972)")
    offs = d.arrays()["off"]
    span = int(offs.max() - offs.min())
    if method >= 2 and (1024 if method == 3 else 256) + span > 8192:
        with pytest.raises(cs.ClspmvError):
            _run(ctx, oracle, A, d, method)
        return
    _run(ctx, oracle, A, d, method)


@pytest.mark.parametrize("name", DIA_CASES)
@pytest.mark.parametrize("method", [0, 1, 2, 3, 4])
def test_bdia(ctx, oracle, name, method):
    A = CASES[name]
    b = cs.coo2bdia(A)
    if b is None:
        pytest.skip("BDIA refused: padded size >= 2*nnz (include/matrix_storage.h:972)")
    _run(ctx, oracle, A, b, method)


BLOCK_CASES = ["block_small", "rand_small", "rand_dyadic", "lap2d_256", "tall", "wide"]


def _bcsr_slots(b) -> int:
    """Slots per block row of the slot-major BCSR encoding the upload picks
    (every block row at most 64 blocks, padding to the longest at most 10 %
    of the blocks), or 0 for the row-pointer encoding."""
    h, rp = b.header(), b.arrays()["rp"]
    nbr, nb = h["b4csr_row_num"], h["b4csr_block_num"]
    w = int(np.diff(rp).max()) if nbr else 0
    return w if nb > 0 and w <= 64 and w * nbr * 10 <= nb * 11 else 0


@pytest.mark.parametrize("name", BLOCK_CASES)
@pytest.mark.parametrize("shape", cs.BLOCK_SHAPES)
def test_bcsr(ctx, oracle, name, shape):
    """Both BCSR encodings (block_small and most lap2d shapes slot-major,
    the random matrices row-pointer) against the oracle."""
    A = CASES[name]
    bh, bw = shape
    b = cs.coo2b4csr(A.copy(), bw, bh)
    assert cs.DeviceMatrix(ctx, b).info.block_slots == _bcsr_slots(b)
    _run(ctx, oracle, A, b, 0)


def _ragged_blocks(bh, bw):
    """Dyadic block rows of 6 blocks, every 20th block row missing one (a
    padding slot in the slot-major encoding)."""
    A = matrices.block_stencil(900, bh, bw, seed=13, offsets=(0, 1, -1, 32, -33, 5), dyadic=True)
    brow, bcol = A.row // bh, A.col // bw
    drop = (brow % 20 == 7) & (bcol == (brow + 5) % 900)
    return cs.Coo(A.row[~drop], A.col[~drop], A.val[~drop], A.height, A.width)


@pytest.mark.parametrize("shape", [(4, 4), (2, 8), (8, 4), (1, 4)])
@pytest.mark.parametrize("x_offset", [0, 1])
def test_bcsr_slot_major_ragged(ctx, oracle, shape, x_offset):
    """Slot-major BCSR with padding slots: bit for bit the oracle's sum on
    dyadic data, with x aligned and unaligned for float4 loads."""
    bh, bw = shape
    A = _ragged_blocks(bh, bw)
    b = cs.coo2b4csr(A.copy(), bw, bh)
    hdr = b.header()
    assert 0 < _bcsr_slots(b) and _bcsr_slots(b) * hdr["b4csr_row_num"] > hdr["b4csr_block_num"]
    assert cs.DeviceMatrix(ctx, b).info.block_slots == _bcsr_slots(b)
    _run(ctx, oracle, A, b, 0, x_offset=x_offset)


@pytest.mark.parametrize("name", BLOCK_CASES)
@pytest.mark.parametrize("shape", cs.BLOCK_SHAPES)
def test_bell(ctx, oracle, name, shape):
    A = CASES[name]
    bh, bw = shape
    owned = cs.coo2b4ell(A.copy(), bw, bh)
    for method in (0, 1):
        _run(ctx, oracle, A, owned, method)


@pytest.mark.parametrize("name", BLOCK_CASES)
@pytest.mark.parametrize("shape", cs.BLOCK_SHAPES)
def test_sbell(ctx, oracle, name, shape):
    A = CASES[name]
    bh, bw = shape
    _run(ctx, oracle, A, cs.coo2sbell(A.copy(), bw, bh), 0)


def test_auto_method_every_format(ctx, oracle):
    A = CASES["stencil27_16"]
    for owned in [cs.coo2csr(A.copy()), A.copy(), cs.coo2ell(A.copy()), cs.coo2sell(A),
                  cs.coo2dia(A), cs.coo2bdia(A), cs.coo2b4csr(A.copy(), 4, 4),
                  cs.coo2b4ell(A.copy(), 4, 4), cs.coo2sbell(A.copy(), 4, 4)]:
        _run(ctx, oracle, A, owned, cs.METHOD_AUTO)


def test_empty_matrix(ctx):
    A = cs.Coo(np.zeros(0, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32), 10, 10)
    dA = cs.DeviceMatrix(ctx, cs.coo2csr(A))
    y0 = np.arange(10, dtype=np.float32)
    dx = cs.DeviceVector(ctx, 10, np.ones(10, np.float32))
    dy = cs.DeviceVector(ctx, 10, y0)
    dA.spmv(dx, dy, 0)
    ctx.sync()
    np.testing.assert_array_equal(dy.download(), y0)


def test_bad_method_rejected(ctx):
    A = CASES["rand_small"]
    dA = cs.DeviceMatrix(ctx, cs.coo2csr(A.copy()))
    dx = cs.DeviceVector(ctx, A.width, np.ones(A.width, np.float32))
    dy = cs.DeviceVector(ctx, A.height, np.zeros(A.height, np.float32))
    with pytest.raises(cs.ClspmvError):
        dA.spmv(dx, dy, 7)


def test_repeat_is_deterministic(ctx):
    """Same inputs, same kernel: bitwise identical results (no atomics)."""
    A = CASES["rand_long_rows"]
    x = matrices.uniform_vector(A.width, seed=3)
    for owned, m in [(cs.coo2csr(A.copy()), 1), (A.copy(), 0)]:
        dA = cs.DeviceMatrix(ctx, owned)
        dx = cs.DeviceVector(ctx, A.width, x)
        outs = []
        for _ in range(3):
            dy = cs.DeviceVector(ctx, A.height, np.zeros(A.height, np.float32))
            dA.spmv(dx, dy, m)
            ctx.sync()
            outs.append(dy.download())
        np.testing.assert_array_equal(outs[0], outs[1])
        np.testing.assert_array_equal(outs[0], outs[2])


PANEL_CASES = ["rand_small", "rand_dyadic", "rand_empty_rows", "rand_long_rows", "rand_long_dyadic",
               "lap2d_256", "tall", "wide", "banded_dyadic"]


@pytest.mark.parametrize("name", PANEL_CASES)
@pytest.mark.parametrize("pw", [8, 64, 1024, 32760])
@pytest.mark.parametrize("fmt", ["coo", "csr"])
def test_panel_encoding(ctx, oracle, name, pw, fmt):
    """x-panel encoding (16-bit in-panel columns, LDS-staged x) at widths from
    one to many panels, COO and CSR, both methods of CSR."""
    A = CASES[name]
    owned = A.sorted() if fmt == "coo" else cs.coo2csr(A.copy())
    if -(-A.width // pw) > 2048:  # more panels than the encoding holds
        with pytest.raises(cs.ClspmvError) as e:
            cs.DeviceMatrix(ctx, owned, panel=pw)
        assert e.value.code == cs.ERR_UNSUPPORTED
        return
    for method in ([0] if fmt == "coo" else [0, 1]):
        _run(ctx, oracle, A, owned, method, panel=pw)


@pytest.mark.parametrize("fmt", ["coo", "csr"])
def test_panel_unaligned_x(ctx, oracle, fmt):
    A = CASES["rand_long_rows"]
    owned = A.sorted() if fmt == "coo" else cs.coo2csr(A.copy())
    _run(ctx, oracle, A, owned, 0, panel=64, x_offset=1)


def test_panel_both_encodings_switch(ctx, oracle):
    """PANEL_BOTH keeps both encodings; each gives the oracle's result."""
    A = matrices.random_sparse(3000, 70000, 0.002, seed=21, long_rows=4, long_len=3000)
    for fmt in ("coo", "csr"):
        owned = A.sorted() if fmt == "coo" else cs.coo2csr(A.copy())
        x = matrices.uniform_vector(A.width, seed=11)
        y64, bound = oracle.spmv_f64(A.row, A.col, A.val, x, A.height)
        dA = cs.DeviceMatrix(ctx, owned, panel=cs.PANEL_BOTH)
        assert dA.info.panel_width > 0 and dA.info.plain == 1
        for use in (True, False):
            dA.set_panel(use)
            dx = cs.DeviceVector(ctx, A.width, x)
            dy = cs.DeviceVector(ctx, A.height, np.zeros(A.height, np.float32))
            dA.spmv(dx, dy, 0)
            ctx.sync()
            err, worst = oracle.scaled_error(dy.download(), y64, bound)
            assert err <= TOL, f"{fmt} panel={use}: {err:.3e} at {worst}"


def test_panel_bad_width_rejected(ctx):
    A = CASES["rand_small"].sorted()
    for bad in (4, 12, 32768, -3):
        with pytest.raises(cs.ClspmvError):
            cs.DeviceMatrix(ctx, A, panel=bad)


@pytest.mark.parametrize("name", DIA_CASES)
@pytest.mark.parametrize("method", [0, 1, 2, 3])
@pytest.mark.parametrize("dtype", [cs.DT_BF16, cs.DT_F16])
def test_dia_16bit_values(ctx, oracle, name, method, dtype):
    """DIA with values stored in BF16 / FP16, accumulated in FP32."""
    A = CASES[name]
    d = cs.coo2dia(A)
    if d is None:
        pytest.skip("DIA refused: padded size >= 2*nnz (include/matrix_storage.h:972)")
    offs = d.arrays()["off"]
    if method >= 2 and (1024 if method == 3 else 256) + int(offs.max() - offs.min()) > 8192:
        pytest.skip("offset span too wide for the LDS window")
    _run(ctx, oracle, A, d, method, dtype=dtype)


@pytest.mark.parametrize("name", ["rand_small", "rand_dyadic", "rand_long_dyadic", "lap2d_256", "wide"])
@pytest.mark.parametrize("dtype", [cs.DT_BF16, cs.DT_F16])
@pytest.mark.parametrize("fmt", ["coo", "csr"])
def test_panel_16bit_values(ctx, oracle, name, dtype, fmt):
    A = CASES[name]
    owned = A.sorted() if fmt == "coo" else cs.coo2csr(A.copy())
    _run(ctx, oracle, A, owned, 0, panel=64, dtype=dtype)
    _run(ctx, oracle, A, owned, 0, dtype=dtype)  # automatic panel width


def test_16bit_needs_panel(ctx):
    A = CASES["rand_small"]
    for panel in (0, cs.PANEL_BOTH):
        with pytest.raises(cs.ClspmvError):
            cs.DeviceMatrix(ctx, A.sorted(), panel=panel, dtype=cs.DT_BF16)


MULTI_CASES = ["rand_small", "rand_dyadic", "rand_long_rows", "rand_long_dyadic", "rand_mid_dyadic", "lap2d_256",
               "stencil27_dyadic", "banded", "tall", "wide"]


@pytest.mark.parametrize("name", MULTI_CASES)
@pytest.mark.parametrize("fmt", ["dia", "csr"])
@pytest.mark.parametrize("dtype", [cs.DT_F32, cs.DT_BF16, cs.DT_F16])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 8, 12, 16])
def test_spmv_multi(ctx, oracle, name, fmt, dtype, k):
    """One pass for k right-hand sides (X row-major, Y column-major) equals k
    oracle SpMVs; 16-bit values are compared with the values as stored."""
    A = CASES[name]
    if fmt == "dia" and A.height != A.width:
        pytest.skip("DIA conversion is defined for square matrices")
    owned = cs.coo2dia(A) if fmt == "dia" else cs.coo2csr(A.copy())
    if owned is None:
        pytest.skip("DIA refused: padded size >= 2*nnz (include/matrix_storage.h:972)")
    dyadic = _is_dyadic(A.val)
    rng = np.random.default_rng(k)
    if dyadic:
        X = (rng.integers(-64, 65, size=(A.width, k)) / 64.0).astype(np.float32)
        Y0 = (rng.integers(-64, 65, size=(k, A.height + 3)) / 64.0).astype(np.float32)
    else:
        X = rng.uniform(-1, 1, size=(A.width, k)).astype(np.float32)
        Y0 = rng.uniform(-1, 1, size=(k, A.height + 3)).astype(np.float32)
    ldy = A.height + 3
    dA = cs.DeviceMatrix(ctx, owned, panel=0 if fmt == "csr" else None, dtype=dtype)
    vals = A.val if dtype == cs.DT_F32 else cs.convert_to_f32(cs.convert_from_f32(A.val, dtype), dtype)
    dX = cs.DeviceVector(ctx, X.size, X.reshape(-1))
    dY = cs.DeviceVector(ctx, Y0.size, Y0.reshape(-1))
    dA.spmv_multi(k, dX, dY, ldy)
    ctx.sync()
    Y = dY.download().reshape(k, ldy)
    for q in range(k):
        y64, bound = oracle.spmv_f64(A.row, A.col, vals, X[:, q].copy(), A.height, Y0[q, :A.height].copy())
        err, worst = oracle.scaled_error(Y[q, :A.height].copy(), y64, bound)
        assert err <= TOL, f"rhs {q}: {err:.3e} at row {worst}"
        if dyadic:
            np.testing.assert_array_equal(Y[q, :A.height], y64.astype(np.float32))
        np.testing.assert_array_equal(Y[q, A.height:], Y0[q, A.height:])

DIA_TILE_OFFSETS = {
    "runs_and_lone": [-7, -1, 0, 1, 9],
    "lone": [-30, -9, 0, 4, 11, 25],
    "many_runs": [-29, -28, -27, -20, -19, -18, -17, -16, -15, -14, -9, -8, -3, -2, -1, 0, 1, 5, 7, 8, 9, 15],
}


@pytest.mark.parametrize("offsets", sorted(DIA_TILE_OFFSETS))
@pytest.mark.parametrize("n,ks", [(33, range(1, 17)), (64, range(1, 17)), (257, range(1, 17)), (1030, (2, 5, 8, 11, 16)),
                                  ((1 << 15) + 5, (9, 12, 15, 16)), ((1 << 19) + 37, (1, 2, 3, 4, 7, 8, 13))])
def test_dia_multi_tiles(ctx, offsets, n, ks):
    """The multi-vector DIA kernel at the edges of its row tiles, over runs of
    consecutive offsets and lone ones, on operands aligned to one float only:
    dyadic inputs, so every sum is exact and equals the FP64 product."""
    off = DIA_TILE_OFFSETS[offsets]
    A = matrices.banded(n, off, seed=n, dyadic=True)
    dtypes = [cs.DT_F32, cs.DT_BF16] if n < 2000 else [cs.DT_F32]
    # The DIA struct by hand: coo2dia refuses short diagonals of a small matrix.
    length = cs.lib.clspmv_aligned_length(n, cs.GPU_ALIGNMENT)
    data, o32 = np.zeros((len(off), length), np.float32), np.array(off, np.int32)
    for j, o in enumerate(off):
        at = A.col.astype(np.int64) - A.row == o
        data[j, A.row[at]] = A.val[at]
    m = cs.DiaMatrix(cs.MatInfo(n, n, A.nnz), len(off), n, length, cs._ip(o32), cs._fp(data))
    dAs = [cs.DeviceMatrix(ctx, m, dtype=dt) for dt in dtypes]
    rng = np.random.default_rng(n)
    for k in ks:
        X = (rng.integers(-64, 65, size=(n, k)) / 64.0).astype(np.float32)
        Y0 = (rng.integers(-64, 65, size=(k, n + 1)) / 64.0).astype(np.float32)
        ref = Y0.astype(np.float64)
        for o in off:
            r0, r1 = max(0, -o), min(n, n - o)
            v = A.val[A.col.astype(np.int64) - A.row == o].astype(np.float64)
            ref[:, r0:r1] += v * X[r0 + o:r1 + o].T
        dX = cs.DeviceVector(ctx, X.size + 1, np.concatenate([[0.0], X.reshape(-1)]).astype(np.float32)).view(1)
        for dA in dAs:
            dY = cs.DeviceVector(ctx, Y0.size + 1, np.concatenate([[0.0], Y0.reshape(-1)]).astype(np.float32))
            dA.spmv_multi(k, dX, dY.view(1), n + 1)
            ctx.sync()
            np.testing.assert_array_equal(dY.download()[1:].reshape(k, n + 1), ref.astype(np.float32))

def _dia_by_hand(n, off, align=32, seed=5):
    """A DIA struct with the diagonals `off` full of dyadic values (zero outside
    the matrix), and the arrays that it refers to."""
    length = cs.lib.clspmv_aligned_length(n, align)
    rng = np.random.default_rng(seed)
    data, o32 = np.zeros((len(off), length), np.float32), np.array(off, np.int32)
    for j, o in enumerate(off):
        r0, r1 = max(0, -o), min(n, n - o)
        data[j, r0:r1] = rng.integers(-64, 65, r1 - r0) / 64.0
    m = cs.DiaMatrix(cs.MatInfo(n, n, int(np.count_nonzero(data))), len(off), n, length, cs._ip(o32), cs._fp(data))
    return m, data, o32


def _dia_product(data, off, n, X, Y):
    """Y (k, n) + A X (n, k) in FP64."""
    out = Y.astype(np.float64)
    for j, o in enumerate(off):
        r0, r1 = max(0, -o), min(n, n - o)
        out[:, r0:r1] += data[j, r0:r1].astype(np.float64) * X[r0 + o:r1 + o].T
    return out


@pytest.mark.parametrize("n", [39_999, 99_999, 100_003, 200_000, 240_001, 300_007, 600_011])
@pytest.mark.parametrize("name, offsets", [("three", [-9, 0, 11]), ("six", [-300, -9, 0, 11, 30, 4000]),
                                           ("seven", [-400, -20, -9, 0, 11, 30, 4000]),
                                           ("runs", [-301, -300, -299, -1, 0, 1, 299, 300, 301]),
                                           ("thirty", [i * 17 for i in range(-15, 15)])])
def test_dia_multi_routes(ctx, name, offsets, n):
    """The multi-vector DIA kernels, staging and direct, at the row and segment
    counts where the choice between them lies; dyadic inputs, exact sums, X and Y
    aligned to one float only."""
    m, data, _ = _dia_by_hand(n, offsets)
    rng = np.random.default_rng(n)
    dAs = [cs.DeviceMatrix(ctx, m, dtype=dt) for dt in (cs.DT_F32, cs.DT_F16)]
    for k in (1, 2, 3, 4, 7, 8, 13):
        X = (rng.integers(-64, 65, size=(n, k)) / 64.0).astype(np.float32)
        Y0 = (rng.integers(-64, 65, size=(k, n + 1)) / 64.0).astype(np.float32)
        ref = Y0.astype(np.float64)
        ref[:, :n] = _dia_product(data, offsets, n, X, Y0[:, :n])
        dX = cs.DeviceVector(ctx, X.size + 1, np.concatenate([[0.0], X.reshape(-1)]).astype(np.float32)).view(1)
        for dA in dAs:
            dY = cs.DeviceVector(ctx, Y0.size + 1, np.concatenate([[0.0], Y0.reshape(-1)]).astype(np.float32))
            dA.spmv_multi(k, dX, dY.view(1), n + 1)
            ctx.sync()
            np.testing.assert_array_equal(dY.download()[1:].reshape(k, n + 1), ref.astype(np.float32))


def _csr_wave_case(name):
    """Dyadic matrices at the edges of the CSR wave kernel: rows at its 512
    entries, runs of empty rows, blocks of 64 rows, and scattered columns in
    narrow windows (staged in LDS), some of them too wide."""
    rng = np.random.default_rng(11)
    if name == "row_lengths":
        width = 6000
        lens = np.concatenate([[0, 1, 512, 513, 0, 0, 3, 511, 1, 600, 5000], np.zeros(130, int), np.ones(200, int),
                               [2, 510, 256, 256, 1, 511, 4096, 4097], rng.integers(0, 20, 300), [0]])
        rows = np.repeat(np.arange(lens.size), lens)
        cols = np.concatenate([np.sort(rng.choice(width, n, replace=False)) for n in lens])
        height = lens.size
    else:
        height = width = 20_001
        lens = rng.integers(8, 41, height)
        rows = np.repeat(np.arange(height), lens)
        cols = np.clip(rows + rng.integers(-900, 901, rows.size), 0, width - 1)
        if name == "windows_some_wide":
            cols[(rows // 50) % 200 == 7] = rng.integers(0, width, int(((rows // 50) % 200 == 7).sum()))
        key = np.unique(rows.astype(np.int64) * width + cols)
        rows, cols = key // width, key % width
    vals = (rng.integers(-64, 65, rows.size) / 64.0).astype(np.float32)
    return cs.Coo(rows.astype(np.int32), cols.astype(np.int32), vals, height, width)


@pytest.mark.parametrize("name", ["row_lengths", "windows", "windows_some_wide"])
@pytest.mark.parametrize("dtype", [cs.DT_F32, cs.DT_BF16, cs.DT_F16])
@pytest.mark.parametrize("x_offset", [0, 1])
def test_csr_wave(ctx, oracle, name, dtype, x_offset):
    """Method 1 (and the automatic method) on dyadic inputs: every partial sum
    is exact, so y equals the FP64 product bit for bit."""
    A = _csr_wave_case(name)
    for method in (1, cs.METHOD_AUTO):
        _run(ctx, oracle, A, cs.coo2csr(A.copy()), method, panel=0, x_offset=x_offset, dtype=dtype)

@pytest.mark.parametrize("name", ["windows", "windows_some_wide"])
@pytest.mark.parametrize("fmt", ["ell", "sell"])
@pytest.mark.parametrize("x_offset", [0, 1])
@pytest.mark.parametrize("repeat", [1, 7])
def test_ell_windows(ctx, oracle, name, fmt, x_offset, repeat):
    """ELL and SELL with x windows in LDS, some work-groups without one, below
    and above the row count where the slots in flight change (`repeat` copies
    of the matrix along the diagonal); dyadic inputs, exact sums."""
    A = _csr_wave_case(name)
    if repeat > 1:
        i = np.arange(repeat, dtype=np.int32)[:, None]
        A = cs.Coo((A.row[None] + i * A.height).ravel(), (A.col[None] + i * A.width).ravel(),
                   np.tile(A.val, repeat), A.height * repeat, A.width * repeat)
    for owned in ([cs.coo2ell(A)] if fmt == "ell" else [cs.coo2sell(A, 32), cs.coo2sell(A, 700)]):
        _run(ctx, oracle, A, owned, 0, x_offset=x_offset)


@pytest.mark.parametrize("chunks", [40, 511, 512, 513])
@pytest.mark.parametrize("x_offset", [0, 1])
def test_staged_x(ctx, oracle, chunks, x_offset):
    """CSR, ELL and SELL work-groups of up to 512 rows of 11 entries (the last one
    partial) that touch `chunks` runs of 16 columns, up to the most that are
    staged and one past it, the last run cut off by the matrix; odd slot
    counts, an empty slice, slices that reach into two work-groups; dyadic
    inputs, exact sums."""
    rows, cols = 3 * 512 + 37, chunks * 16 - 5
    r = np.repeat(np.arange(rows), 11)
    c = np.minimum((np.arange(r.size) * 7 % chunks) * 16 + r % 16, cols - 1)
    key = np.unique(r.astype(np.int64) * cols + c)
    r, c = key // cols, key % cols
    v = (np.random.default_rng(chunks).integers(1, 65, r.size) / 64.0).astype(np.float32)
    A = cs.Coo(r.astype(np.int32), c.astype(np.int32), v, rows, cols)
    odd = (r % 16 != 3) & (r // 32 != 2) | (r % 8 == 1) & (r // 32 != 2)  # a slice of none
    B = cs.Coo(A.row[odd], A.col[odd], A.val[odd], rows, cols)
    _run(ctx, oracle, A, cs.coo2csr(A.copy()), cs.METHOD_AUTO, panel=0, x_offset=x_offset)
    for M, owned in ((A, cs.coo2ell(A)), (B, cs.coo2sell(B, 32)), (A, cs.coo2sell(A, 48)), (B, cs.coo2sell(B, 700))):
        _run(ctx, oracle, M, owned, 0, x_offset=x_offset)
    info = cs.DeviceMatrix(ctx, cs.coo2ell(A)).info
    assert (info.device_bytes >= 10 * info.stored) == (chunks <= 512)


@pytest.mark.parametrize("chunks", [127, 128, 129, 256, 257, 384, 511, 512, 513])
@pytest.mark.parametrize("fmt", ["csr", "csr_bf16", "ell", "sell"])
def test_staged_x_rounds(ctx, oracle, fmt, chunks):
    """Staged x with exactly `chunks` runs of 16 columns in every work-group, in
    one to four rounds of its loads, up to the most that are staged (and one past
    it: none are), the last run cut off by the matrix and a last partial
    work-group; dyadic inputs, exact sums."""
    csr = fmt.startswith("csr")
    per_row = 32 if csr else 8  # 4,096 entries a work-group: 8 blocks of 16 rows, or 512 rows
    groups, rows = 390, 390 * (4096 // per_row) + 37
    cols = chunks * 16 - 5
    r = np.repeat(np.arange(rows), per_row)
    i = np.arange(r.size)
    chunk = (i * 11 + i // 4096 * 5) % chunks  # 11 shares no factor with the counts: all of them, distinct in a row
    c = np.minimum(chunk * 16 + (i * 7) % 16, cols - 1)
    key = np.unique(r.astype(np.int64) * cols + c)
    assert key.size == r.size and all(np.unique(chunk[g * 4096:(g + 1) * 4096]).size == chunks for g in (0, 7, groups - 1))
    v = (np.random.default_rng(chunks).integers(1, 65, r.size) / 64.0).astype(np.float32)
    A = cs.Coo(r.astype(np.int32), (key % cols).astype(np.int32), v, rows, cols)
    dtype = cs.DT_BF16 if fmt == "csr_bf16" else cs.DT_F32
    owned = cs.coo2csr(A.copy()) if csr else cs.coo2ell(A) if fmt == "ell" else cs.coo2sell(A, 48)
    kw = dict(panel=0, dtype=dtype) if csr else {}
    for x_offset in (0, 1):
        _run(ctx, oracle, A, owned, 1 if csr else 0, x_offset=x_offset, **kw)
    info = cs.DeviceMatrix(ctx, owned, **kw).info
    own = (6 if fmt == "csr_bf16" else 8) * info.stored
    assert (info.device_bytes >= own + 2 * info.stored) == (chunks <= 512)


@pytest.mark.parametrize("chunks", [40, 301])
@pytest.mark.parametrize("x_offset", [0, 1])
def test_staged_x_slices(ctx, oracle, chunks, x_offset):
    """ELL and SELL with staged x where the launch takes it (101 work-groups, the
    last one partial): odd slot counts, empty slices beside full ones, slices that
    reach into two work-groups; dyadic inputs, exact sums."""
    rows, cols = 100 * 512 + 37, chunks * 16 - 5
    r = np.repeat(np.arange(rows), 11)
    c = np.minimum((np.arange(r.size) * 13 % chunks) * 16 + r % 16, cols - 1)
    key = np.unique(r.astype(np.int64) * cols + c)
    r, c = key // cols, key % cols
    v = (np.random.default_rng(chunks).integers(1, 65, r.size) / 64.0).astype(np.float32)
    A = cs.Coo(r.astype(np.int32), c.astype(np.int32), v, rows, cols)
    keep = (r // 32 % 9 != 2) & ((r % 16 != 3) | (c // 16 % 2 == 0))  # slices of none, rows of fewer
    B = cs.Coo(A.row[keep], A.col[keep], A.val[keep], rows, cols)
    for M, owned in ((A, cs.coo2ell(A)), (B, cs.coo2ell(B)), (B, cs.coo2sell(B, 32)), (A, cs.coo2sell(A, 48)),
                     (B, cs.coo2sell(B, 48)), (B, cs.coo2sell(B, 700))):
        _run(ctx, oracle, M, owned, 0, x_offset=x_offset)
        info = cs.DeviceMatrix(ctx, owned).info
        assert info.device_bytes >= 10 * info.stored


@pytest.mark.parametrize("groups, near, staged", [(639, 1, False), (640, 1, True), (383, 7, False), (384, 7, True)])
def test_staged_x_short_rows(ctx, oracle, groups, near, staged):
    """Five slots a row: where consecutive rows' columns follow each other x is
    staged from more work-groups of 512 rows on; exact sums on both sides."""
    rows = (groups - 1) * 512 + 200
    off = np.array([-700, -1, 0, 1, 700])
    r = np.repeat(np.arange(rows), 5)
    c = r + np.tile(off, rows) + (np.arange(rows) % near * 40)[r]
    ok = (c >= 0) & (c < rows)
    v = (np.random.default_rng(near).integers(1, 65, r.size) / 64.0).astype(np.float32)
    A = cs.Coo(r[ok].astype(np.int32), c[ok].astype(np.int32), v[ok], rows, rows)
    for owned in (cs.coo2ell(A), cs.coo2sell(A, 32)):
        _run(ctx, oracle, A, owned, 0)
        info = cs.DeviceMatrix(ctx, owned).info
        assert (info.device_bytes >= 10 * info.stored) == staged


def test_staged_x_with_panels(ctx, oracle):
    """A CSR upload that keeps its own arrays stages x for them (2 bytes an entry
    beside the 8 of columns and values), with panels beside them too."""
    A = matrices.banded(60_000, list(range(-13, 14)), seed=3, dyadic=True)
    csr = cs.coo2csr(A.copy())
    own, panels, both = (cs.DeviceMatrix(ctx, csr, panel=p).info for p in (0, cs.PANEL_AUTO, cs.PANEL_BOTH))
    assert own.plain and both.plain and both.panel_active and not panels.plain
    assert own.device_bytes >= 10 * A.nnz
    assert both.device_bytes - panels.device_bytes >= 10 * A.nnz
    for p in (0, cs.PANEL_AUTO, cs.PANEL_BOTH):
        _run(ctx, oracle, A, csr, 1, panel=p)


@pytest.mark.parametrize("width", [1, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 24, 27])
@pytest.mark.parametrize("rows", [100, (1 << 17) + 3])
def test_ell_slot_groups(ctx, oracle, width, rows):
    """Row widths around the groups of slots in flight, both group sizes, SELL
    slices of different widths in one wave; dyadic inputs, exact sums."""
    rng = np.random.default_rng(width)
    lens = np.where(np.arange(rows) % 64 < 32, width, width // 2)
    r = np.repeat(np.arange(rows), lens)
    first = np.cumsum(lens) - lens
    c = np.minimum(r, rows - 40) + (np.arange(r.size) - first[r])  # consecutive columns, distinct per row
    A = cs.Coo(r.astype(np.int32), c.astype(np.int32), (rng.integers(-64, 65, r.size) / 64.0).astype(np.float32),
               rows, rows)
    _run(ctx, oracle, A, cs.coo2ell(A), cs.METHOD_AUTO)
    _run(ctx, oracle, A, cs.coo2sell(A, 32), cs.METHOD_AUTO)


@pytest.mark.parametrize("rows, width", [(65, w) for w in (1, 2, 3, 4, 7, 9, 10, 15, 17, 23, 24, 31, 32, 33, 48, 49, 64)] +
                         [((1 << 17) - 1, 9), ((1 << 17) - 1, 12)] +
                         [((1 << 17) + 3, w) for w in (2, 3, 4, 9, 10, 23, 24, 25, 33)])
def test_ell_gathered(ctx, oracle, rows, width):
    """ELL and SELL without staged x (columns anywhere) at the mean row lengths
    where the work-group and the slots in flight change; slices of 32 rows, of
    a multiple of it and of neither, of different widths; dyadic inputs, exact
    sums."""
    rng = np.random.default_rng(width)
    lens = np.where(np.arange(rows) % 64 < 32, width, max(1, width - 3))
    cols = 50_000
    r = np.repeat(np.arange(rows), lens)
    first = np.repeat(np.cumsum(lens) - lens, lens)
    c = (rng.integers(0, cols, rows)[r] + (np.arange(r.size) - first) * 769) % cols  # distinct in a row
    o = np.lexsort((c, r))
    A = cs.Coo(r.astype(np.int32), c[o].astype(np.int32), (rng.integers(-64, 65, r.size) / 64.0).astype(np.float32),
               rows, cols)
    _run(ctx, oracle, A, cs.coo2ell(A), 0)
    for h in (32, 96, 40):
        _run(ctx, oracle, A, cs.coo2sell(A, h), cs.METHOD_AUTO)


@pytest.mark.parametrize("height", [1, 8, 20, 32, 100])
@pytest.mark.parametrize("rows, least", [(5_003, 3), (5_003, 12), (200_003, 3)])
def test_skewed_slices(ctx, oracle, rows, least, height):
    """SELL and SBELL slices of few rows whose widths differ a lot within a wave,
    empty ones and a first wave of none among them: a row adds nothing of the
    wave's widest, infinite x that only that one has included; dyadic inputs,
    exact sums."""
    rng = np.random.default_rng(least)
    lens = np.minimum((least / rng.random(rows) ** 0.9).astype(int), 150)
    lens[rng.random(rows) < 0.2] = 0
    lens[:80] = 0
    lens[3_000] = 160
    cols = 50_000
    r = np.repeat(np.arange(rows), lens)
    at = np.arange(r.size) - np.repeat(np.cumsum(lens) - lens, lens)
    c = (rng.integers(0, cols, rows)[r] + at * 769) % cols  # distinct in a row
    o = np.lexsort((c, r))
    A = cs.Coo(r.astype(np.int32), c[o].astype(np.int32), (rng.integers(-64, 65, r.size) / 64.0).astype(np.float32),
               rows, cols + 8)
    _run(ctx, oracle, A, cs.coo2sell(A, height), 0)
    for bw, bh in ((4, 1), (4, 4), (8, 2)):
        _run(ctx, oracle, A, cs.coo2sbell(A.copy(), bw, bh, height, cap=False), 0)
    last = (A.row == 3_000).nonzero()[0][-1]
    A.col[last], A.val[last] = cols + 3, 1.0
    x = matrices.dyadic_vector(cols + 8, seed=11)
    x[cols + 3] = np.inf
    dx, dy = cs.DeviceVector(ctx, cols + 8, x), cs.DeviceVector(ctx, rows, np.zeros(rows, np.float32))
    cs.DeviceMatrix(ctx, cs.coo2sell(A, height)).spmv(dx, dy, 0)
    ctx.sync()
    y = dy.download()
    assert np.isinf(y[3_000]) and np.isfinite(np.delete(y, 3_000)).all()


@pytest.mark.parametrize("nbr", [(3 << 15) - 1, 3 << 15, (3 << 16) - 1, (3 << 16) + 77])
@pytest.mark.parametrize("shape, width", [((4, 1), 5), ((4, 2), 2), ((4, 4), 3), ((8, 2), 1)])
def test_block_walks(ctx, oracle, nbr, shape, width):
    """Block rows of width and width - 1 blocks on both sides of the block-row
    counts where the kernels' walk over the slots changes; dyadic inputs, exact
    sums."""
    bw, bh = shape
    lens = np.where(np.arange(nbr) % 12 == 5, width - 1, width)
    br = np.repeat(np.arange(nbr), lens)
    bc = (br + 3 * (np.arange(br.size) - (np.cumsum(lens) - lens)[br])) % nbr
    bc = bc[np.lexsort((bc, br))]
    r = (br[:, None, None] * bh + np.arange(bh)[:, None] + np.zeros(bw, int)).reshape(-1)
    c = (bc[:, None, None] * bw + np.zeros((bh, 1), int) + np.arange(bw)).reshape(-1)
    o = np.argsort(r, kind="stable")
    v = (np.random.default_rng(nbr).integers(-64, 65, o.size) / 64.0).astype(np.float32)
    A = cs.Coo(r[o].astype(np.int32), c[o].astype(np.int32), v, nbr * bh, nbr * bw)
    _run(ctx, oracle, A, cs.coo2b4csr(A.copy(), bw, bh), 0)
    for m in (0, 1):
        _run(ctx, oracle, A, cs.coo2b4ell(A.copy(), bw, bh), m)
    _run(ctx, oracle, A, cs.coo2sbell(A.copy(), bw, bh), 0)


@pytest.mark.parametrize("rows, lens", [(30_000, 2), (30_000, 3), (262_143, 2), (262_144, 2), (20_000, 26), (20_000, 27),
                                        (8_000, 64), (8_000, 65), (300, 300)])
@pytest.mark.parametrize("skew", [False, True])
def test_csr_auto(ctx, oracle, rows, lens, skew):
    """The automatic CSR method around the sizes where it changes kernels, with
    rows of equal lengths and with one long one; dyadic inputs, exact sums."""
    n = np.full(rows, lens)
    if skew:
        n[rows // 2] = 9 * max(lens, 4)
    r = np.repeat(np.arange(rows), n)
    first = np.repeat(np.cumsum(n) - n, n)
    width = 9 * 65 + rows
    c = (r + (np.arange(r.size) - first)) % width
    o = np.lexsort((c, r))
    A = cs.Coo(r.astype(np.int32), c[o].astype(np.int32),
               (np.random.default_rng(lens).integers(-64, 65, r.size) / 64.0).astype(np.float32), rows, width)
    for dtype in (cs.DT_F32, cs.DT_F16):
        for method in (cs.METHOD_AUTO, 1):
            _run(ctx, oracle, A, cs.coo2csr(A.copy()), method, panel=0, dtype=dtype)


@pytest.mark.parametrize("dtype", [cs.DT_F32, cs.DT_BF16])
@pytest.mark.parametrize("others", [0, 1, 2, 15, 31, 32, 62, 63])
def test_csr_wide_rows(ctx, oracle, others, dtype):
    """Rows around the wave kernel's bound for rows summed by the whole wave
    (64, 65, 128, ... entries beside `others` rows of up to two, in front of
    and behind them; several in a block), longer ones of mixed lengths among
    them; dyadic inputs, exact sums."""
    lens = []
    for wide in (63, 64, 65, 127, 128, 129, 256, 257, 300, 511, 512, 513, 700, 600):
        lens += [wide] + [j % 3 for j in range(others)] + [wide]
    lens += [65, 70, 0, 66, 100, 1, 3, 65]
    rng = np.random.default_rng(others)
    r = np.repeat(np.arange(len(lens)), lens)
    c = np.concatenate([np.sort(rng.choice(900, n, replace=False)) for n in lens])
    A = cs.Coo(r.astype(np.int32), c.astype(np.int32), (rng.integers(-64, 65, r.size) / 64.0).astype(np.float32),
               len(lens), 900)
    _run(ctx, oracle, A, cs.coo2csr(A.copy()), cs.METHOD_AUTO, panel=0, dtype=dtype)


@pytest.mark.parametrize("shape", [(4, 1), (4, 2), (4, 4), (4, 8), (8, 1), (8, 4), (8, 8)])
@pytest.mark.parametrize("width", [1, 2, 3, 4, 5, 7, 8, 9, 12, 13])
def test_block_slot_groups(ctx, oracle, shape, width):
    """Block rows of width and width - 1 blocks around the groups of slots in
    flight, SBELL slices of different widths (one empty) in one wave, rows and
    columns that are no multiple of the block; dyadic inputs, exact sums."""
    bw, bh = shape
    rng = np.random.default_rng(width)
    nbr = 131
    lens = np.where(np.arange(nbr) % 12 == 5, width - 1, width)
    br = np.repeat(np.arange(nbr), lens)
    bc = br + np.arange(br.size) - (np.cumsum(lens) - lens)[br]  # consecutive block columns
    r = (br[:, None, None] * bh + np.arange(bh)[:, None] + np.zeros(bw, int)).reshape(-1)
    c = (bc[:, None, None] * bw + np.zeros((bh, 1), int) + np.arange(bw)).reshape(-1)
    o = np.lexsort((c, r))
    rows, cols = nbr * bh - bh // 2, (nbr + width - 1) * bw - 3
    o = o[(r[o] < rows) & (c[o] < cols)]
    A = cs.Coo(r[o].astype(np.int32), c[o].astype(np.int32), (rng.integers(-64, 65, o.size) / 64.0).astype(np.float32),
               rows, cols)
    b = cs.coo2b4csr(A.copy(), bw, bh)
    assert _bcsr_slots(b) == width
    _run(ctx, oracle, A, b, 0)
    for m in (0, 1):
        _run(ctx, oracle, A, cs.coo2b4ell(A.copy(), bw, bh), m)
    keep = (r[o] // bh) // 32 != 1  # block rows 32..63 empty: an empty slice beside a full one
    E = cs.Coo(A.row[keep], A.col[keep], A.val[keep], rows, cols)
    _run(ctx, oracle, E, cs.coo2sbell(E.copy(), bw, bh), 0)


@pytest.mark.parametrize("dtype", [cs.DT_F32, cs.DT_BF16])
@pytest.mark.parametrize("x_offset", [0, 1])
def test_csr_multi_units(ctx, dtype, x_offset):
    """The multi-vector CSR kernel on rows around its blocks and units (empty
    rows, rows of 7..17, 511..513, 4096, 4097 and 5000 entries) for every k:
    dyadic inputs, so Y equals the FP64 product, and each right-hand side's
    bits on random inputs do not depend on k."""
    A = _csr_wave_case("row_lengths")
    dA = cs.DeviceMatrix(ctx, cs.coo2csr(A.copy()), panel=0, dtype=dtype)
    R = cs.Coo(A.row, A.col, np.random.default_rng(3).standard_normal(A.nnz).astype(np.float32), A.height, A.width)
    dR = cs.DeviceMatrix(ctx, cs.coo2csr(R.copy()), panel=0, dtype=dtype)
    rng = np.random.default_rng(5)
    Xd = (rng.integers(-64, 65, size=(A.width, 16)) / 64.0).astype(np.float32)
    Xr = rng.uniform(-1, 1, size=(A.width, 16)).astype(np.float32)
    Y0 = (rng.integers(-64, 65, size=(16, A.height)) / 64.0).astype(np.float32)
    ref = Y0.astype(np.float64)
    for q in range(16):
        np.add.at(ref[q], A.row, A.val.astype(np.float64) * Xd[A.col, q])

    def run(m, X, k):
        pad = np.zeros(x_offset, np.float32)
        dX = cs.DeviceVector(ctx, X[:, :k].size + x_offset, np.concatenate([pad, X[:, :k].reshape(-1)])).view(x_offset)
        dY = cs.DeviceVector(ctx, k * A.height, Y0[:k].reshape(-1))
        m.spmv_multi(k, dX, dY, A.height)
        ctx.sync()
        return dY.download().reshape(k, A.height)

    wide = run(dR, Xr, 16)
    for k in range(1, 17):
        np.testing.assert_array_equal(run(dA, Xd, k), ref[:k].astype(np.float32))
        np.testing.assert_array_equal(run(dR, Xr, k), wide[:k])

@pytest.mark.parametrize("dtype", [cs.DT_F32, cs.DT_F16])
@pytest.mark.parametrize("medium", [4095, 4096, 4100])
def test_csr_multi_long_rows(ctx, medium, dtype):
    """Rows longer than a block (single-vector FP32 and multi-vector kernels), by a
    wave or a work-group each as their number decides, around the kernels' rounds (513, 576, 577, 1024, 2047..2049 and
    longer), and blocks of rows of 0..4 entries, which have a path of their own up
    to four right-hand sides: dyadic inputs, so Y equals the FP64 product, and
    each right-hand side's bits on random inputs do not depend on k."""
    rng = np.random.default_rng(medium)
    width = 6000
    lens = np.concatenate([rng.choice([513, 514, 576, 577, 640, 1024, 2047, 2048], medium), rng.integers(0, 5, 3000),
                           [2049, 4096, 4097, 5000, 4, 5, 0, 3], rng.integers(0, 3, 700)])
    rng.shuffle(lens)
    r = np.repeat(np.arange(lens.size), lens)
    first = np.repeat(np.cumsum(lens) - lens, lens)
    c = np.sort((rng.integers(0, width, lens.size)[r] + np.arange(r.size) - first) % width + r * np.int64(width)) % width
    Ad = cs.Coo(r.astype(np.int32), c.astype(np.int32), (rng.integers(-8, 9, r.size) / 8.0).astype(np.float32),
                lens.size, width)
    Ar = cs.Coo(Ad.row, Ad.col, rng.standard_normal(r.size).astype(np.float32), lens.size, width)
    dA, dR = (cs.DeviceMatrix(ctx, cs.coo2csr(m.copy()), panel=0, dtype=dtype) for m in (Ad, Ar))
    Xd = (rng.integers(-8, 9, size=(width, 16)) / 8.0).astype(np.float32)
    Xr = rng.uniform(-1, 1, size=(width, 16)).astype(np.float32)
    Y0 = (rng.integers(-8, 9, size=(16, lens.size)) / 8.0).astype(np.float32)
    import scipy.sparse as sp
    S = sp.csr_matrix((Ad.val.astype(np.float64), (Ad.row, Ad.col)), shape=(lens.size, width))
    ref = Y0 + (S @ Xd.astype(np.float64)).T

    def run(m, X, k):
        dX = cs.DeviceVector(ctx, k * width, np.ascontiguousarray(X[:, :k]).reshape(-1))
        dY = cs.DeviceVector(ctx, k * lens.size, Y0[:k].reshape(-1))
        m.spmv_multi(k, dX, dY, lens.size)
        ctx.sync()
        return dY.download().reshape(k, lens.size)

    dx, dy = cs.DeviceVector(ctx, width, Xd[:, 3].copy()), cs.DeviceVector(ctx, lens.size, Y0[3])
    dA.spmv(dx, dy, 1)
    ctx.sync()
    np.testing.assert_array_equal(dy.download(), ref[3].astype(np.float32))
    wide = run(dR, Xr, 16)
    for k in (1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16):
        np.testing.assert_array_equal(run(dA, Xd, k), ref[:k].astype(np.float32))
        np.testing.assert_array_equal(run(dR, Xr, k), wide[:k])


@pytest.mark.parametrize("offsets", [[-900, -30, 0, 31, 1000], [-900, -30, -2, 0, 31, 1000],
                                     [a + b * 40 for b in range(-4, 5) for a in (-1, 0, 1)],
                                     [a + b * 40 for b in range(-4, 5) for a in (-1, 0, 1)][:-1],
                                     [a + b * 40 for b in range(-4, 6) for a in (-1, 0, 1)]])
@pytest.mark.parametrize("n", [(15 << 16) - 1, (15 << 16) + 37, (7 << 18) + 1])
def test_dia_quad_segments(ctx, offsets, n):
    """16-bit DIA at the segment counts where a lane takes four rows or one:
    five and six lone diagonals, nine and ten full runs, nine with one cut short;
    dyadic inputs, exact sums."""
    m, data, _ = _dia_by_hand(n, offsets)
    x, y0 = matrices.dyadic_vector(n, seed=11), matrices.dyadic_vector(n, seed=12)
    ref = _dia_product(data, offsets, n, x[:, None], y0[None])
    dA = cs.DeviceMatrix(ctx, m, dtype=cs.DT_BF16)
    dx, dy = cs.DeviceVector(ctx, n, x), cs.DeviceVector(ctx, n, y0)
    dA.spmv(dx, dy, 0)
    ctx.sync()
    np.testing.assert_array_equal(dy.download(), ref[0].astype(np.float32))


@pytest.mark.parametrize("offsets", sorted(DIA_TILE_OFFSETS))
@pytest.mark.parametrize("n,align", [((3 << 18) - 1, 32), ((3 << 18) + 37, 32), ((3 << 18) + 37, 1),
                                     ((1 << 21) + 5, 32)])
@pytest.mark.parametrize("dtype", [cs.DT_F16, cs.DT_BF16])
def test_dia_quad(ctx, offsets, n, align, dtype):
    """DIA method 0 at and around the row count from which a lane takes four
    rows, and with a stored length that is no multiple of 4; dyadic inputs on
    vectors aligned to one float only: y equals the FP64 product."""
    off = DIA_TILE_OFFSETS[offsets]
    A = matrices.banded(n, off, seed=7, dyadic=True)
    length = cs.lib.clspmv_aligned_length(n, align)
    data, o32 = np.zeros((len(off), length), np.float32), np.array(off, np.int32)
    diff = A.col.astype(np.int64) - A.row
    x, y0 = matrices.dyadic_vector(n, seed=11), matrices.dyadic_vector(n, seed=12)
    ref = y0.astype(np.float64)
    for j, o in enumerate(off):
        at = diff == o
        data[j, A.row[at]] = A.val[at]
        ref[A.row[at]] += A.val[at].astype(np.float64) * x[A.col[at]]
    m = cs.DiaMatrix(cs.MatInfo(n, n, A.nnz), len(off), n, length, cs._ip(o32), cs._fp(data))
    dA = cs.DeviceMatrix(ctx, m, dtype=dtype)
    dx = cs.DeviceVector(ctx, n + 1, np.concatenate([[0], x]).astype(np.float32))
    dy = cs.DeviceVector(ctx, n + 1, np.concatenate([[0], y0]).astype(np.float32))
    dA.spmv(dx.view(1), dy.view(1), 0)
    ctx.sync()
    np.testing.assert_array_equal(dy.download()[1:], ref.astype(np.float32))


@pytest.mark.parametrize("name", ["rand_small", "rand_dyadic", "rand_long_rows"])
@pytest.mark.parametrize("dtype", [cs.DT_BF16, cs.DT_F16])
def test_csr_16bit_values(ctx, oracle, name, dtype):
    """CSR's own arrays with 16-bit values through clspmv_spmv (every method)."""
    A = CASES[name]
    for method in (0, 1):
        _run(ctx, oracle, A, cs.coo2csr(A.copy()), method, panel=0, dtype=dtype)


@pytest.mark.parametrize("dtype", [cs.DT_BF16, cs.DT_F16])
def test_csr_16bit_both_encodings(ctx, oracle, dtype):
    """16-bit CSR values in both encodings: the panel SpMV, the plain SpMV
    after clspmv_dmat_set_panel(0), and a multi-vector pass each match the
    oracle on the values as stored."""
    A = matrices.random_sparse(20000, 30000, 0.0005, seed=12, long_rows=4, long_len=5000)
    vals = cs.convert_to_f32(cs.convert_from_f32(A.val, dtype), dtype)
    dA = cs.DeviceMatrix(ctx, cs.coo2csr(A.copy()), panel=cs.PANEL_BOTH, dtype=dtype)
    assert dA.info.plain == 1 and dA.info.panel_active == 1 and dA.info.dtype == dtype
    x = matrices.uniform_vector(A.width, seed=3)
    y0 = matrices.uniform_vector(A.height, seed=4)
    y64, bound = oracle.spmv_f64(A.row, A.col, vals, x, A.height, y0)
    dx = cs.DeviceVector(ctx, A.width, x)
    for panel in (True, False):
        dA.set_panel(panel)
        assert dA.info.panel_active == int(panel)
        y = cs.DeviceVector(ctx, A.height, y0)
        dA.spmv(dx, y)
        ctx.sync()
        err, worst = oracle.scaled_error(y.download(), y64, bound)
        assert err <= TOL, f"panel={panel}: {err:.3e} at row {worst}"
    k = 4
    X = np.random.default_rng(5).uniform(-1, 1, size=(A.width, k)).astype(np.float32)
    dY = cs.DeviceVector(ctx, k * A.height, np.zeros(k * A.height, np.float32))
    dA.spmv_multi(k, cs.DeviceVector(ctx, X.size, X.reshape(-1)), dY, A.height)
    ctx.sync()
    Y = dY.download().reshape(k, A.height)
    for q in range(k):
        y64q, bq = oracle.spmv_f64(A.row, A.col, vals, X[:, q].copy(), A.height)
        err, worst = oracle.scaled_error(Y[q].copy(), y64q, bq)
        assert err <= TOL, f"rhs {q}: {err:.3e} at row {worst}"


def test_panel_block_with_many_long_rows(ctx, oracle):
    """Pass-2 blocks holding more than 1024 rows of more than 8 slots (the
    long-row list then takes more than one round of the work-group)."""
    # Every row: one entry in each of 10 distinct panels (of 16), so 10 slots.
    rng = np.random.default_rng(17)
    n, pw = 700_000, 4096
    r = np.repeat(np.arange(n, dtype=np.int64), 10)
    j = np.tile(np.arange(10, dtype=np.int64), n)
    cols = ((r + 3 * j) % 16) * pw + rng.integers(0, pw, size=r.size)
    A = cs.Coo(r, cols, rng.standard_normal(r.size).astype(np.float32), n, 16 * pw).sorted()
    dA = cs.DeviceMatrix(ctx, cs.coo2csr(A.copy()), panel=pw)
    assert dA.info.panel_active == 1
    assert n / dA.info.panel_blocks > 1024  # more than 1024 long rows per block
    x = matrices.uniform_vector(A.width, seed=5)
    y0 = matrices.uniform_vector(A.height, seed=6)
    y = cs.DeviceVector(ctx, A.height, y0)
    dA.spmv(cs.DeviceVector(ctx, A.width, x), y)
    ctx.sync()
    y64, bound = oracle.spmv_f64(A.row, A.col, A.val, x, A.height, y0)
    err, worst = oracle.scaled_error(y.download(), y64, bound)
    assert err <= TOL, f"{err:.3e} at row {worst}"


def test_panel_row_too_long_falls_back(ctx, oracle):
    """A row whose segments exceed one pass-2 block: an explicit panel width
    is refused, the automatic choice keeps the plain arrays; both give the
    oracle's result where they run."""
    rng = np.random.default_rng(23)
    # About n_long / 512 segments (one per sub-chunk) against 16384 per
    # pass-2 block.
    n_long = 9_000_000
    rows = np.concatenate([np.zeros(n_long, np.int64), rng.integers(1, 2000, size=20000)])
    cols = rng.integers(0, 4_000_000, size=rows.size)
    A = cs.Coo(rows, cols, rng.standard_normal(rows.size).astype(np.float32), 2000, 4_000_000).sorted()
    with pytest.raises(cs.ClspmvError):
        cs.DeviceMatrix(ctx, A, panel=32760)
    dA = cs.DeviceMatrix(ctx, A, panel=cs.PANEL_AUTO)
    assert dA.info.panel_active == 0 and dA.info.plain == 1
    x = matrices.uniform_vector(A.width, seed=5)
    y = cs.DeviceVector(ctx, A.height, np.zeros(A.height, np.float32))
    dA.spmv(cs.DeviceVector(ctx, A.width, x), y)
    ctx.sync()
    y64, bound = oracle.spmv_f64(A.row, A.col, A.val, x, A.height)
    err, worst = oracle.scaled_error(y.download(), y64, bound)
    assert err <= TOL, f"{err:.3e} at row {worst}"


def test_spmv_multi_refuses_other_formats(ctx):
    A = CASES["rand_small"]
    dA = cs.DeviceMatrix(ctx, cs.coo2ell(A.copy()))
    dX = cs.DeviceVector(ctx, A.width * 2)
    dY = cs.DeviceVector(ctx, A.height * 2)
    with pytest.raises(cs.ClspmvError):
        dA.spmv_multi(2, dX, dY, A.height)


@pytest.mark.parametrize("fmt", ["dia", "csr"])
def test_time_spmv_multi_accumulates(ctx, oracle, fmt):
    """clspmv_time_spmv_multi runs warmup + ntimes passes into the same Y: on
    dyadic data Y = Y0 + (warmup + ntimes) A X exactly, and the time is
    positive."""
    A = CASES["stencil27_dyadic"]
    owned = cs.coo2dia(A) if fmt == "dia" else cs.coo2csr(A.copy())
    k, warmup, ntimes = 5, 2, 3
    rng = np.random.default_rng(8)
    X = (rng.integers(-8, 9, size=(A.width, k)) / 8.0).astype(np.float32)
    Y0 = (rng.integers(-8, 9, size=(k, A.height)) / 8.0).astype(np.float32)
    dA = cs.DeviceMatrix(ctx, owned, panel=0 if fmt == "csr" else None)
    dY = cs.DeviceVector(ctx, Y0.size, Y0.reshape(-1))
    ms = dA.time_multi(k, cs.DeviceVector(ctx, X.size, X.reshape(-1)), dY, A.height, warmup, ntimes)
    assert ms > 0
    Y = dY.download().reshape(k, A.height)
    for q in range(k):
        y64, _ = oracle.spmv_f64(A.row, A.col, A.val, X[:, q].copy(), A.height)
        np.testing.assert_array_equal(Y[q], (Y0[q] + (warmup + ntimes) * y64).astype(np.float32))
    with pytest.raises(cs.ClspmvError):
        dA.time_multi(k, cs.DeviceVector(ctx, X.size, X.reshape(-1)), dY, A.height, 0, 0)
