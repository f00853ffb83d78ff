"""GPU CRS -> BCRS conversion, BCRS SpMV and BCRS SpMM against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle
from smaxkernels_amd import capi, matgen
from tests.helpers import almost_equal, arr, assert_bitwise, reference_kats

pytestmark = pytest.mark.gpu
KATS = reference_kats()


def gpu_bcrs(ctx, n_rows, n_cols, rp, col, val, bh, bw, hp, wp, cm):
    d = [ctx.upload(a) for a in (rp, col, val)]
    b = ctx.bcrs_from_crs(n_rows, n_cols, int(rp[-1]), d[0], d[1], d[2],
                          val.dtype.itemsize, bh, bw, hp, wp, cm)
    for a in d:
        a.free()
    return b


@pytest.mark.parametrize("name", ["spmv_bcrs_1_1_test_1.hpp",
                                  "spmv_bcrs_1_1_test_2.hpp"])
def test_kat_bcrs_conversion_on_gpu(ctx, name):
    k = KATS[name]
    c = {n: v["value"] for n, v in k["consts"].items()}
    b = gpu_bcrs(ctx, 4, 4, arr(k, "A_crs->row_ptr", np.int32),
                 arr(k, "A_crs->col", np.int32), arr(k, "A_crs->val", np.float64),
                 c["target_b_height"], c["target_b_width"], c["target_height_pad"],
                 c["target_width_pad"], c["use_blocked_column_major"])
    got = b.arrays(np.float64)
    assert b.info.n_blocks == k["ctors"]["A_bcrs_exp"]["args"][2]
    assert_bitwise(got["col"], arr(k, "A_bcrs_exp->col", np.int32))
    assert_bitwise(got["row_ptr"], arr(k, "A_bcrs_exp->row_ptr", np.int32))
    assert almost_equal(got["val"], arr(k, "A_bcrs_exp->val", np.float64)).all()
    b.destroy()


def test_kat_bcrs_spmv_on_gpu(ctx):
    k = KATS["spmv_bcrs_1_1_test_3.hpp"]
    nbr, nbc, nb, bh, bw, hp, wp = k["ctors"]["A_bcrs"]["args"]
    d = [ctx.upload(arr(k, n, t)) for n, t in (("A_bcrs->col", np.int32),
                                               ("A_bcrs->row_ptr", np.int32),
                                               ("A_bcrs->val", np.float64))]
    dx, dy = ctx.upload(np.ones(nbc * wp)), ctx.zeros(nbr * hp, np.float64)
    ctx.bcrs_spmv(capi.F64, nbr, bh, bw, hp, wp, d[0], d[1], d[2], True, dx, dy)
    assert almost_equal(ctx.download(dy), arr(k, "y_expected", np.float64)).all()


@pytest.mark.parametrize("cm", [True, False])
def test_laplace_blocked_equals_crs_on_gpu(ctx, cm):
    """spmv_bcrs_laplace_test.hpp: 16x16 1-D Laplacian, 4x8 blocks."""
    from tests.test_oracle import laplace1d
    rp, col, val = laplace1d(16)
    b = gpu_bcrs(ctx, 16, 16, rp, col, val, 4, 8, 4, 8, cm)
    x = 1.0 / (((np.arange(16) + 3) % 23) + 1.0)
    dx, dy = ctx.upload(x), ctx.zeros(16, np.float64)
    i = b.info
    ctx.bcrs_spmv(capi.F64, i.n_block_rows, 4, 8, 4, 8, i.col, i.row_ptr, i.val,
                  cm, dx, dy)
    assert almost_equal(ctx.download(dy), oracle.crs_spmv(rp, col, val, x)).all()
    b.destroy()


def vals_for(vt, v64):
    if vt == capi.F64:
        return v64
    if vt == capi.F32:
        return v64.astype(np.float32)
    return matgen.to_bf16(v64)


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("bh,bw,hp,wp,cm", [(4, 4, 4, 4, True), (4, 4, 4, 4, False),
                                            (4, 4, 5, 6, True), (2, 4, 3, 4, False),
                                            (2, 4, 2, 4, True), (2, 2, 2, 2, False)])
def test_block7_conversion_spmv_spmm(ctx, vt, bh, bw, hp, wp, cm):
    A = matgen.block7(10, 4)  # 4000 rows, 4x4 dense blocks
    val = vals_for(vt, A.val)
    b = gpu_bcrs(ctx, A.n_rows, A.n_cols, A.row_ptr, A.col, val, bh, bw, hp, wp, cm)
    want = oracle.crs_to_bcrs(A.n_rows, A.n_cols, A.row_ptr, A.col, val, bh, bw, hp,
                              wp, cm)
    got = b.arrays(val.dtype)
    assert b.info.n_blocks == want["n_blocks"]
    for f in ("col", "row_ptr"):
        assert_bitwise(got[f], want[f], f)
    assert_bitwise(got["val"].view(np.uint8), want["val"].view(np.uint8), "val")
    i = b.info
    xt = np.float64 if vt == capi.F64 else np.float32
    x = matgen.uniform_f64(3, i.n_block_cols * wp).astype(xt)
    dx, dy = ctx.upload(x), ctx.zeros(i.n_block_rows * hp, xt)
    ctx.bcrs_spmv(vt, i.n_block_rows, bh, bw, hp, wp, i.col, i.row_ptr, i.val, cm,
                  dx, dy)
    yw = oracle.bcrs_spmv(i.n_block_rows, bh, bw, hp, wp, want["col"],
                          want["row_ptr"], want["val"], cm, x)
    rows = (np.arange(i.n_block_rows * hp) % hp) < bh
    assert_bitwise(ctx.download(dy)[rows], yw[rows], "bcrs spmv")
    # shift 1: X and Y one entry past a 16-byte boundary (no 16-byte runs; the
    # same chains).  k = 8, 10 and misaligned 16 with 4-byte X entries and
    # dense blocks take column pairs per lane
    for k, shift in ((1, 0), (6, 0), (8, 0), (8, 1), (10, 0), (16, 0), (16, 1), (32, 0),
                     (64, 0)):
        X = matgen.uniform_f64(4, i.n_block_cols * wp * k).astype(xt)
        n_y = i.n_block_rows * hp * k
        dX = ctx.upload(np.concatenate([X[:shift], X]))
        dY = ctx.zeros(n_y + shift, xt)
        ctx.bcrs_spmm(vt, i.n_block_rows, bh, bw, hp, wp, i.col, i.row_ptr, i.val,
                      cm, k, dX.ptr + shift * X.itemsize, dY.ptr + shift * X.itemsize)
        Yw = oracle.bcrs_spmm(i.n_block_rows, bh, bw, hp, wp, want["col"],
                              want["row_ptr"], want["val"], cm, k, X)
        rk = np.repeat(rows, k)
        assert_bitwise(ctx.download(dY)[shift:][rk], Yw[rk], f"bcrs spmm k={k} shift={shift}")
        dX.free()
        dY.free()
    b.destroy()


@pytest.mark.parametrize("vt", [capi.F32, capi.BF16])
@pytest.mark.parametrize("cm", [True, False])
@pytest.mark.parametrize("k", [8, 16, 32, 64])
def test_bcrs_spmm_ragged_block_rows(ctx, vt, cm, k):
    """Dense 4x4 blocks at k = 64 (one value per lane, broadcast across the
    block row's 16 lanes) and k = 8 and 16 (a quarter block per lane,
    broadcast across the row's 4 lanes): empty block rows, rows of 1-9 blocks (every
    remainder of the 4-block groups) and rows of 40 blocks, with a block row
    count that leaves the last workgroup partly empty; bit for bit against
    the oracle."""
    rng = np.random.default_rng(64)
    nbr, nbc = 203, 300
    lens = rng.integers(1, 10, nbr)
    lens[::5] = 0
    lens[3::17] = 40
    row_ptr = np.zeros(nbr + 1, np.int32)
    row_ptr[1:] = np.cumsum(lens)
    col = np.concatenate([np.sort(rng.choice(nbc, n, replace=False)) for n in lens]
                         ).astype(np.int32)
    val = vals_for(vt, rng.uniform(-1.0, 1.0, int(row_ptr[-1]) * 16))
    X = rng.uniform(-1.0, 1.0, nbc * 4 * k).astype(np.float32)
    d = [ctx.upload(a) for a in (col, row_ptr, val, X)]
    dY = ctx.upload(np.full(nbr * 4 * k, 7.0, np.float32))
    ctx.bcrs_spmm(vt, nbr, 4, 4, 4, 4, d[0], d[1], d[2], cm, k, d[3], dY)
    want = oracle.bcrs_spmm(nbr, 4, 4, 4, 4, col, row_ptr, val, cm, k, X)
    got = ctx.download(dY)
    assert_bitwise(got, want, f"bcrs spmm k={k}")
    assert (got.reshape(nbr, -1)[lens == 0] == 0).all()
    for a in (*d, dY):
        a.free()


def test_bcrs_scalar_equivalence(ctx):
    """BCRS SpMV of the 7-point block matrix equals the CRS SpMV up to
    summation order (rows of the block matrix padded by zeros)."""
    A = matgen.block7(12, 4)
    b = gpu_bcrs(ctx, A.n_rows, A.n_cols, A.row_ptr, A.col, A.val, 4, 4, 4, 4, True)
    x = matgen.uniform_f64(8, A.n_cols)
    dx, dy = ctx.upload(x), ctx.zeros(A.n_rows, np.float64)
    i = b.info
    ctx.bcrs_spmv(capi.F64, i.n_block_rows, 4, 4, 4, 4, i.col, i.row_ptr, i.val,
                  True, dx, dy)
    want = oracle.crs_spmv(A.row_ptr, A.col, A.val, x)
    np.testing.assert_allclose(ctx.download(dy), want, rtol=1e-13, atol=1e-13)
    b.destroy()


@pytest.mark.parametrize("bh,bw", [(3, 3), (8, 2), (16, 4), (6, 1)])
def test_bcrs_conversion_other_block_heights(ctx, bh, bw):
    """Block heights outside the register-specialised {1, 2, 4} (8 included)
    take the generic block-row merge: arrays equal the oracle's conversion
    and the SpMV equals the oracle's BCRS SpMV."""
    A = matgen.lomax_band(4800, half=300)  # ascending columns; 4800 = 3*16*100
    b = gpu_bcrs(ctx, A.n_rows, A.n_cols, A.row_ptr, A.col, A.val, bh, bw, bh, bw, False)
    want = oracle.crs_to_bcrs(A.n_rows, A.n_cols, A.row_ptr, A.col, A.val, bh, bw, bh, bw,
                              False)
    got = b.arrays(np.float64)
    assert b.info.n_blocks == want["n_blocks"]
    for f in ("col", "row_ptr"):
        assert_bitwise(got[f], want[f], f)
    assert_bitwise(got["val"], want["val"], "val")
    i = b.info
    x = matgen.uniform_f64(9, A.n_cols)
    dx, dy = ctx.upload(x), ctx.zeros(A.n_rows, np.float64)
    ctx.bcrs_spmv(capi.F64, i.n_block_rows, bh, bw, bh, bw, i.col, i.row_ptr, i.val, False,
                  dx, dy)
    assert_bitwise(ctx.download(dy), oracle.bcrs_spmv(i.n_block_rows, bh, bw, bh, bw,
                                                      want["col"], want["row_ptr"],
                                                      want["val"], False, x))
    for d in (dx, dy):
        d.free()
    b.destroy()


def test_bcrs_conversion_duplicate_entries_last_wins(ctx):
    """A CRS row may list a column twice (Matrix Market files can): the
    reference places the values in order, so the later one stays; the GPU
    conversion places each row's values in order too."""
    rp = np.array([0, 3, 4, 6, 7], np.int32)
    col = np.array([0, 1, 1, 2, 2, 2, 3], np.int32)
    val = np.array([1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 7.0])
    b = gpu_bcrs(ctx, 4, 4, rp, col, val, 2, 2, 2, 2, False)
    want = oracle.crs_to_bcrs(4, 4, rp, col, val, 2, 2, 2, 2, False)
    got = b.arrays(np.float64)
    for f in ("col", "row_ptr", "val"):
        assert_bitwise(got[f], want[f], f)
    b.destroy()


def mixed_row_lengths(n, short, long_from, long_len, seed):
    """n x n CRS: rows below long_from hold `short` ascending columns near the
    diagonal, the others long_len distinct ascending random columns."""
    rng = np.random.default_rng(seed)
    cols = []
    for r in range(n):
        if r < long_from:
            c = np.clip(np.arange(r - short // 2, r - short // 2 + short), 0, n - 1)
            cols.append(np.unique(c))
        else:
            cols.append(np.sort(rng.choice(n, long_len, replace=False)))
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum([len(c) for c in cols])
    col = np.concatenate(cols).astype(np.int32)
    return rp, col, rng.uniform(-1.0, 1.0, int(rp[-1]))


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("cm", [True, False])
def test_bcrs_conversion_long_rows_read_from_memory(ctx, vt, cm):
    """Workgroups whose CRS range exceeds the LDS tile merge straight from
    memory: rows 0..511 are short (staged), rows 512..1023 hold 600 entries
    each (256 such rows per workgroup, far past the tile)."""
    rp, col, v64 = mixed_row_lengths(1024, 3, 512, 600, 11)
    val = vals_for(vt, v64)
    b = gpu_bcrs(ctx, 1024, 1024, rp, col, val, 4, 4, 4, 4, cm)
    want = oracle.crs_to_bcrs(1024, 1024, rp, col, val, 4, 4, 4, 4, cm)
    got = b.arrays(val.dtype)
    assert b.info.n_blocks == want["n_blocks"]
    for f in ("col", "row_ptr"):
        assert_bitwise(got[f], want[f], f)
    assert_bitwise(got["val"].view(np.uint8), want["val"].view(np.uint8), "val")
    b.destroy()


def test_bcrs_conversion_of_a_matrix_without_entries(ctx):
    """nnz = 0: no blocks, an all-zero block row pointer, and an SpMV that
    writes zeros."""
    rp = np.zeros(9, np.int32)
    b = gpu_bcrs(ctx, 8, 8, rp, np.zeros(0, np.int32), np.zeros(0), 2, 2, 2, 2, False)
    i = b.info
    assert i.n_blocks == 0 and i.n_block_rows == 4
    assert (b.arrays(np.float64)["row_ptr"] == 0).all()
    dx, dy = ctx.upload(np.ones(8)), ctx.upload(np.full(8, 5.0))
    ctx.bcrs_spmv(capi.F64, 4, 2, 2, 2, 2, i.col, i.row_ptr, i.val, False, dx, dy)
    assert (ctx.download(dy) == 0).all()
    for d in (dx, dy):
        d.free()
    b.destroy()


def test_bcrs_conversion_rejects_columns_out_of_range(ctx):
    """A column index outside [0, n_cols) would place a value outside its
    block: the conversion refuses the matrix."""
    rp = np.array([0, 2, 3, 4, 4], np.int32)
    for bad in (4, -1, 1 << 30):
        col = np.array([0, 1, bad, 2], np.int32)
        with pytest.raises(capi.SmaxHipError) as e:
            gpu_bcrs(ctx, 4, 4, rp, col, np.ones(4), 2, 2, 2, 2, False)
        assert e.value.status == capi.ERROR_INVALID_VALUE
        assert "outside" in str(e.value)


def test_bcrs_conversion_rejects_what_the_reference_rejects(ctx):
    A = matgen.poisson2d(6)  # 36 x 36
    for bh, bw, hp, wp in ((5, 4, 5, 4), (4, 5, 4, 5), (4, 4, 3, 4), (4, 4, 4, 3)):
        with pytest.raises(capi.SmaxHipError) as e:
            gpu_bcrs(ctx, 36, 36, A.row_ptr, A.col, A.val, bh, bw, hp, wp, True)
        assert e.value.status == capi.ERROR_INVALID_VALUE
    # a row whose block columns descend (convert_formats.hpp:230-234 throws)
    rp = np.array([0, 2, 2, 2, 2], np.int32)
    col = np.array([3, 0], np.int32)
    with pytest.raises(capi.SmaxHipError) as e:
        gpu_bcrs(ctx, 4, 4, rp, col, np.ones(2), 2, 2, 2, 2, True)
    assert "Blocked Column" in str(e.value)


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("cm", [True, False])
def test_bcrs_adjoint_transpose_spmm_sddmm(ctx, vt, cm):
    """C5 at reduced size: A^T through the transposed block layout equals the
    reference BCRS conversion of the explicit A^T (bytes), its SpMM equals the
    reference CRS SpMM of A^T bit for bit, and the block SDDMM matches FP64."""
    A = matgen.block7(8, 4)  # 2048 rows, dense 4x4 blocks
    val = vals_for(vt, A.val)
    b = gpu_bcrs(ctx, A.n_rows, A.n_cols, A.row_ptr, A.col, val, 4, 4, 4, 4, cm)
    T = b.transpose()
    trp, tcol, tval = oracle.crs_transpose(A.n_rows, A.n_cols, A.row_ptr, A.col, val)
    want = oracle.crs_to_bcrs(A.n_cols, A.n_rows, trp, tcol, tval, 4, 4, 4, 4, not cm)
    got = T.arrays(val.dtype)
    assert T.info.block_col_major == (0 if cm else 1)
    for f in ("col", "row_ptr"):
        assert_bitwise(got[f], want[f], f)
    assert_bitwise(got["val"].view(np.uint8), want["val"].view(np.uint8), "val")
    xt = np.float64 if vt == capi.F64 else np.float32
    for k in (1, 8, 64):
        G = matgen.uniform_f64(11, A.n_rows * k).astype(xt)
        dG, dZ = ctx.upload(G), ctx.zeros(A.n_cols * k, xt)
        T.spmm(vt, k, dG, dZ)
        assert_bitwise(ctx.download(dZ), oracle.crs_spmm(trp, tcol, tval, k, True, G),
                       f"A^T G k={k}")
    # refresh after a value change keeps A^T current
    new = vals_for(vt, matgen.uniform_f64(123, A.nnz))
    b2 = gpu_bcrs(ctx, A.n_rows, A.n_cols, A.row_ptr, A.col, new, 4, 4, 4, 4, cm)
    T.refresh_values(b2.info.val)
    t2 = oracle.crs_transpose(A.n_rows, A.n_cols, A.row_ptr, A.col, new)
    w2 = oracle.crs_to_bcrs(A.n_cols, A.n_rows, *t2, 4, 4, 4, 4, not cm)
    assert_bitwise(T.arrays(val.dtype)["val"].view(np.uint8), w2["val"].view(np.uint8))
    # block SDDMM vs FP64 at every stored scalar position
    k = 8
    G = matgen.uniform_f64(12, A.n_rows * k).astype(xt)
    X = matgen.uniform_f64(13, A.n_cols * k).astype(xt)
    dv = ctx.zeros(b.info.n_blocks * 16, xt)
    b.sddmm(vt, k, ctx.upload(G), ctx.upload(X), dv)
    got = ctx.download(dv).astype(np.float64)
    ref = oracle.sddmm_f64(A.row_ptr, A.col, k, G.astype(np.float64),
                           X.astype(np.float64))
    rows = np.repeat(np.arange(A.n_rows), np.diff(A.row_ptr))
    bi = b.arrays(val.dtype)
    br, bc = rows // 4, A.col // 4
    blk = np.array([bi["row_ptr"][r] + np.searchsorted(
        bi["col"][bi["row_ptr"][r]:bi["row_ptr"][r + 1]], c) for r, c in zip(br, bc)])
    off = (A.col % 4) * 4 + rows % 4 if cm else (rows % 4) * 4 + A.col % 4
    mine = got[blk * 16 + off]
    scale = np.abs(G.astype(np.float64).reshape(-1, k)[rows] *
                   X.astype(np.float64).reshape(-1, k)[A.col]).sum(axis=1)
    u = np.finfo(xt).eps / 2
    assert (np.abs(mine - ref) <= (np.log2(k) + 1) * u * scale + 1e-300).all()
    for h in (T, b, b2):
        h.destroy()


@pytest.mark.parametrize("vt", [capi.F64, capi.BF16])
@pytest.mark.parametrize("bh,bw,hp,wp,cm", [(1, 1, 1, 1, False), (4, 4, 4, 4, False),
                                            (4, 4, 4, 4, True), (3, 2, 4, 4, False),
                                            (2, 3, 2, 5, True), (5, 6, 5, 6, False)])
@pytest.mark.parametrize("k,shift", [(1, 0), (2, 0), (3, 0), (8, 0), (8, 1), (20, 0), (32, 0),
                                     (33, 0), (64, 0), (70, 0)])
def test_bcrs_sddmm_block_lines(ctx, vt, bh, bw, hp, wp, cm, k, shift):
    """Block SDDMM over ragged block rows (empty ones, runs of them, and one
    that spans several workgroups) for every load width (k = 8 with G and X
    one entry off their 16-byte alignment), against binary64 (binary128 for
    FP64) sums.  Per position: KP chains of q = ceil(k / KP) terms (KP the
    power of two >= k, at most 64) and log2 KP additions of partial sums, so
    |d - d_exact| <= (q + log2 KP) u sum |g x|; padding positions are zero."""
    rng = np.random.default_rng(hp * 100 + k)
    nbr, nbc = 260, 2100
    per = rng.integers(0, 6, nbr)
    per[[0, 7, 8, 9, nbr - 1]] = 0
    per[40] = nbc
    brp = np.concatenate([[0], np.cumsum(per)]).astype(np.int64)
    bcol = np.concatenate([np.sort(rng.choice(nbc, p, replace=False)) for p in per])
    # scalar CRS with dense blocks
    rp = np.concatenate([[0], np.cumsum(np.repeat(per * bw, bh))]).astype(np.int32)
    col = np.concatenate([np.tile((bcol[s:e, None] * bw + np.arange(bw)).ravel(), bh)
                          for s, e in zip(brp, brp[1:])]).astype(np.int32)
    vec = np.float64 if vt == capi.F64 else np.float32
    val = np.zeros(col.size, np.float64 if vt == capi.F64 else np.uint16)
    b = gpu_bcrs(ctx, nbr * bh, nbc * bw, rp, col, val, bh, bw, hp, wp, cm)
    assert b.info.n_blocks == brp[-1]
    G = rng.uniform(-1, 1, (nbr * hp, k)).astype(vec)
    X = rng.uniform(-1, 1, (nbc * wp, k)).astype(vec)
    pad = np.zeros(shift, vec)
    dG, dX = (ctx.upload(np.concatenate([pad, a.ravel()])) for a in (G, X))
    n = int(brp[-1]) * hp * wp
    dv = ctx.upload(np.full(n, 7, vec))
    off = shift * vec().itemsize
    b.sddmm(vt, k, dG.ptr + off, dX.ptr + off, dv)
    got = ctx.download(dv).reshape((-1, wp, hp) if cm else (-1, hp, wp))
    if cm:
        got = got.transpose(0, 2, 1)
    brow = np.repeat(np.arange(nbr), per)
    wide = np.longdouble if vt == capi.F64 else np.float64
    Gb = G.reshape(nbr, hp, k)[brow].astype(wide)
    Xb = X.reshape(nbc, wp, k)[bcol].astype(wide)
    want, scale = np.zeros((2, brow.size, hp, wp), wide)
    for v in range(k):
        t = Gb[:, :, None, v] * Xb[:, None, :, v]
        want += t
        scale += np.abs(t)
    kp = min(64, 1 << (k - 1).bit_length())
    bound = (-(-k // kp) + np.log2(kp)) * np.finfo(vec).eps / 2 * scale
    real = np.zeros((hp, wp), bool)
    real[:bh, :bw] = True
    assert (np.abs(got - want) <= bound)[:, real].all()
    assert (got[:, ~real] == 0).all()
    for d in (dG, dX, dv):
        d.free()
    b.destroy()


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("bh,bw,hp,wp", [(1, 1, 1, 1), (2, 2, 2, 2), (3, 3, 3, 3), (3, 3, 4, 4),
                                         (5, 1, 5, 1)])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_bcrs_transpose_refresh_unit_widths(ctx, vt, bh, bw, hp, wp, shift):
    """The transpose's blocks are copied in the widest unit (16, 8, 4 or 2
    bytes) that the block size and both addresses allow: block sizes of every
    class, and source values 0, 1 or 2 entries off their alignment."""
    n = 5
    A = matgen.block7(n, 1)
    nb = n ** 3
    per = np.diff(A.row_ptr)
    rp = np.concatenate([[0], np.cumsum(np.repeat(per * bw, bh))]).astype(np.int32)
    col = np.concatenate([np.tile((A.col[s:e, None].astype(np.int64) * bw + np.arange(bw)).ravel(), bh)
                          for s, e in zip(A.row_ptr, A.row_ptr[1:])]).astype(np.int32)
    dt = {capi.F64: np.float64, capi.F32: np.float32, capi.BF16: np.uint16}[vt]
    b = gpu_bcrs(ctx, nb * bh, nb * bw, rp, col, np.zeros(col.size, dt), bh, bw, hp, wp, False)
    T = b.transpose()
    src = np.random.default_rng(shift).integers(0, 1 << 14, (b.info.n_blocks, hp * wp)).astype(dt)
    d = ctx.upload(np.concatenate([np.zeros(shift, dt), src.ravel()]))
    T.refresh_values(d.ptr + shift * dt().itemsize)
    order = ctx.download_ptr(T.info.src_block, T.info.n_blocks, np.int32)
    assert np.array_equal(np.sort(order), np.arange(b.info.n_blocks))
    assert_bitwise(T.arrays(dt)["val"], src[order].ravel())
    d.free()
    for h in (T, b):
        h.destroy()


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("b,n_blocks", [(3, 116_508), (3, 116_509), (5, 41_943), (5, 41_944),
                                        (4, 140_001)])
def test_bcrs_transpose_refresh_around_four_units(ctx, vt, b, n_blocks):
    """From 2^20 units of 8 bytes and less a thread moves four: one block below
    and above that (9 and 25 units a block), and 16-byte units, one a thread."""
    dt = {capi.F64: np.float64, capi.F32: np.float32, capi.BF16: np.uint16}[vt]
    rng = np.random.default_rng(b)
    rp = np.arange(n_blocks * b + 1, dtype=np.int32) * b
    col = (rng.permutation(n_blocks)[:, None, None] * b + np.zeros((1, b, 1), int)
           + np.arange(b)).ravel().astype(np.int32)
    A = gpu_bcrs(ctx, n_blocks * b, n_blocks * b, rp, col, np.zeros(col.size, dt), b, b, b, b, False)
    T = A.transpose()
    src = rng.integers(0, 1 << 14, (n_blocks, b * b)).astype(dt)
    d = ctx.upload(src)
    T.refresh_values(d)
    order = ctx.download_ptr(T.info.src_block, n_blocks, np.int32)
    assert_bitwise(T.arrays(dt)["val"], src[order].ravel())
    d.free()
    for h in (T, A):
        h.destroy()


@pytest.mark.parametrize("n_cols", [1, 2, 255, 256, 257, 4097, 65536, 65537, (1 << 17) + 3])
@pytest.mark.parametrize("nnz", [1, 63, 4095, 4096, 4097, 30011])
def test_transposed_pattern_digit_and_tile_edges(ctx, n_cols, nnz):
    """The sort behind the transposes, through 1x1 blocks: one to three digits
    (1 to 18 bit keys), partial tiles, runs of empty rows and one row longer
    than a wavefront's share, against a stable host sort by column."""
    rng = np.random.default_rng(nnz)
    n_rows = 700
    cut = np.sort(rng.integers(0, nnz + 1, n_rows - 1))
    cut[100:400] = cut[100]          # empty rows
    cut[400:] = np.maximum(cut[400:], cut[100])
    rp = np.concatenate([[0], cut, [nnz]]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n_cols, e - s, replace=e - s > n_cols))
                          for s, e in zip(rp, rp[1:])]).astype(np.int32)
    # a block row keeps each column once
    keep = np.ones(nnz, bool)
    keep[1:] = col[1:] != col[:-1]
    keep[rp[:-1][rp[:-1] < nnz]] = True
    rp = np.concatenate([[0], np.cumsum(keep)])[rp].astype(np.int32)
    col = col[keep]
    b = gpu_bcrs(ctx, n_rows, n_cols, rp, col, np.arange(col.size, dtype=np.float64), 1, 1, 1, 1,
                 False)
    T = b.transpose()
    order = np.argsort(col, kind="stable").astype(np.int32)
    rows = np.repeat(np.arange(n_rows), np.diff(rp)).astype(np.int32)
    got = T.arrays(np.float64)
    assert_bitwise(ctx.download_ptr(T.info.src_block, col.size, np.int32), order, "src_block")
    assert_bitwise(got["col"], rows[order], "col")
    assert_bitwise(got["row_ptr"], np.searchsorted(col[order], np.arange(n_cols + 1))
                   .astype(np.int32), "row_ptr")
    assert_bitwise(got["val"], order.astype(np.float64), "val")
    for h in (T, b):
        h.destroy()


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("cm", [True, False])
@pytest.mark.parametrize("bh,bw,hp,wp", [(3, 3, 3, 3), (6, 3, 7, 4), (3, 6, 3, 8), (6, 6, 6, 6),
                                         (5, 5, 5, 5), (10, 5, 11, 5), (7, 7, 7, 7),
                                         (1, 8, 1, 8), (3, 2, 3, 2), (9, 9, 9, 9),
                                         (2, 2, 2, 2), (4, 4, 4, 5)])
def test_bcrs_products_of_any_block_shape(ctx, vt, cm, bh, bw, hp, wp):
    """SpMV by rows (b_w <= 8) and SpMM in parts of a block: block rows of 0 to
    9 and of 40 blocks (every remainder of the groups), padded blocks, k below,
    at and past a run of columns, X and Y one entry past a 16-byte boundary;
    bit for bit against the oracle."""
    rng = np.random.default_rng(65)
    nbr, nbc = 157, 90
    lens = rng.integers(0, 10, nbr)
    lens[3::17] = 40
    row_ptr = np.zeros(nbr + 1, np.int32)
    row_ptr[1:] = np.cumsum(lens)
    col = np.concatenate([np.sort(rng.choice(nbc, n, replace=False)) for n in lens]
                         ).astype(np.int32)
    val = vals_for(vt, rng.uniform(-1.0, 1.0, int(row_ptr[-1]) * hp * wp))
    xt = np.float64 if vt == capi.F64 else np.float32
    d = [ctx.upload(a) for a in (col, row_ptr, val)]
    rows = (np.arange(nbr * hp) % hp) < bh
    x = rng.uniform(-1.0, 1.0, nbc * wp).astype(xt)
    dx, dy = ctx.upload(x), ctx.zeros(nbr * hp, xt)
    ctx.bcrs_spmv(vt, nbr, bh, bw, hp, wp, *d, cm, dx, dy)
    want = oracle.bcrs_spmv(nbr, bh, bw, hp, wp, col, row_ptr, val, cm, x)
    assert_bitwise(ctx.download(dy)[rows], want[rows], "spmv")
    dx.free()
    dy.free()
    for k in (1, 2, 3, 4, 5, 8, 11, 32):
        X = rng.uniform(-1.0, 1.0, nbc * wp * k).astype(xt)
        dX = ctx.upload(np.concatenate([X[:1], X]))
        dY = ctx.zeros(nbr * hp * k + 1, xt)
        ctx.bcrs_spmm(vt, nbr, bh, bw, hp, wp, *d, cm, k, dX.ptr + X.itemsize,
                      dY.ptr + X.itemsize)
        want = oracle.bcrs_spmm(nbr, bh, bw, hp, wp, col, row_ptr, val, cm, k, X)
        rk = np.repeat(rows, k)
        got = ctx.download(dY)[1:]
        assert_bitwise(got[rk], want[rk], f"spmm k={k}")
        assert not got[~rk].any(), f"spmm k={k} wrote padding rows"
        dX.free()
        dY.free()
    for a in d:
        a.free()


@pytest.mark.parametrize("vt", [capi.F64, capi.F32, capi.BF16])
@pytest.mark.parametrize("cm", [False, True])
@pytest.mark.parametrize("bh,bw,n,k", [
    # one output row a thread below 2^14 (3 x 2^14, 2^18) threads of several rows
    (3, 3, 16383, 4), (3, 3, 16384, 4), (3, 3, 8192, 8), (5, 5, 4096, 13), (5, 5, 16384, 2),
    (6, 6, 8192, 4), (6, 6, 8191, 4), (6, 3, 24576, 4), (9, 3, 43691, 2), (2, 2, 49151, 4),
    (2, 2, 49152, 4), (4, 4, 4096, 8),
    # the register-blocked kernel once Y is 90 or 100 MB (2x2), 64 MB (4x4, even k)
    (2, 2, 351_562, 16), (2, 2, 351_563, 16), (2, 2, 781_250, 16), (2, 2, 351_563, 17),
    (4, 4, 250_000, 8), (4, 4, 249_999, 8), (4, 4, 222_223, 9),
    # and for k = 3 in FP32 (2x2) from 2^13 block rows to 5 MB
    (2, 2, 8191, 3), (2, 2, 8192, 3), (2, 2, 208_333, 3), (2, 2, 208_334, 3)])
def test_bcrs_spmm_around_the_kernel_choices(ctx, vt, cm, bh, bw, n, k):
    """Whole numbers, so that every order gives the exact product."""
    import scipy.sparse as sp
    rng = np.random.default_rng(n + k)
    per = rng.integers(0, 3, n)
    per[rng.integers(0, n, 3)] = 40
    rp = np.concatenate([[0], np.cumsum(per)]).astype(np.int32)
    n_cols = 5000
    col = np.concatenate([np.sort(rng.choice(n_cols, p, replace=False)) if p > 2 else
                          np.arange(p) * 2000 for p in per]).astype(np.int32)
    blocks = rng.integers(-3, 4, (rp[-1], bh, bw)).astype(np.float64)
    vec = np.float64 if vt == capi.F64 else np.float32
    X = rng.integers(-4, 5, (n_cols * bw, k)).astype(vec)
    stored = (blocks.transpose(0, 2, 1) if cm else blocks).ravel()
    val = stored if vt == capi.F64 else stored.astype(np.float32) if vt == capi.F32 else matgen.to_bf16(stored)
    d = [ctx.upload(a) for a in (col, rp, val, X)]
    Y = ctx.zeros(n * bh * k, vec)
    ctx.bcrs_spmm(vt, n, bh, bw, bh, bw, *d[:3], cm, k, d[3], Y)
    want = sp.bsr_matrix((blocks, col, rp), shape=(n * bh, n_cols * bw)) @ X.astype(np.float64)
    assert_bitwise(ctx.download(Y), want.astype(vec).ravel())
    for a in (*d, Y):
        a.free()
