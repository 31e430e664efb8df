"""GPU checks of the GEMMs on the bf16 matrix cores (zn_sgemm_<layout>_s*,
operands split into three bf16 parts) and of the convolutions on them:
Backend.matMul and its transposes (src/backend.zig:169-325).  The policy takes
them for part of the problems of 2^30 multiply-adds and more with K of 256 or
more; the tests name each tile (zn_hip_set_gemm_tile), at small extents, and
take the policy's choice at large ones.

- every layout against fp64 within 2e-7 * sqrt(K) of the componentwise bound
  (a fiftieth of the fp32 kernels' bar), at extents one below and above the
  tiles' and at K tails of 1 to 31;
- values near the ends of the fp32 range, where unscaled parts would be
  subnormal, keep that bound;
- Inf, NaN and sums beyond 2^80 give what fp32 arithmetic gives;
- the fused epilogues, accumulation, padded leading dimensions, unaligned
  bases and strided batches.
"""
from __future__ import annotations

import contextlib

import numpy as np
import pytest

from _parity import uniform
from gpu_common import announce, assert_close, ref_gemm, run_gemm, stored_shapes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from zigneuron_amd import Context
    c = Context(0)
    yield c
    c.close()


TILES = ["256x256s", "256x128s", "128x128s", "128x64s", "128x128sc"]


@contextlib.contextmanager
def forced(ctx, tile, splits=0):
    ctx.set_gemm_tile(tile)
    ctx.set_gemm_splits(splits)
    try:
        yield
    finally:
        ctx.set_gemm_tile("auto")
        ctx.set_gemm_splits(0)


def as_mk(a, layout):
    return a.T if layout == "tn" else a


def as_kn(b, layout):
    return b.T if layout == "nt" else b


def check_rows(out, layout, a, b, k, rows, what):
    """Componentwise against fp64.  The bound: the flushed kernels round once per 32 of K on sums of 32, the 256x256
    tile six times per 32 of K on the whole sum, at most 6K/32 roundings of 2^-24, which as a random walk stay under
    sqrt(6K/32) * 2^-24 * 8 = 2e-7 * sqrt(K)."""
    a64, b64 = as_mk(a, layout)[rows].astype(np.float64), as_kn(b, layout).astype(np.float64)
    ref, den = a64 @ b64, np.abs(a64) @ np.abs(b64)
    err = np.abs(out[rows] - ref) / np.maximum(den, 1e-300)
    assert np.isfinite(out).all() and err.max() <= 2e-7 * np.sqrt(k), f"{what}: {err.max():.3g}"


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k,splits", [(257, 129, 33, 0),    # one row and column past the tiles; K tails of 1 ...
                                          (255, 191, 287, 0),   # ... and 31
                                          (128, 256, 64, 0),    # whole tiles and K slices
                                          (3, 5, 31, 0),        # less than a slice
                                          (300, 260, 1029, 3)])  # K split in three with the reduce
def test_split_tile_against_fp64(ctx, layout, tile, m, n, k, splits):
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a_shape, b_shape = stored_shapes(layout, m, n, k)
    a, b = uniform(rng, a_shape), uniform(rng, b_shape)
    announce(f"split {tile} {layout} {m}x{n}x{k} splits {splits}")
    with forced(ctx, tile, splits):
        out = run_gemm(ctx, layout, a, b, m, n, k)
    check_rows(out, layout, a, b, k, np.arange(m), f"{tile} {layout} {m}x{n}x{k}")


SHAPES = [(4097, 1023, 777),    # split 128x128 tiles, and one row on the fp32 kernels
          (4096, 1025, 257),    # fp32: one column past the tiles
          (4100, 4097, 288),    # split 256x128 tiles
          (300, 260, 16389),    # fp32 in K slices
          (1024, 1000, 8195)]   # split 256x128 tiles in K slices


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_policy_against_fp64(ctx, layout, m, n, k):
    """Problems around the line between the split and the fp32 kernels, which stay within the same bound here."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a_shape, b_shape = stored_shapes(layout, m, n, k)
    a, b = uniform(rng, a_shape), uniform(rng, b_shape)
    announce(f"split {layout} {m}x{n}x{k}")
    rows = np.unique(np.r_[0, 1, m // 2, np.arange(max(0, m - 130), m, 7), m - 1])
    check_rows(run_gemm(ctx, layout, a, b, m, n, k), layout, a, b, k, rows, f"policy {layout} {m}x{n}x{k}")


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_split_largest_tile(ctx, layout):
    """The 256x256 tile (4096 x 4096 and a K tail of 5)."""
    m, n, k = 4095, 4096, 517
    rng = np.random.default_rng(5)
    a_shape, b_shape = stored_shapes(layout, m, n, k)
    a, b = uniform(rng, a_shape), uniform(rng, b_shape)
    announce(f"split 256x256 {layout}")
    check_rows(run_gemm(ctx, layout, a, b, m, n, k), layout, a, b, k, np.r_[0:256:5, 3840:4095:11], "256x256")


@pytest.mark.parametrize("scale_a,scale_b", [(2e-38, 1.0), (1.0, 2e-38), (1e-30, 1e30), (1e28, 1e-20)])
@pytest.mark.parametrize("tile", TILES)
def test_split_keeps_small_values(ctx, tile, scale_a, scale_b):
    """Elements at the lower end of the fp32 range (their third parts would be subnormal bf16 numbers unscaled)."""
    m, n, k = 391, 277, 287
    rng = np.random.default_rng(9)
    a = (uniform(rng, (m, k)) * np.float32(scale_a)).astype(np.float32)
    b = (uniform(rng, (k, n)) * np.float32(scale_b)).astype(np.float32)
    announce(f"split range {tile} {scale_a} {scale_b}")
    with forced(ctx, tile):
        out = run_gemm(ctx, "nn", a, b, m, n, k)
    rows = np.arange(m)
    a64, b64 = a[rows].astype(np.float64), b.astype(np.float64)
    err = np.abs(out[rows] - a64 @ b64)
    # results below 2^-126 round to multiples of 2^-149
    assert np.all(err <= 2e-7 * np.sqrt(k) * (np.abs(a64) @ np.abs(b64)) + 2.0 ** -148)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("tile,splits", [(t, 0) for t in TILES] + [("256x256s", 3), ("128x128s", 3)])
def test_split_non_finite_and_huge(ctx, layout, tile, splits):
    """Inf, NaN and sums past 2^80 (where the scaled split overflows): the same values as fp32 arithmetic, and the rows
    and columns they do not touch stay within the bound."""
    m, n, k = 1001, 1030, 287
    rng = np.random.default_rng(10)
    a, b = np.abs(uniform(rng, (m, k))) + np.float32(0.1), np.abs(uniform(rng, (k, n))) + np.float32(0.1)
    a[5, 7], a[130, k - 1], a[700, 0], a[m - 1, 3] = np.inf, np.nan, -np.inf, np.float32(3e38)
    a[900] *= np.float32(1e30)  # finite in fp32: 1e30 * 300
    b[11, 40], b[2, 1000] = np.inf, np.nan
    ast = np.ascontiguousarray(a.T) if layout == "tn" else a
    bst = np.ascontiguousarray(b.T) if layout == "nt" else b
    announce(f"split non-finite {tile} {layout} splits {splits}")
    with forced(ctx, tile, splits):
        out = run_gemm(ctx, layout, ast, bst, m, n, k)
    with np.errstate(all="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
        ref32 = np.where(np.abs(ref) > np.finfo(np.float32).max, np.sign(ref) * np.inf, ref)
    fin = np.isfinite(ref32)
    np.testing.assert_array_equal(np.isnan(out), np.isnan(ref32))
    np.testing.assert_array_equal(np.isposinf(out), np.isposinf(ref32))
    np.testing.assert_array_equal(np.isneginf(out), np.isneginf(ref32))
    assert np.all(np.abs(out[fin] - ref[fin]) <= 1e-5 * np.sqrt(k) * np.abs(ref[fin]))


@pytest.mark.parametrize("act", ["linear", "relu", "sigmoid", "tanh"])
@pytest.mark.parametrize("tile,splits", [(t, 0) for t in TILES] + [("128x128s", 2)])
def test_split_epilogues(ctx, act, tile, splits):
    m, n, k = 391, 277, 260
    rng = np.random.default_rng(12)
    a, b, bias = uniform(rng, (m, k)), uniform(rng, (k, n)), uniform(rng, (n,))
    announce(f"split epilogue {tile} {act} splits {splits}")
    with forced(ctx, tile, splits):
        out = run_gemm(ctx, "nn", a, b, m, n, k, bias=bias, act=act)
    rows = np.r_[0:m:13, m - 1]
    assert_close(out[rows], ref_gemm("nn", np.ascontiguousarray(a[rows]), b, len(rows), n, k, bias=bias, act=act), "nn",
                 np.ascontiguousarray(a[rows]), b, len(rows), n, k, bias=bias, act=act, what=f"split {act}")


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("tile", TILES)
def test_split_padded_rows_accumulate_batches(ctx, layout, tile):
    """Leading dimensions and bases off 16 bytes, accumulation, NaN in the row padding (never read as a value), and a
    strided batch with a shared B."""
    m, n, k, batch = 259, 131, 73, 5
    rng = np.random.default_rng(13)
    a_shape, b_shape = stored_shapes(layout, m, n, k)
    lda, ldb, ldc = a_shape[1] + 3, b_shape[1] + 1, n + 5
    sa, sc = a_shape[0] * lda + 1, m * ldc + 3
    a = np.full((batch, sa), np.nan, np.float32)
    av = uniform(rng, (batch,) + a_shape)
    a[:, :a_shape[0] * lda].reshape(batch, a_shape[0], lda)[:, :, :a_shape[1]] = av
    b = np.full((b_shape[0], ldb), np.nan, np.float32)
    bv = uniform(rng, b_shape)
    b[:, :b_shape[1]] = bv
    c0 = uniform(rng, (batch, sc))
    da = ctx.to_device(np.concatenate([[0.0], a.ravel()]).astype(np.float32))
    db = ctx.to_device(b)
    dc = ctx.to_device(np.concatenate([[0.0], c0.ravel()]).astype(np.float32))
    announce(f"split padded batch {tile} {layout}")
    with forced(ctx, tile):
        ctx.sgemm_strided_batched(layout, m, n, k, da.offset(1), lda, sa, db, ldb, 0, dc.offset(1), ldc, sc, batch, True)
    out = dc.download()[1:].reshape(batch, sc)
    for i in range(batch):
        view, old = (x[i, :m * ldc].reshape(m, ldc) for x in (out, c0))
        np.testing.assert_array_equal(view[:, n:], old[:, n:])
        rows = np.arange(m)
        a64, b64 = as_mk(av[i], layout)[rows].astype(np.float64), as_kn(bv, layout).astype(np.float64)
        ref = old[rows, :n] + a64 @ b64
        den = np.abs(old[rows, :n]) + np.abs(a64) @ np.abs(b64)
        assert np.all(np.abs(view[rows, :n] - ref) <= 2e-7 * np.sqrt(k) * den), i
    np.testing.assert_array_equal(out[:, m * ldc:], c0[:, m * ldc:])
    for buf in (da, db, dc):
        buf.close()


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_forced_tile_takes_the_named_kernel(ctx, layout):
    """zn_hip_set_gemm_tile at a size that the policy gives to the split kernels (4096 x 1024 x 512): the fp32 tiles agree
    bit for bit with each other and not with the policy's result, the split tile does."""
    m, n, k = 4096, 1024, 512
    rng = np.random.default_rng(21)
    a_shape, b_shape = stored_shapes(layout, m, n, k)
    a, b = uniform(rng, a_shape), uniform(rng, b_shape)
    out = {}
    try:
        ctx.set_gemm_splits(1)
        for tile in ("auto", "128x128", "64x64", "256x256", "128x128s", "128x64s"):
            announce(f"forced {tile} {layout}")
            ctx.set_gemm_tile(tile)
            out[tile] = run_gemm(ctx, layout, a, b, m, n, k).view(np.uint32)
    finally:
        ctx.set_gemm_tile("auto")
        ctx.set_gemm_splits(0)
    np.testing.assert_array_equal(out["128x128"], out["64x64"])
    np.testing.assert_array_equal(out["128x128"], out["256x256"])
    np.testing.assert_array_equal(out["128x128s"], out["auto"])
    np.testing.assert_array_equal(out["128x64s"], out["auto"])
    assert not np.array_equal(out["128x128"], out["auto"])


@pytest.mark.parametrize("m,n,k,split", [(1792, 1536, 1024, False), (3200, 768, 1024, False), (2176, 1408, 832, False), (3520, 896, 1280, True)])
def test_transposed_product_below_a_round_of_split_tiles(ctx, m, n, k, split):
    """Whole float4s, TN, 128x128 tiles for 59 to 77% of the CUs: on the fp32 kernels where their 64x64 tiles fill a round,
    by the bits."""
    rng = np.random.default_rng(24)
    a, b = uniform(rng, (k, m)), uniform(rng, (k, n))
    announce(f"tn policy {m}x{n}x{k}")
    auto = run_gemm(ctx, "tn", a, b, m, n, k)
    with forced(ctx, "128x128s" if split else "64x64", 1):
        np.testing.assert_array_equal(auto.view(np.uint32), run_gemm(ctx, "tn", a, b, m, n, k).view(np.uint32))
    check_rows(auto, "tn", a, b, k, np.r_[0:m:97, m - 1], "tn policy")


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("tiles", [("256x256s", "128x128sc"), ("256x128s", "128x128s", "128x64s")], ids=["chain", "flush"])
def test_split_tiles_agree_bit_for_bit(ctx, layout, tiles):
    """The split tiles of one kind of sum, at an extent past each one's tiles and with a K tail."""
    m, n, k = 391, 277, 165
    rng = np.random.default_rng(22)
    a, b = uniform(rng, (m, k)), uniform(rng, (k, n))
    ast, bst = np.ascontiguousarray(as_mk(a, layout)), np.ascontiguousarray(as_kn(b, layout))
    out = []
    try:
        for tile in tiles:
            announce(f"tiles agree {layout} {tile}")
            ctx.set_gemm_tile(tile)
            out.append(run_gemm(ctx, layout, ast, bst, m, n, k).view(np.uint32))
    finally:
        ctx.set_gemm_tile("auto")
    for other in out[1:]:
        np.testing.assert_array_equal(out[0], other)


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 2048),   # 256x256 tiles; the chunks have 1024 rows
                                   (4097, 1023, 1100)])  # 128x128 tiles and a one-row tail; three chunks
def test_chunked_host_call_has_the_bits_of_the_device_call(ctx, m, n, k):
    """Backend.matMul cuts a large A into row chunks, which take the tiles of their own size and the whole call's kind of
    sum."""
    from zigneuron_amd import Backend
    rng = np.random.default_rng(m + k)
    a, b = uniform(rng, (m, k)), uniform(rng, (k, n))
    announce(f"chunked host call {m}x{n}x{k}")
    backend = Backend.init(0)
    for layout, name, rhs in (("nn", "matMul", b), ("nt", "matMulTransposeB", np.ascontiguousarray(b.T))):
        host = np.empty((m, n), np.float32)
        getattr(backend, name)(a, rhs, host, m, n, k)
        np.testing.assert_array_equal(host, run_gemm(ctx, layout, a, rhs, m, n, k), err_msg=name)
    backend.deinit()


def test_chunked_host_call_of_few_rows_and_long_k(ctx):
    """1024 x 1000 x 8195 in chunks of 256 rows, whose few tiles split K: K slices of whole 32s, the last one with a tail."""
    from zigneuron_amd import Backend
    m, n, k = 1024, 1000, 8195
    rng = np.random.default_rng(23)
    a, b = uniform(rng, (m, k)), uniform(rng, (k, n))
    announce(f"chunked host call {m}x{n}x{k}")
    backend = Backend.init(0)
    host = np.empty((m, n), np.float32)
    backend.matMul(a, b, host, m, n, k)
    backend.deinit()
    check_rows(host, "nn", a, b, k, np.r_[0:m:61, m - 1], "chunked")


CONVS = [(3, 64, 20, 28, 96, 3, 1, 1),   # channels of 32: one tap per K slice; rows of whole fours of pixels (the _u kernels)
         (3, 36, 21, 19, 100, 3, 1, 1),  # taps change inside a slice; rows of 19 pixels
         (5, 32, 31, 29, 48, 5, 2, 2),   # stride 2
         (2, 64, 22, 22, 40, 3, 1, 0),   # no padding
         (2, 4, 17, 16, 4, 3, 1, 1)]     # fewer channels than a tile's rows, K of little more than a slice
TILED = [(c, t) for c in CONVS for t in ("conv128x128s", "conv64x128s")]


@pytest.mark.parametrize("case,tile", TILED + [((16, 32, 63, 63, 128, 3, 2, 1), "auto")])
@pytest.mark.parametrize("poison", [False, True])
def test_split_convolutions(ctx, case, tile, poison):
    """The convolution forward and backward (im2col branch, src/backend.zig:3881-4065) on each tile of the split kernels,
    against fp64 on the reference's im2col; poison: an Inf in the input and a NaN in grad_output reach exactly the results
    they reach in fp64.  The kernels taken: test_forced_convolution_tiles."""
    from oracle import oracle
    B, C, H, W, OC, ker, st, pd = case
    OH, OW = (H + 2 * pd - ker) // st + 1, (W + 2 * pd - ker) // st + 1
    rng = np.random.default_rng(sum(case))
    x, w = uniform(rng, (B, C, H, W)), uniform(rng, (OC, ker * ker * C))
    bias, g = uniform(rng, (OC,)), uniform(rng, (B * OH * OW, OC))
    if poison:
        x[B - 1, 3, H // 2, W - 1] = np.inf
        g[7, 2] = np.nan
    dx, dw, db, dg = (ctx.to_device(a) for a in (x, w, bias, g))
    y, gx, gw, gb = (ctx.alloc(n).fill(0.5) for n in (B * OC * OH * OW, x.size, w.size, OC))
    geom = (B, C, OC, ker, ker, H, W, OH, OW, st, st, pd, pd)
    announce(f"split convolution {case} {tile} poison {poison}")
    with forced(ctx, tile):
        ctx.conv2d_forward_im2col(dx, dw, db, y, *geom)
        ctx.conv2d_backward_im2col(dx, dw, dg, gx, gw, gb, *geom)
    col = oracle.im2col(x, B, C, H, W, ker, ker, stride=(st, st), pad=(pd, pd)).reshape(B * OH * OW, -1).astype(np.float64)
    w64, g64 = w.astype(np.float64), g.astype(np.float64)

    def check(got, ref, den, k, what):
        fin = np.isfinite(ref)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(ref), err_msg=what)
        np.testing.assert_array_equal(np.isinf(got), np.isinf(ref), err_msg=what)
        assert np.all(np.abs(got[fin] - ref[fin]) <= (1e-5 if poison else 4e-7) * np.sqrt(k) * den[fin]), what

    with np.errstate(all="ignore"):
        taps = ker * ker * C
        ref = col @ w64.T + bias
        den = np.where(np.isfinite(ref), np.nan_to_num(np.abs(col), posinf=0) @ np.abs(w64).T + np.abs(bias), 0)
        check(y.download().reshape(B, OC, OH * OW).transpose(0, 2, 1).reshape(-1, OC), ref, den, taps, "forward")
        ref = g64.T @ col
        den = np.nan_to_num(np.abs(g64)).T @ np.nan_to_num(np.abs(col), posinf=0)
        check(gw.download().reshape(OC, taps), ref, den, B * OH * OW, "weight gradient")
        gcol, dcol = g64 @ w64, np.nan_to_num(np.abs(g64)) @ np.abs(w64)
        ref, den = (np.zeros((B, H + 2 * pd, W + 2 * pd, C)) for _ in range(2))
        for kh in range(ker):
            for kw in range(ker):
                at = np.s_[:, kh:kh + st * OH:st, kw:kw + st * OW:st]
                sl = np.s_[:, (kh * ker + kw) * C:(kh * ker + kw + 1) * C]
                ref[at] += gcol[sl].reshape(B, OH, OW, C)
                den[at] += dcol[sl].reshape(B, OH, OW, C)
        inner = np.s_[:, pd:pd + H, pd:pd + W]
        check(gx.download().reshape(B, C, H, W).transpose(0, 2, 3, 1), ref[inner], den[inner], taps // C * OC, "input gradient")
    for b in (dx, dw, db, dg, y, gx, gw, gb):
        b.close()


@pytest.mark.parametrize("case", [CONVS[0], CONVS[1]])
def test_forced_convolution_tiles(ctx, case):
    """Forward, input and weight gradient take the forced kernels: unsplit in K, both split tiles give the same bits and
    the fp32 64x64 tile others."""
    B, C, H, W, OC, ker, st, pd = case
    OH, OW = (H + 2 * pd - ker) // st + 1, (W + 2 * pd - ker) // st + 1
    rng = np.random.default_rng(31)
    x, w, bias, g = (uniform(rng, n) for n in ((B, C, H, W), (OC, ker * ker * C), (OC,), (B * OH * OW, OC)))
    dx, dw, db, dg = (ctx.to_device(v) for v in (x, w, bias, g))
    y, gx, gw, gb = (ctx.alloc(n) for n in (B * OC * OH * OW, x.size, w.size, OC))
    geom = (B, C, OC, ker, ker, H, W, OH, OW, st, st, pd, pd)
    out = {}
    for tile in ("conv128x128s", "conv64x128s", "64x64"):
        announce(f"forced convolution {case} {tile}")
        with forced(ctx, tile, 1):
            ctx.conv2d_forward_im2col(dx, dw, db, y, *geom)
            ctx.conv2d_backward_im2col(dx, dw, dg, gx, gw, gb, *geom)
        out[tile] = [v.download().view(np.uint32) for v in (y, gx, gw)]
    for i, what in enumerate(("forward", "input gradient", "weight gradient")):
        np.testing.assert_array_equal(out["conv128x128s"][i], out["conv64x128s"][i], err_msg=what)
        assert not np.array_equal(out["conv128x128s"][i], out["64x64"][i]), what
    for b in (dx, dw, db, dg, y, gx, gw, gb):
        b.close()


def test_split_convolution_non_finite_far_into_a_long_col(ctx):
    """One image of 512 x 512 x 256 under 3x3: its col matrix has more than 2^29 values, and value (pixel 455 * 512 + 56,
    tap (2, 2) of channel 0) is number 2^29, byte 2^31.  An Inf there reaches exactly the outputs, input gradients and
    weight gradients that it reaches in the reference's im2col (src/backend.zig:3881-4065).  Everything else is 1, so
    every other value is a count, exact in fp32 in any order."""
    C, H, W = 256, 512, 512
    assert (455 * W + 56) * 9 * C + 8 * C == 2 ** 29
    dx, dg = ctx.alloc(C * H * W).fill(1.0), ctx.alloc(H * W * C).fill(1.0)
    dw, db = ctx.alloc(C * 9 * C).fill(1.0), ctx.alloc(C).fill(0.0)
    y, gx, gw, gb = (ctx.alloc(n).fill(0.5) for n in (C * H * W, C * H * W, C * 9 * C, C))
    inf = ctx.to_device(np.full(1, np.inf, np.float32))
    ctx.copy(dx.offset(456 * W + 57), inf.ptr, 1)        # channel 0 (NCHW)
    ctx.copy(dg.offset((454 * W + 55) * C), inf.ptr, 1)  # output channel 0 ([pixel][channel])
    geom = (1, C, C, 3, 3, H, W, H, W, 1, 1, 1, 1)
    announce("split convolution, Inf at byte 2^31 of col")
    ctx.conv2d_forward_im2col(dx, dw, db, y, *geom)
    ctx.conv2d_backward_im2col(dx, dw, dg, gx, gw, gb, *geom)
    rows = np.r_[2.0, np.full(H - 2, 3.0), 2.0]  # taps that lie in the image
    want = np.outer(rows, rows).astype(np.float32) * C
    fwd, back = want.copy(), want.copy()
    fwd[455:458, 56:59] = np.inf
    back[453:456, 54:57] = np.inf
    for got, ref, what in ((y, fwd, "forward"), (gx, back, "input gradient")):
        got = got.download().reshape(C, H, W)
        assert all(np.array_equal(got[c], ref) for c in range(C)), what
    span = np.r_[H - 1.0, H, H - 1.0]
    wgrad = np.broadcast_to(np.outer(span, span).reshape(1, 9, 1), (C, 9, C)).astype(np.float32).copy()
    wgrad[0], wgrad[:, :, 0] = np.inf, np.inf
    np.testing.assert_array_equal(gw.download().reshape(C, 9, C), wgrad)
    for b in (dx, dg, dw, db, y, gx, gw, gb, inf):
        b.close()
