"""GPU parity of the RMS norm operators around the MoE layer against the CPU oracle, through the C ABI
(dataflow_submit_default_rms_norm* -> handle->submit_op -> gfx950 kernel).

Bar: the saved statistic within 1e-5 relative (fp32 sums in a different order); bf16 outputs within 1 bf16 step
of the oracle's result where only a product chain is involved (forward, recompute), and within 1e-2 of the
tensor's scale where a sum feeds every element (backward), typically 1 step."""
import numpy as np
import pytest

import oracle_lib as O
from ml_dataflow_amd import binding as B
from util import f32_to_bf16, bf16_to_f64, normal_bf16, bf16_ulp_diff

pytestmark = pytest.mark.gpu

BF = B.DATAFLOW_BF16
CS = 1
EPS = 1e-5


def close(got, want, tol=1e-2):
    g, w = bf16_to_f64(got), bf16_to_f64(want)
    scale = max(float(np.abs(w).max()), 1e-30)
    assert float(np.abs(g - w).max()) <= tol * scale


# 16384 and 10000 columns exceed what a work-group keeps in registers (8192): the second-pass path
SHAPES = [(1, 8), (3, 64), (100, 4096), (257, 2048), (33, 1000), (5, 16384), (7, 10000)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_rms_norm_forward_and_recompute(backend, oracle, rows, cols):
    print("case rms_norm rows=%d cols=%d" % (rows, cols), flush=True)
    be = backend
    rng = np.random.default_rng(rows * 7 + cols)
    X = normal_bf16(rng, (rows, cols), 1.5)
    W = f32_to_bf16(1.0 + 0.1 * rng.standard_normal(cols).astype(np.float32))
    d_X, d_W = be.upload(X), be.upload(W)
    d_out, d_rms, d_out2 = be.alloc(rows * cols * 2), be.alloc(rows * 4), be.alloc(rows * cols * 2)
    assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, rows, cols, EPS, d_W.ptr, d_X.ptr, d_out.ptr, d_rms.ptr) == 0
    assert be.lib.dataflow_submit_default_rms_norm_recompute(be.hp, CS, BF, rows, cols, d_W.ptr, d_rms.ptr, d_X.ptr, d_out2.ptr) == 0
    be.sync(CS)
    want, rms = np.zeros_like(X), np.zeros(rows, np.float32)
    oracle.oracle_rms_norm(rows, cols, EPS, O.ptr(W), O.ptr(X), O.ptr(want), O.ptr(rms))
    g_rms = be.read(d_rms.ptr, (rows,), np.float32)
    np.testing.assert_allclose(g_rms, rms, rtol=1e-5)
    got = be.read(d_out.ptr, (rows, cols), np.uint16)
    assert bf16_ulp_diff(got, want).max() <= 1
    # recompute uses the GPU's own statistic: identical bits to the forward output
    assert (be.read(d_out2.ptr, (rows, cols), np.uint16) == got).all()
    # the statistic is optional, and the output may alias the input
    assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, rows, cols, EPS, d_W.ptr, d_X.ptr, d_X.ptr, None) == 0
    be.sync(CS)
    assert (be.read(d_X.ptr, (rows, cols), np.uint16) == got).all()


# rows on one wave, four to a work-group (8192 rows and more of up to 1024 columns), and unrolled ones (2500 and more of over 4608) give the bits of rows on a work-group (two calls of half the rows)
@pytest.mark.parametrize("rows,cols", [(8192, 8), (8193, 64), (8195, 512), (8194, 520), (8192, 1016), (8193, 1024), (8192, 1032),
                                       (2500, 4608), (2500, 4616), (2501, 8192), (2500, 8200)])
def test_rms_norm_rows_on_a_wave_and_unrolled(backend, rows, cols):
    print("case rms_norm rows=%d cols=%d" % (rows, cols), flush=True)
    be = backend
    rng = np.random.default_rng(rows * 3 + cols)
    X = normal_bf16(rng, (rows, cols), 1.5)
    X[5], X[6, 0], X[7, cols - 1] = 0, 0x7F80, 0x7FC0                  # a row of zeros, an infinity, a NaN
    W = f32_to_bf16(1.0 + 0.1 * rng.standard_normal(cols).astype(np.float32))
    d_X, d_W = be.upload(X), be.upload(W)
    d_out, d_rms, d_part, d_prms = be.alloc(rows * cols * 2), be.alloc(rows * 4), be.alloc(rows * cols * 2), be.alloc(rows * 4)
    assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, rows, cols, EPS, d_W.ptr, d_X.ptr, d_out.ptr, d_rms.ptr) == 0
    half = rows // 2
    for first, n in ((0, half), (half, rows - half)):
        at = first * cols * 2
        assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, n, cols, EPS, d_W.ptr, d_X.ptr + at, d_part.ptr + at, d_prms.ptr + first * 4) == 0
    be.sync(CS)
    assert (be.read(d_rms.ptr, (rows,), np.uint32) == be.read(d_prms.ptr, (rows,), np.uint32)).all()
    assert (be.read(d_out.ptr, (rows, cols), np.uint16) == be.read(d_part.ptr, (rows, cols), np.uint16)).all()
    # the statistic is optional, and the output may alias the input
    assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, rows, cols, EPS, d_W.ptr, d_X.ptr, d_X.ptr, None) == 0
    be.sync(CS)
    assert (be.read(d_X.ptr, (rows, cols), np.uint16) == be.read(d_part.ptr, (rows, cols), np.uint16)).all()


@pytest.mark.parametrize("with_out", [True, False])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_rms_norm_bwd_x(backend, oracle, rows, cols, with_out):
    print("case rms_norm_bwd_x rows=%d cols=%d out=%d" % (rows, cols, with_out), flush=True)
    be = backend
    rng = np.random.default_rng(rows * 11 + cols)
    X, G = normal_bf16(rng, (rows, cols), 1.5), normal_bf16(rng, (rows, cols))
    W = f32_to_bf16(1.0 + 0.1 * rng.standard_normal(cols).astype(np.float32))
    start = normal_bf16(rng, (rows, cols), 0.5)
    rms, fwd = np.zeros(rows, np.float32), np.zeros_like(X)
    oracle.oracle_rms_norm(rows, cols, EPS, O.ptr(W), O.ptr(X), O.ptr(fwd), O.ptr(rms))
    d_X, d_G, d_W, d_rms, d_dX = be.upload(X), be.upload(G), be.upload(W), be.upload(rms), be.upload(start)
    d_out = be.alloc(rows * cols * 2)
    assert be.lib.dataflow_submit_default_rms_norm_bwd_x(be.hp, CS, BF, BF, rows, cols, EPS, d_rms.ptr, d_W.ptr, d_X.ptr, d_G.ptr,
                                                         d_dX.ptr, d_out.ptr if with_out else None) == 0
    be.sync(CS)
    want, want_out = start.copy(), np.zeros_like(X)
    oracle.oracle_rms_norm_bwd_x(rows, cols, EPS, O.ptr(rms), O.ptr(W), O.ptr(X), O.ptr(G), O.ptr(want), O.ptr(want_out))
    close(be.read(d_dX.ptr, (rows, cols), np.uint16), want)
    assert np.percentile(bf16_ulp_diff(be.read(d_dX.ptr, (rows, cols), np.uint16), want), 99) <= 1
    if with_out:
        assert (be.read(d_out.ptr, (rows, cols), np.uint16) == want_out).all()      # a product chain of the same inputs


@pytest.mark.parametrize("rows,cols,groups", [(1, 8, 4), (100, 4096, 512), (1000, 2048, 512), (777, 1000, 3), (64, 16384, 1), (9000, 64, 512)])
def test_rms_norm_bwd_w(backend, oracle, rows, cols, groups):
    print("case rms_norm_bwd_w rows=%d cols=%d groups=%d" % (rows, cols, groups), flush=True)
    be = backend
    rng = np.random.default_rng(rows + cols)
    X, G = normal_bf16(rng, (rows, cols)), normal_bf16(rng, (rows, cols))
    rms = (0.5 + rng.random(rows)).astype(np.float32)
    start = normal_bf16(rng, (cols,))
    d_X, d_G, d_rms, d_dW = be.upload(X), be.upload(G), be.upload(rms), be.upload(start)
    ws_bytes = 256 + groups * cols * 4                       # room for exactly `groups` partial rows
    d_ws = be.alloc(ws_bytes)
    assert be.lib.dataflow_submit_default_rms_norm_bwd_w(be.hp, CS, BF, BF, rows, cols, EPS, d_rms.ptr, d_X.ptr, d_G.ptr, d_dW.ptr,
                                                         ws_bytes, d_ws.ptr) == 0
    be.sync(CS)
    launched = int(be.read(d_ws.ptr, (1,), np.int32)[0])
    assert launched == min(groups, rows, 512)
    want = start.copy()
    oracle.oracle_rms_norm_bwd_w(rows, cols, EPS, O.ptr(rms), O.ptr(X), O.ptr(G), O.ptr(want))
    got = be.read(d_dW.ptr, (cols,), np.uint16)
    close(got, want)
    assert np.percentile(bf16_ulp_diff(got, want), 99) <= 1


@pytest.mark.parametrize("rows", [1, 2, 127, 128, 129, 511, 1024, 1535, 1536, 1537])
@pytest.mark.parametrize("cols", [8, 56, 72, 520])
def test_rms_norm_bwd_w_few_rows_and_more(backend, rows, cols):
    """One launch up to 1536 rows, two above: row counts at the edges of its 128 row lanes and of the rule, columns at those of
    its 64.  Whole numbers whose sums fp32 holds exactly in any order, so the result is exact up to its rounding to bf16."""
    print("case rms_norm_bwd_w few rows=%d cols=%d" % (rows, cols), flush=True)
    be = backend
    rng = np.random.default_rng(rows + cols)
    x, g = rng.integers(-4, 5, (rows, cols)), rng.integers(-4, 5, (rows, cols))
    rms = np.exp2(rng.integers(-1, 2, rows)).astype(np.float32)
    start = rng.integers(-8, 9, cols)
    d_X, d_G, d_rms, d_dW = be.upload(f32_to_bf16(x.astype(np.float32))), be.upload(f32_to_bf16(g.astype(np.float32))), be.upload(rms), be.upload(f32_to_bf16(start.astype(np.float32)))
    ws_bytes = 256 + 512 * cols * 4
    d_ws = be.alloc(ws_bytes)
    assert be.lib.dataflow_submit_default_rms_norm_bwd_w(be.hp, CS, BF, BF, rows, cols, EPS, d_rms.ptr, d_X.ptr, d_G.ptr, d_dW.ptr, ws_bytes, d_ws.ptr) == 0
    be.sync(CS)
    assert int(be.read(d_ws.ptr, (1,), np.int32)[0]) == min(rows, 512)
    want = f32_to_bf16((start + (x * g * rms[:, None].astype(np.float64)).sum(axis=0)).astype(np.float32))
    assert (be.read(d_dW.ptr, (cols,), np.uint16) == want).all()


@pytest.mark.parametrize("rows,cols", [(1537, 4600), (1537, 4608), (4099, 4600), (4099, 4608), (6200, 72), (2048, 6152)])
def test_rms_norm_bwd_w_rows_in_fours_and_one_by_one(backend, rows, cols):
    """Three to twelve rows a work-group, on both sides of the row length from which on they go one by one.  Whole numbers as above: exact."""
    print("case rms_norm_bwd_w fours rows=%d cols=%d" % (rows, cols), flush=True)
    be = backend
    rng = np.random.default_rng(rows + cols)
    x, g = rng.integers(-4, 5, (rows, cols)).astype(np.float32), rng.integers(-4, 5, (rows, cols)).astype(np.float32)
    rms = np.exp2(rng.integers(-1, 2, rows)).astype(np.float32)
    d_X, d_G, d_rms, d_dW = be.upload(f32_to_bf16(x)), be.upload(f32_to_bf16(g)), be.upload(rms), be.upload(np.zeros(cols, np.uint16))
    ws_bytes = 256 + 512 * cols * 4
    d_ws = be.alloc(ws_bytes)
    assert be.lib.dataflow_submit_default_rms_norm_bwd_w(be.hp, CS, BF, BF, rows, cols, EPS, d_rms.ptr, d_X.ptr, d_G.ptr, d_dW.ptr, ws_bytes, d_ws.ptr) == 0
    be.sync(CS)
    want = f32_to_bf16(np.einsum("rc,r->c", x * g, rms, dtype=np.float64).astype(np.float32))
    assert (be.read(d_dW.ptr, (cols,), np.uint16) == want).all()


@pytest.mark.parametrize("with_out", [True, False])
@pytest.mark.parametrize("rows,cols", [(1536, 64), (1536, 4104), (1536, 8200), (1537, 64), (1537, 2056), (1537, 8192), (1537, 8200), (1800, 6152),
                                       (8192, 8), (8193, 64), (8195, 512), (8194, 520), (8193, 1024), (8192, 1032)])
def test_rms_norm_bwd_x_with_few_rows_and_more(backend, rows, cols, with_out):
    """Up to 1536 rows and beyond are two forms of one kernel, 8192 rows of up to 1024 columns, one on a wave, have their own: a row's result has the same
    bits from each.  The first 700 rows alone run on the first form, and so do all 1536."""
    print("case rms_norm_bwd_x forms rows=%d cols=%d out=%d" % (rows, cols, with_out), flush=True)
    be = backend
    rng = np.random.default_rng(rows + cols)
    X, G, W, start = normal_bf16(rng, (rows, cols), 1.5), normal_bf16(rng, (rows, cols)), normal_bf16(rng, (cols,)), normal_bf16(rng, (rows, cols), 0.5)
    rms = (0.5 + rng.random(rows)).astype(np.float32)
    d_X, d_G, d_W, d_rms = be.upload(X), be.upload(G), be.upload(W), be.upload(rms)
    got = {}
    for n in (700, rows):
        d_dX, d_out = be.upload(start), be.upload(np.full((rows, cols), 0x4242, np.uint16))
        assert be.lib.dataflow_submit_default_rms_norm_bwd_x(be.hp, CS, BF, BF, n, cols, EPS, d_rms.ptr, d_W.ptr, d_X.ptr, d_G.ptr, d_dX.ptr, d_out.ptr if with_out else None) == 0
        be.sync(CS)
        got[n] = be.read(d_dX.ptr, (rows, cols), np.uint16), be.read(d_out.ptr, (rows, cols), np.uint16)
        assert (got[n][0][n:] == start[n:]).all() and (got[n][1][n if with_out else 0:] == 0x4242).all()
    for few, many in zip(got[700], got[rows]):
        assert (few[:700] == many[:700]).all()
    assert (got[rows][0] != start).any(axis=1).all()


def test_rms_norm_rejects_bad_shapes_and_small_workspace(backend):
    be = backend
    buf = be.alloc(4096)
    assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, 4, 12, EPS, buf.ptr, buf.ptr, buf.ptr, None) == -1     # row length not a multiple of 8
    assert be.lib.dataflow_submit_default_rms_norm_bwd_w(be.hp, CS, BF, BF, 4, 64, EPS, buf.ptr, buf.ptr, buf.ptr, buf.ptr, 300, buf.ptr) == -1
    assert be.lib.dataflow_submit_default_rms_norm_bwd_w(be.hp, CS, BF, BF, 4, 64, EPS, buf.ptr, buf.ptr, buf.ptr, buf.ptr, 4096, None) == -1
    # zero rows: nothing is launched, nothing fails
    assert be.lib.dataflow_submit_default_rms_norm(be.hp, CS, BF, 0, 64, EPS, buf.ptr, buf.ptr, buf.ptr, None) == 0
    be.sync(CS)
