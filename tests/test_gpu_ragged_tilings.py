"""The tilings of a ragged-N launch without C (token rows in tiles of 288, 384, 224 or 192, chosen from the group sizes)
against the one of 288 rows: bit for bit.  Every element is accumulated over k in the same order whatever the tile."""
import ctypes as C
import os

import numpy as np
import pytest

from ml_dataflow_amd import binding as B
from util import normal_bf16

pytestmark = pytest.mark.gpu

BF, CS = B.DATAFLOW_BF16, 1
AUTO, EIGHT = 0, 8

# mean rows that the short tilings are candidates at (170: 192 rows, 430: 224, 650 x 3 m-tiles: three rounds of either),
# with groups on both sides of one, two and three tiles; the last two are so uneven that another candidate wins
COUNTS = {
    "192": [170, 191, 192, 160, 165, 150, 168, 180, 155, 172, 166, 190, 1, 0, 192, 187] * 2,
    "224": [430, 447, 448, 425, 410, 420, 435, 400, 445, 415, 428, 223, 224, 432, 440, 444] * 2,
    "three": [650, 575, 576, 577, 671, 672, 640, 660, 655, 630, 645, 670, 668, 600, 620, 665] * 2,
    "one large": [2000] + [110] * 30 + [1],
    "spilling": [449, 450, 193, 385, 580, 673, 455, 460] * 4,
}


@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("transa", [1, 0])
@pytest.mark.parametrize("name", sorted(COUNTS))
@pytest.mark.parametrize("M,K", [(1408, 1536), (1000, 1544)])      # whole k-tiles; a k tail, a partial m-tile, no 384 rows
def test_tilings_bit_identical(backend, M, K, name, transa, gathered):
    be = backend
    lib = C.CDLL(os.path.join(os.path.dirname(B.__file__), "lib", "libamd_matmul.so"))
    lib.amd_matmul_select_kernel.argtypes = [C.c_int]
    counts = np.array(COUNTS[name], dtype=np.int32)
    G, total, src_rows = len(counts), int(counts.sum()), 777
    print("case tilings %s M=%d K=%d ta=%d gathered=%s rows=%d" % (name, M, K, transa, gathered, total), flush=True)
    rng = np.random.default_rng(M + K + total + transa)
    W = normal_bf16(rng, (G * M * K,), 0.05)
    X = normal_bf16(rng, (src_rows if gathered else total, K))
    d_W, d_X, d_cum = be.upload(W), be.upload(X), be.upload(np.cumsum(counts).astype(np.int32))
    d_map = be.upload(rng.integers(0, src_rows, size=total).astype(np.int32))
    guard = 64                                                         # rows behind the last group keep their value
    got = {}
    for kernel in (EIGHT, AUTO):
        d_D = be.upload(np.full((total + guard, M), 0x4242, dtype=np.uint16))
        assert lib.amd_matmul_select_kernel(kernel) == 0
        head = (be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, transa, 0, B.AMD_GROUPED_RAGGED_N, M, K, total, G, d_cum.ptr, 1.0, 0.0,
                d_W.ptr, M * K * 2, d_X.ptr, None, d_D.ptr, 0)
        ret = be.lib.dataflow_submit_amd_grouped_matmul_gathered(*head, d_map.ptr, src_rows) if gathered else be.lib.dataflow_submit_amd_grouped_matmul(*head)
        assert lib.amd_matmul_select_kernel(AUTO) == 0
        assert ret == 0
        be.sync(CS)
        got[kernel] = be.read(d_D.ptr, (total + guard, M), np.uint16)
        d_D.free()
    assert (got[AUTO][total:] == 0x4242).all() and (got[EIGHT][total:] == 0x4242).all()
    bad = got[AUTO] != got[EIGHT]
    assert not bad.any(), "%d of %d elements differ, first at %s" % (int(bad.sum()), bad.size, np.argwhere(bad)[:4].tolist())
    for d in (d_W, d_X, d_cum, d_map):
        d.free()


@pytest.mark.parametrize("kernel,M,K,rows", [(AUTO, 72, 64, 2000), (EIGHT, 256, 64, 33400), (384, 256, 128, 50000)])
@pytest.mark.parametrize("G", [1, 2, 63, 64, 65, 127, 128, 129, 200])
def test_group_of_every_row_at_the_edges_of_the_scan(backend, G, kernel, M, K, rows):
    """The group of a tile is found by a scan over 64 groups at a time: group counts on both sides of one, two and three
    steps, empty groups at the lanes where a step begins and ends.  The operands are whole numbers whose sums bf16 holds
    exactly (at most 256), so the result is exact."""
    print("case scan G=%d kernel=%d M=%d K=%d" % (G, kernel, M, K), flush=True)
    be = backend
    lib = C.CDLL(os.path.join(os.path.dirname(B.__file__), "lib", "libamd_matmul.so"))
    lib.amd_matmul_select_kernel.argtypes = [C.c_int]
    rng = np.random.default_rng(G + M)
    share = rng.random(G) + 0.1
    for g in (0, 15, 16, 31, 32, 62, 63, 64, 126, 127, 128, 191):
        if g < G - 1:
            share[g] = 0.0
    counts = np.floor(share / share.sum() * rows).astype(np.int64)
    counts[-1] += rows - counts.sum()
    W = rng.integers(-2, 3, size=(G, M, K)).astype(np.float32)
    X = rng.integers(-2, 3, size=(rows, K)).astype(np.float32)
    X[:, 256 // 4:] = 0.0                                              # |sum| <= 64 products of at most 4
    as_bf16 = lambda a: (a.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    want, row = np.empty((rows, M), dtype=np.float32), 0
    for g in range(G):
        want[row:row + counts[g]] = X[row:row + counts[g]] @ W[g].T
        row += int(counts[g])
    d_W, d_X, d_cum, d_D = be.upload(as_bf16(W)), be.upload(as_bf16(X)), be.upload(np.cumsum(counts).astype(np.int32)), be.alloc(rows * M * 2)
    assert lib.amd_matmul_select_kernel(kernel) == 0
    ret = be.lib.dataflow_submit_amd_grouped_matmul(be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 1, 0, B.AMD_GROUPED_RAGGED_N, M, K, rows, G,
                                                    d_cum.ptr, 1.0, 0.0, d_W.ptr, M * K * 2, d_X.ptr, None, d_D.ptr, 0)
    assert lib.amd_matmul_select_kernel(AUTO) == 0
    assert ret == 0
    be.sync(CS)
    assert (be.read(d_D.ptr, (rows, M), np.uint16) == as_bf16(want)).all()
    for d in (d_W, d_X, d_cum, d_D):
        d.free()


# rows of a group on both sides of one tile of 32, 64 and 128 rows, each mean on another of those tiles
FEW_ROWS = {
    "32": [0, 1, 31, 32, 33, 2, 16, 64, 65, 0, 30, 7, 32, 31, 5, 1],
    "64": [63, 64, 65, 1, 0, 32, 33, 128, 129, 60, 64, 63, 40, 90, 50, 64],
    "128": [127, 128, 129, 255, 256, 257, 0, 1, 100, 128, 127, 140, 90, 120, 128, 110],
    "96 in the mean": [127, 128, 129, 1, 0, 100, 128, 127, 90, 120, 128, 10, 64, 255, 126, 3],
}


@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("transa", [1, 0])
@pytest.mark.parametrize("name", sorted(FEW_ROWS))
def test_streamed_weights_bit_identical(backend, name, transa, gathered):
    """16 groups with 64 MiB of weights: enough that those of groups with one tile of rows are loaded non-temporally where the mean group has one; against one plain
    matmul a group, which loads them as ever.  Every element is accumulated over k in the same order: bit for bit."""
    be, M, K = backend, 2048, 1032
    counts = np.array(FEW_ROWS[name], dtype=np.int32)
    G, total, src_rows = len(counts), int(counts.sum()), 333
    print("case streamed weights %s ta=%d gathered=%s rows=%d" % (name, transa, gathered, total), flush=True)
    rng = np.random.default_rng(total + transa)
    W, X, row_map = normal_bf16(rng, (G * M * K,), 0.05), normal_bf16(rng, (src_rows if gathered else total, K)), rng.integers(0, src_rows, size=total).astype(np.int32)
    ends = np.cumsum(counts).astype(np.int32)
    d_W, d_X, d_packed, d_cum, d_map = be.upload(W), be.upload(X), be.upload(np.ascontiguousarray(X[row_map]) if gathered else X), be.upload(ends), be.upload(row_map)
    d_D, d_E = (be.upload(np.full((total, M), 0x4242, dtype=np.uint16)) for _ in range(2))
    head = (be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, transa, 0, B.AMD_GROUPED_RAGGED_N, M, K, total, G, d_cum.ptr, 1.0, 0.0,
            d_W.ptr, M * K * 2, d_X.ptr, None, d_D.ptr, 0)
    assert (be.lib.dataflow_submit_amd_grouped_matmul_gathered(*head, d_map.ptr, src_rows) if gathered else be.lib.dataflow_submit_amd_grouped_matmul(*head)) == 0
    for g in range(G):
        first = int(ends[g] - counts[g])
        assert be.lib.dataflow_submit_matmul(be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, transa, 0, M, K, int(counts[g]), 1.0, 0.0,
                                             d_W.ptr + g * M * K * 2, d_packed.ptr + first * K * 2, None, d_E.ptr + first * M * 2, 0, None) == 0
    be.sync(CS)
    bad = be.read(d_D.ptr, (total, M), np.uint16) != be.read(d_E.ptr, (total, M), np.uint16)
    assert not bad.any(), "%d of %d elements differ, first at %s" % (int(bad.sum()), bad.size, np.argwhere(bad)[:4].tolist())
    for d in (d_W, d_X, d_packed, d_cum, d_map, d_D, d_E):
        d.free()
