"""What the four-wave GEMM kernels do between two tiles (epilogue, walk over the tiles), at the edges of tiles, groups and k-tiles:
bit for bit what the eight-wave kernel leaves, which test_gpu_ops.py holds to the oracle, and nothing past the end of D."""
import ctypes as C
import os

import numpy as np
import pytest

from ml_dataflow_amd import binding as B
from util import normal_bf16

pytestmark = pytest.mark.gpu

BF = B.DATAFLOW_BF16
CS = 1
AUTO, EIGHT, FOUR_384 = 0, 8, 384
GUARD = 4096            # elements behind D that have to stay as they are


@pytest.fixture(scope="module")
def select_kernel(backend):
    lib = C.CDLL(os.path.join(os.path.dirname(B.__file__), "lib", "libamd_matmul.so"))
    lib.amd_matmul_select_kernel.argtypes = [C.c_int]
    lib.amd_matmul_planned_sliced.argtypes = [C.c_int] * 6
    yield lib.amd_matmul_select_kernel
    assert lib.amd_matmul_select_kernel(AUTO) == 0


def runs_sliced(select_kernel, kernel, M, K, N, groups, has_c):
    """what the library says of a launch (amd_matmul_plan.h): a comparison of the eight-wave kernel with itself shows nothing"""
    lib = C.CDLL(os.path.join(os.path.dirname(B.__file__), "lib", "libamd_matmul.so"))
    assert select_kernel(kernel) == 0
    sliced = lib.amd_matmul_planned_sliced(M, K, N, groups, int(has_c), 256)
    assert select_kernel(AUTO) == 0
    return sliced == 1


def both(be, select_kernel, other, elements, start, submit):
    """D of the eight-wave kernel and of `other`, from the same values in it, and the guard behind the second"""
    got = {}
    filled = np.concatenate([start.reshape(-1), np.full(GUARD, 0x4242, np.uint16)])
    for kernel in (EIGHT, other):
        d_D = be.upload(filled)
        assert select_kernel(kernel) == 0
        assert submit(d_D) == 0
        be.sync(CS)
        got[kernel] = be.read(d_D.ptr, (elements + GUARD,), np.uint16)
        d_D.free()
    assert select_kernel(AUTO) == 0
    assert (got[other][elements:] == 0x4242).all()
    bad = got[other] != got[EIGHT]
    assert not bad.any(), "%d of %d elements differ, first at %s" % (int(bad.sum()), bad.size, np.flatnonzero(bad)[:4].tolist())
    return got[other][:elements]


@pytest.mark.parametrize("transa", [1, 0])
@pytest.mark.parametrize("alpha", [1.0, -0.75])
@pytest.mark.parametrize("M,K,groups", [(1304, 128, 70), (520, 384, 64), (2048, 256, 130)])
def test_ragged_n_many_groups(backend, select_kernel, transa, alpha, M, K, groups):
    """more groups than lanes, and as many; tiles partial in both directions; a work-group walks over many short tiles"""
    be = backend
    rng = np.random.default_rng(M + K + groups + transa)
    counts = rng.choice([0, 1, 95, 96, 97, 191, 193, 288, 383, 384, 385, 500], size=groups).astype(np.int32)
    counts[0], counts[-1] = 385, 97
    total = int(counts.sum())
    assert total // 256 * -(-M // 256) >= 128                          # from there on a named kernel runs, not the direct one on both sides
    print("case four waves, N: ta=%d alpha=%g M=%d K=%d G=%d rows=%d" % (transa, alpha, M, K, groups, total), flush=True)
    d_W = be.upload(normal_bf16(rng, (groups, M, K) if transa else (groups, K, M), 0.05))
    d_X, d_cum = be.upload(normal_bf16(rng, (total, K))), be.upload(np.cumsum(counts).astype(np.int32))
    both(be, select_kernel, FOUR_384, total * M, np.zeros(total * M, np.uint16), lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul(
        be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, transa, 0, B.AMD_GROUPED_RAGGED_N, M, K, total, groups, d_cum.ptr, alpha, 0.0,
        d_W.ptr, M * K * 2, d_X.ptr, None, d_D.ptr, 0))
    for d in (d_W, d_X, d_cum):
        d.free()


@pytest.mark.parametrize("transa", [1, 0])
@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("n_tiles", [20, 48, 60, 70, 112])
def test_ragged_n_partial_last_rounds(backend, select_kernel, n_tiles, gathered, transa):
    """A die's last round in pieces: the only round, in two (15 tiles for 32 work-groups), a second one in three and in two (4, 13), none (21), a third in
    two and three; tiles of few rows, that have fewer blocks of columns than pieces, and of a group of many tiles."""
    be = backend
    M, K, src_rows = 1304, 256, 997
    rng = np.random.default_rng(n_tiles + 2 * gathered + transa)
    counts = [3500] if n_tiles > 20 else []
    counts += [1] if n_tiles % 20 == 0 else []
    while sum(-(-c // 384) for c in counts) < n_tiles:
        counts.append(int(rng.choice([1, 63, 129, 193, 257, 320, 383, 384, 385, 449, 640, 768])))
        if sum(-(-c // 384) for c in counts) > n_tiles:
            counts[-1] = 384
    counts = np.array(counts[1:] + counts[:1], np.int32)
    total, groups = int(counts.sum()), len(counts)
    # the named kernel runs from this many rows on: an upper bound of them is what a launch is told
    most = max(total, 256 * 22)
    assert most // 256 * -(-M // 256) >= 128
    print("case partial last rounds: tiles=%d gathered=%d ta=%d rows=%d groups=%d" % (n_tiles, gathered, transa, total, groups), flush=True)
    d_W = be.upload(normal_bf16(rng, (groups, M, K) if transa else (groups, K, M), 0.05))
    d_X = be.upload(normal_bf16(rng, (src_rows if gathered else most, K)))
    d_cum, d_map = be.upload(np.cumsum(counts).astype(np.int32)), be.upload(rng.integers(-1, src_rows + 1, most).astype(np.int32))
    args = (be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, transa, 0, B.AMD_GROUPED_RAGGED_N, M, K, most, groups, d_cum.ptr, 1.0, 0.0,
            d_W.ptr, M * K * 2, d_X.ptr, None)
    if gathered:
        submit = lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul_gathered(*args, d_D.ptr, 0, d_map.ptr, src_rows)
    else:
        submit = lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul(*args, d_D.ptr, 0)
    both(be, select_kernel, FOUR_384, total * M, np.zeros(total * M, np.uint16), submit)
    for d in (d_W, d_X, d_cum, d_map):
        d.free()


@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("groups,tiles", [(20, 2), (33, 2), (16, 8), (20, 3), (17, 4)])
def test_ragged_n_groups_of_the_same_tiles(backend, select_kernel, groups, tiles, gathered):
    """Groups of as many tiles each, four tiles high: 8, 16 and 32 of them go into a die's 32 work-groups, whose last tiles are not cut then, 12 do not;
    partial last rounds, rows of a group from one in its last tile to all."""
    be = backend
    M, K, src_rows = 1016, 256, 997
    rng = np.random.default_rng(groups + tiles)
    counts = (384 * (tiles - 1) + rng.choice([1, 63, 64, 65, 128, 129, 192, 193, 257, 320, 383, 384], size=groups)).astype(np.int32)
    counts[0], counts[-1] = 384 * tiles, 384 * (tiles - 1) + 1
    total = int(counts.sum())
    assert total // 256 * -(-M // 256) >= 128                          # from there on a named kernel runs, not the direct one on both sides
    print("case groups of the same tiles: groups=%d tiles=%d gathered=%d rows=%d" % (groups, tiles, gathered, total), flush=True)
    d_W, d_X = be.upload(normal_bf16(rng, (groups, M, K), 0.05)), be.upload(normal_bf16(rng, (src_rows if gathered else total, K)))
    d_cum, d_map = be.upload(np.cumsum(counts).astype(np.int32)), be.upload(rng.integers(-1, src_rows + 1, total).astype(np.int32))
    args = (be.hp, CS, BF, BF, B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 1, 0, B.AMD_GROUPED_RAGGED_N, M, K, total, groups, d_cum.ptr, 1.0, 0.0, d_W.ptr, M * K * 2, d_X.ptr, None)
    if gathered:
        submit = lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul_gathered(*args, d_D.ptr, 0, d_map.ptr, src_rows)
    else:
        submit = lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul(*args, d_D.ptr, 0)
    both(be, select_kernel, FOUR_384, total * M, np.zeros(total * M, np.uint16), submit)
    for d in (d_W, d_X, d_cum, d_map):
        d.free()


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (1.0, 1.0), (-0.75, 0.0), (1.5, -0.5)])
@pytest.mark.parametrize("M,N,groups", [(264, 520, 64), (1304, 264, 70), (256, 256, 300)])
def test_ragged_k_tiles_and_slices(backend, select_kernel, alpha, beta, M, N, groups):
    """reductions of no slice to more than the ring holds, last slices of 1 to 32 k-rows; tiles partial in both directions"""
    be = backend
    rng = np.random.default_rng(M + N + groups)
    counts = rng.choice([0, 1, 31, 32, 33, 128, 159, 160, 161, 255, 256, 257, 352, 353, 500], size=groups).astype(np.int32)
    counts[0], counts[-1] = 353, 1
    total = int(counts.sum())
    rows = 2048 * groups                                               # what K says decides on the kernel only: here, that it is the sliced one
    assert runs_sliced(select_kernel, FOUR_384, M, rows, N, groups, beta)
    print("case four waves, K: alpha=%g beta=%g M=%d N=%d G=%d rows=%d" % (alpha, beta, M, N, groups, total), flush=True)
    d_A, d_B = be.upload(normal_bf16(rng, (total, M), 0.05)), be.upload(normal_bf16(rng, (total, N)))
    d_cum = be.upload(np.cumsum(counts).astype(np.int32))
    start = normal_bf16(rng, (groups, N, M))
    both(be, select_kernel, FOUR_384, groups * N * M, start, lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul(
        be.hp, CS, BF, BF, BF if beta else B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 0, 1, B.AMD_GROUPED_RAGGED_K, M, rows, N, groups, d_cum.ptr, alpha, beta,
        d_A.ptr, 0, d_B.ptr, d_D.ptr if beta else None, d_D.ptr, N * M * 2))
    for d in (d_A, d_B, d_cum):
        d.free()


@pytest.mark.parametrize("alpha,beta,M,N,K", [(1.0, 0.0, 4104, 4008, 1057), (1.0, 1.0, 4104, 4008, 545), (0.5, -2.0, 4104, 4008, 545),
                                              (1.0, 0.0, 2816, 4096, 2056), (1.0, 1.0, 2816, 4096, 1000), (0.5, -2.0, 2816, 4096, 1000),
                                              (1.0, 0.0, 4096, 4096, 2048), (1.0, 1.0, 4096, 4096, 256), (0.5, -2.0, 4096, 4096, 256)])
def test_k_major_operands_of_one_problem(backend, select_kernel, alpha, beta, M, N, K):
    """one or two tiles a work-group, partial ones in both directions, a last slice of one k-row, of eight, and a whole one"""
    assert runs_sliced(select_kernel, FOUR_384, M, K, N, 0, beta)
    be = backend
    rng = np.random.default_rng(M + N + K)
    print("case four waves, k-major: alpha=%g beta=%g M=%d N=%d K=%d" % (alpha, beta, M, N, K), flush=True)
    d_A, d_B, d_ws = be.upload(normal_bf16(rng, (K, M), 0.05)), be.upload(normal_bf16(rng, (K, N))), be.upload(np.zeros(1 << 20, np.uint8))
    both(be, select_kernel, FOUR_384, N * M, normal_bf16(rng, (N, M)), lambda d_D: be.lib.dataflow_submit_matmul(
        be.hp, CS, BF, BF, BF if beta else B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 0, 1, M, K, N, alpha, beta,
        d_A.ptr, d_B.ptr, d_D.ptr if beta else None, d_D.ptr, 1 << 20, d_ws.ptr))
    for d in (d_A, d_B, d_ws):
        d.free()


@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_ragged_k_by_default_with_c_apart_and_gaps_between_groups(backend, select_kernel, beta):
    """the caller's count of rows as K, no kernel named; C in an array of its own, which stays as it is; groups of D further apart than they are long"""
    be = backend
    M = N = 1016
    groups, gap = 32, 72
    rng = np.random.default_rng(5)
    counts = rng.choice([0, 1, 33, 352, 640, 700, 760, 1200], size=groups).astype(np.int32)
    counts[3], counts[-1] = 3500, 6000
    total = int(counts.sum())
    assert runs_sliced(select_kernel, AUTO, M, total, N, groups, beta)
    print("case four waves, K by default: beta=%g rows=%d" % (beta, total), flush=True)
    stride = N * M + gap
    d_A, d_B = be.upload(normal_bf16(rng, (total, M), 0.05)), be.upload(normal_bf16(rng, (total, N)))
    d_cum = be.upload(np.cumsum(counts).astype(np.int32))
    c = normal_bf16(rng, (groups * stride,))
    d_C = be.upload(c)
    start = np.full(groups * stride, 0x3131, np.uint16)

    def submit(d_D):
        return be.lib.dataflow_submit_amd_grouped_matmul(be.hp, CS, BF, BF, BF if beta else B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 0, 1, B.AMD_GROUPED_RAGGED_K, M, total, N, groups,
                                                         d_cum.ptr, 1.0, beta, d_A.ptr, 0, d_B.ptr, d_C.ptr if beta else None, d_D.ptr, stride * 2)
    d = both(be, select_kernel, AUTO, groups * stride, start, submit).reshape(groups, stride)
    assert (d[:, N * M:] == 0x3131).all()
    untouched = (counts == 0) & (beta != 0.0)
    assert (d[untouched] == 0x3131).all() and (d[~untouched, :N * M] != 0x3131).any(axis=1).all()
    assert (be.read(d_C.ptr, (groups * stride,), np.uint16) == c).all()
    for buffer in (d_A, d_B, d_C, d_cum):
        buffer.free()


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("M,N,groups", [(520, 264, 70), (1304, 512, 24)])
def test_ragged_k_gathered_rows_on_slices(backend, select_kernel, beta, M, N, groups):
    """Rows of a group on both sides of a slice, of the eight slices whose rows a wave holds and of the fewest a tile has; entries outside the
    source; groups without rows; more groups than lanes.  The sliced kernel against the eight-wave one, which gathers too."""
    be = backend
    counts = np.array([0, 1, 31, 32, 33, 255, 256, 257, 288, 289, 511, 512, 513, 0, 3000, 2047, 2048, 2049, 160, 161, 96, 768, 1025, 1500], dtype=np.int32)
    counts = np.concatenate([counts, np.full(groups - len(counts), 900, np.int32)])
    total, src_rows = int(counts.sum()), 1237
    # lines of the sliced kernel: 512 rows a group in the mean with C, 640 without
    assert runs_sliced(select_kernel, FOUR_384, M, total, N, groups, beta != 0.0) and total >= 640 * groups
    print("case gathered slices M=%d N=%d groups=%d rows=%d beta=%g" % (M, N, groups, total, beta), flush=True)
    rng = np.random.default_rng(M + groups)
    row_map = rng.integers(0, src_rows, total).astype(np.int32)
    row_map[rng.integers(0, total, 50)] = -1
    row_map[rng.integers(0, total, 50)] = src_rows
    d_A, d_B = be.upload(normal_bf16(rng, (src_rows, M))), be.upload(normal_bf16(rng, (total, N), 0.05))
    d_cum, d_map = be.upload(np.cumsum(counts).astype(np.int32)), be.upload(row_map)
    both(be, select_kernel, FOUR_384, groups * N * M, normal_bf16(rng, (groups * N * M,)),
         lambda d_D: be.lib.dataflow_submit_amd_grouped_matmul_gathered(be.hp, CS, BF, BF, BF if beta else B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 0, 1, B.AMD_GROUPED_RAGGED_K,
                                                                        M, total, N, groups, d_cum.ptr, 1.0, beta, d_A.ptr, 0, d_B.ptr, d_D.ptr if beta else None, d_D.ptr,
                                                                        N * M * 2, d_map.ptr, src_rows))
    for d in (d_A, d_B, d_cum, d_map):
        d.free()
