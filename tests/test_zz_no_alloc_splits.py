"""amd_matmul_no_alloc where the matmul op splits K into partial sums of more than 8 MiB: the library's scratch holds them, so the
call leaves the bits that the op leaves with any workspace that is large enough."""
import numpy as np
import pytest

import test_zz_no_alloc as small
from ml_dataflow_amd import binding as B
from util import normal_bf16

pytestmark = pytest.mark.gpu

BF = B.DATAFLOW_BF16


@pytest.mark.parametrize("workspace_bytes", [64 << 20, 100 << 20])
@pytest.mark.parametrize("transa,transb,M,K,N,beta", [(0, 1, 1536, 6520, 1536, 1.0), (0, 1, 3456, 7200, 640, 1.0), (0, 1, 2176, 8264, 1152, 0.0), (1, 0, 2176, 8264, 1152, 1.0),
                                                     (1, 0, 64, 2880, 33, 0.0)])
def test_equals_the_op_with_a_workspace_that_holds_its_split(backend, transa, transb, M, K, N, beta, workspace_bytes):
    print("case no-alloc split ta=%d tb=%d M=%d K=%d N=%d" % (transa, transb, M, K, N), flush=True)
    be, fn = backend, small.entry_point()
    rng = np.random.default_rng(M + K + N)
    A, Bm, Cin = normal_bf16(rng, (M * K,), 0.05), normal_bf16(rng, (N * K,)), normal_bf16(rng, (N * M,))
    d_A, d_B, d_op, d_here, d_ws = be.upload(A), be.upload(Bm), be.upload(Cin), be.upload(Cin), be.alloc(workspace_bytes)
    c_dt = BF if beta else B.DATAFLOW_NONE
    assert be.lib.dataflow_submit_matmul(be.hp, 1, BF, BF, c_dt, BF, B.DATAFLOW_FP32, transa, transb, M, K, N, 1.0, beta,
                                         d_A.ptr, d_B.ptr, d_op.ptr if beta else None, d_op.ptr, workspace_bytes, d_ws.ptr) == 0
    assert fn(be.hp, 1, transa, transb, M, K, N, 1.0, beta, d_A.ptr, d_B.ptr, d_here.ptr if beta else None, d_here.ptr) == 0
    be.sync(1)
    assert (be.read(d_op.ptr, (N, M), np.uint16) == be.read(d_here.ptr, (N, M), np.uint16)).all()
    for buf in (d_A, d_B, d_op, d_here, d_ws):
        buf.free()
