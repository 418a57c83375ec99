"""The up-projections of the grouped and the per-expert schedule under amd_matmul_select_kernel: a named kernel is obeyed there too
(two GEMMs and the activation instead of the fused launch, which only the small-tile kernel has), with the same bits."""
import ctypes as C
import os

import numpy as np
import pytest

from ml_dataflow_amd import MoeLayer, binding as B
from util import normal_bf16

pytestmark = pytest.mark.gpu

CS = 1
AUTO, EIGHT, FOUR_384 = 0, 8, 384
CAPTURE_RELAXED = 2


@pytest.fixture(scope="module")
def select_kernel(backend):
    lib = C.CDLL(os.path.join(os.path.dirname(B.__file__), "lib", "libamd_matmul.so"))
    lib.amd_matmul_select_kernel.argtypes = [C.c_int]
    yield lib.amd_matmul_select_kernel
    assert lib.amd_matmul_select_kernel(AUTO) == 0


def launches_of(be, submit):
    """number of nodes that `submit` records on the compute stream"""
    hip = C.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphGetNodes.argtypes = [C.c_void_p, C.c_void_p, C.POINTER(C.c_size_t)]
    hip.hipGraphDestroy.argtypes = [C.c_void_p]
    be.sync()
    graph, count = C.c_void_p(), C.c_size_t()
    assert hip.hipStreamBeginCapture(be.stream(CS), CAPTURE_RELAXED) == 0
    submit()
    assert hip.hipStreamEndCapture(be.stream(CS), C.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(count)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return count.value


@pytest.mark.parametrize("schedule", [B.AMD_MOE_GROUPED, B.AMD_MOE_PER_EXPERT])
@pytest.mark.parametrize("T,D,E,K,H", [(300, 512, 4, 2, 264), (4100, 256, 4, 2, 1024)])      # too few tiles for the persistent kernels; enough
def test_named_kernel_leaves_the_same_bits(backend, select_kernel, T, D, E, K, H, schedule):
    print("case up-projections T=%d D=%d E=%d K=%d H=%d schedule=%d" % (T, D, E, K, H, schedule), flush=True)
    be, rng = backend, np.random.default_rng(T + D)
    layer = MoeLayer(be, T, D, E, K, H)
    layer.load_weights(*(normal_bf16(rng, s, 0.02) for s in ((E, D), (E, H, D), (E, H, D), (E, D, H))))
    d_X, resid = be.upload(normal_bf16(rng, (T, D))), normal_bf16(rng, (T, D))
    got, nodes = {}, {}
    for kernel in (AUTO, EIGHT, FOUR_384):
        d_out = be.upload(resid)
        assert select_kernel(kernel) == 0
        layer.forward(T, d_X.ptr, d_out.ptr, None, schedule)
        be.sync()
        got[kernel] = (be.read(d_out.ptr, (T, D), np.uint16),) + tuple(layer.read_up_projections(T))
        if schedule == B.AMD_MOE_GROUPED:
            nodes[kernel] = launches_of(be, lambda: layer.forward(T, d_X.ptr, d_out.ptr, None, schedule))
        assert select_kernel(AUTO) == 0
        d_out.free()
    for kernel in (EIGHT, FOUR_384):
        for name, a, b in zip(("out", "x1", "x3"), got[AUTO], got[kernel]):
            assert (a == b).all(), name
    if nodes:
        # one launch under AUTO; w1, w3 and the activation otherwise (a ragged-N launch is one launch under a named kernel and
        # may be two under AUTO: the w2 product behind them)
        assert nodes[EIGHT] == nodes[FOUR_384] and nodes[EIGHT] >= nodes[AUTO] + 1
    layer.free()
    d_X.free()
