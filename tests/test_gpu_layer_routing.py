"""The layer's routing (one op: split router product, selection, counts, permutation) against the op sequence it stands
in for, called through the submit wrappers on the same inputs: every output bit for bit."""
import ctypes as C

import numpy as np
import pytest

from ml_dataflow_amd import MoeLayer, binding as B
from util import normal_bf16

pytestmark = pytest.mark.gpu

BF, CS = B.DATAFLOW_BF16, 1


def outputs(be, L, T, E, K):
    be.sync()
    return {"logits": be.read(L.x_routed, (T, E), np.uint16), "weights": be.read(L.token_expert_weights, (T, K), np.uint32),
            "chosen": be.read(L.chosen_experts, (T, K), np.uint16), "counts": be.read(L.expert_counts, (E + 1,), np.int32),
            "cumsum": be.read(L.expert_counts_cumsum, (E,), np.int32), "expert_mapping": be.read(L.expert_mapping, (T * K,), np.int32),
            "token_mapping": be.read(L.token_mapping, (T, K), np.int32),
            "host_counts": np.ctypeslib.as_array(C.cast(L.host_expert_counts, C.POINTER(C.c_int32)), (E,)).copy()}


@pytest.mark.parametrize("T,E,K,D,bias", [
    (1, 8, 2, 64, False), (16, 64, 8, 4096, False), (31, 5, 3, 512, True), (128, 64, 8, 1024, False), (129, 64, 8, 1024, True),
    (256, 8, 2, 512, False), (257, 8, 2, 512, False), (255, 17, 4, 64, True), (1000, 7, 1, 2048, False), (3001, 32, 4, 2048, True),
    (500, 130, 6, 1032, False), (333, 512, 9, 576, False), (96, 40, 32, 512, False), (2000, 64, 17, 64, True), (8192, 64, 8, 512, False),
    (300, 600, 4, 64, False)])
def test_routing_equals_the_op_sequence(backend, T, E, K, D, bias):
    print("case routing T=%d E=%d K=%d D=%d bias=%s" % (T, E, K, D, bias), flush=True)
    be = backend
    rng = np.random.default_rng(T + E + K + D)
    X, Wr = normal_bf16(rng, (T, D)), normal_bf16(rng, (E, D), 0.02)
    layer = MoeLayer(be, T, D, E, K, 256)             # a workspace with room for both: the product splits the same way
    L = layer.L
    d_X, d_out = be.upload(X), be.alloc(T * D * 2)
    d_bias = be.upload(normal_bf16(rng, (T, E))) if bias else None
    be.zero(L.slab, L.slab_bytes, CS)
    be.sync(CS)
    be.write(L.w_router, Wr)
    layer.forward(T, d_X.ptr, d_out.ptr, d_bias.ptr if bias else None, B.AMD_MOE_FUSED)
    got = outputs(be, L, T, E, K)
    be.zero(L.x_routed, T * E * 2, CS)
    be.zero(L.expert_counts, (E + 1) * 4, CS)
    be.zero(L.expert_counts_cumsum, E * 4, CS)
    be.zero(L.expert_mapping, T * K * 4, CS)
    be.zero(L.token_mapping, T * K * 4, CS)
    lib, hp, bptr = be.lib, be.hp, d_bias.ptr if bias else None
    assert lib.dataflow_submit_matmul(hp, CS, BF, BF, BF if bias else B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 1, 0, E, D, T, 1.0, 1.0 if bias else 0.0,
                                      L.w_router, d_X.ptr, bptr, L.x_routed, L.kernel_workspace_bytes, L.kernel_workspace) == 0
    assert lib.dataflow_submit_default_select_experts(hp, CS, BF, T, E, K, L.x_routed, L.token_expert_weights, L.chosen_experts, L.expert_counts,
                                                      L.expert_counts_cumsum, L.host_expert_counts) == 0
    assert lib.dataflow_submit_default_build_expert_mapping(hp, CS, T, E, K, L.chosen_experts, L.expert_counts_cumsum, L.expert_mapping,
                                                            L.token_mapping) == 0
    want = outputs(be, L, T, E, K)
    for name in want:
        assert (got[name] == want[name]).all(), name
    assert got["counts"][:E].sum() == T * K
    layer.free()
