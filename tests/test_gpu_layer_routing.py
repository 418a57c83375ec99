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


def compare(be, L, layer, T, E, K, D, d_X, d_out, d_bias):
    """a forward, then the same routing op by op; returns what both left"""
    layer.forward(T, d_X.ptr, d_out.ptr, d_bias.ptr if d_bias else None, B.AMD_MOE_FUSED)
    got = outputs(be, L, T, E, K)
    be.zero(L.x_routed, T * E * 2, CS)
    be.zero(L.expert_counts, (E + 1) * 4, CS)
    be.zero(L.expert_counts_cumsum, E * 4, CS)
    be.zero(L.expert_mapping, T * K * 4, CS)
    be.zero(L.token_mapping, T * K * 4, CS)
    lib, hp, bptr = be.lib, be.hp, d_bias.ptr if d_bias else None
    assert lib.dataflow_submit_matmul(hp, CS, BF, BF, BF if d_bias else B.DATAFLOW_NONE, BF, B.DATAFLOW_FP32, 1, 0, E, D, T, 1.0, 1.0 if d_bias else 0.0,
                                      L.w_router, d_X.ptr, bptr, L.x_routed, L.kernel_workspace_bytes, L.kernel_workspace) == 0
    assert lib.dataflow_submit_default_select_experts(hp, CS, BF, T, E, K, L.x_routed, L.token_expert_weights, L.chosen_experts, L.expert_counts,
                                                      L.expert_counts_cumsum, L.host_expert_counts) == 0
    assert lib.dataflow_submit_default_build_expert_mapping(hp, CS, T, E, K, L.chosen_experts, L.expert_counts_cumsum, L.expert_mapping,
                                                            L.token_mapping) == 0
    want = outputs(be, L, T, E, K)
    for name in want:
        assert (got[name] == want[name]).all(), name
    return got


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
    got = compare(be, L, layer, T, E, K, D, d_X, d_out, d_bias)
    assert got["counts"][:E].sum() == T * K
    layer.free()


@pytest.mark.parametrize("T,E,K,D,room", [(512, 64, 8, 4096, -4), (512, 64, 8, 4096, 0), (512, 64, 8, 4096, 1020), (512, 64, 8, 4096, 1024),
                                          (100, 20, 4, 2048, 0), (3001, 32, 4, 2048, 100), (256, 8, 2, 1024, 0)])
def test_routing_splits_the_product_as_the_matmul_does(backend, T, E, K, D, room):
    """a workspace of the partial sums' size plus `room` bytes: without it the product runs unsplit, in another order of its
    sums; the counts that the routing keeps there too (1024 bytes for 512 tokens and 64 experts) do not take it from them"""
    print("case routing workspace T=%d E=%d K=%d D=%d room=%d" % (T, E, K, D, room), flush=True)
    be = backend
    k_tiles, cus = (D + 63) // 64, be.device_info.cu_count
    splits = cus // (((T + 127) // 128) * ((E + 127) // 128))
    per = max(4, (-(-k_tiles // splits) + 3) & ~3)
    splits = -(-k_tiles // per)
    assert splits > 1
    rng = np.random.default_rng(T + E + K + D)
    X, Wr = normal_bf16(rng, (T, D)), normal_bf16(rng, (E, D), 0.02)
    layer = MoeLayer(be, T, D, E, K, 256)
    L = layer.L
    assert L.kernel_workspace_bytes >= splits * T * E * 4 + room
    L.kernel_workspace_bytes = splits * T * E * 4 + room            # what the ops are told: the layer's own is larger
    d_X, d_out = be.upload(X), be.alloc(T * D * 2)
    be.zero(L.slab, L.slab_bytes, CS)
    be.sync(CS)
    be.write(L.w_router, Wr)
    got = compare(be, L, layer, T, E, K, D, d_X, d_out, None)
    assert got["counts"][:E].sum() == T * K
    layer.free()


NEG_INF, INF, NAN = 0xFF80, 0x7F80, 0x7FC0


@pytest.mark.parametrize("T,E,K,D,offset", [(40, 8, 2, 64, 0), (100, 20, 4, 512, 1), (33, 7, 3, 512, 0), (256, 64, 4, 1024, 1), (300, 64, 8, 1024, 0),
                                            (700, 13, 5, 2048, 1), (1000, 32, 4, 64, 1), (290, 512, 9, 576, 0), (64, 40, 32, 512, 0)])
def test_routing_of_masked_infinite_and_nan_logits(backend, T, E, K, D, offset):
    """experts masked with a bias of -inf, down to rows with fewer than K experts left (slots without an expert) and with none;
    NaN and +inf logits; offset 1: a bias that starts 2 bytes off every larger alignment"""
    print("case routing special T=%d E=%d K=%d D=%d offset=%d" % (T, E, K, D, offset), flush=True)
    be = backend
    rng = np.random.default_rng(T + E + K + D)
    X, Wr = normal_bf16(rng, (T, D)), normal_bf16(rng, (E, D), 0.02)
    bias = normal_bf16(rng, (T, E))
    bias[rng.random((T, E)) < 0.3] = NEG_INF
    bias[0] = NEG_INF                                     # no expert left
    bias[1, :], bias[1, E // 2] = NEG_INF, 0              # one
    bias[2, :], bias[2, E - K:] = NEG_INF, 0              # just enough
    bias[3, 1] = NAN
    bias[4, :] = NAN
    bias[5, E - 1] = INF
    bias[6, 0], bias[6, 2] = INF, NAN
    bias[T - 1, :K - 1], bias[T - 1, K - 1:] = 0, NEG_INF  # one too few, in the last token
    layer = MoeLayer(be, T, D, E, K, 256)
    L = layer.L
    d_X, d_out = be.upload(X), be.alloc(T * D * 2)
    d_bias = be.upload(np.concatenate([np.zeros(offset, np.uint16), bias.ravel()]))
    d_bias.ptr += 2 * offset
    be.zero(L.slab, L.slab_bytes, CS)                     # the mappings of slots without an expert are left as they are: in range
    be.sync(CS)
    be.write(L.w_router, Wr)
    got = compare(be, L, layer, T, E, K, D, d_X, d_out, d_bias)
    d_bias.ptr -= 2 * offset
    assert (got["chosen"][0] == 0xFFFF).all() and sorted(got["chosen"][1])[0] == E // 2 and (got["chosen"][4] == 0xFFFF).all()
    assert sorted(got["chosen"][2]) == list(range(E - K, E))
    assert (got["chosen"][T - 1] == 0xFFFF).sum() == 1 and (got["chosen"][5] == E - 1).any() and (got["chosen"][6] == 0).any()
    valid = got["chosen"] < E
    assert (got["counts"][:E] == np.bincount(got["chosen"][valid], minlength=E)).all()
    assert (np.sort(got["token_mapping"][valid]) == np.arange(valid.sum())).all()
    layer.free()


def test_routing_writes_logits_at_any_element(backend):
    """x_routed 2 bytes off an 8-byte boundary, rows of whole quads: element by element, nothing in front or behind touched"""
    print("case routing unaligned logits", flush=True)
    be, (T, E, K, D) = backend, (31, 20, 4, 512)
    rng = np.random.default_rng(3)
    X, Wr = normal_bf16(rng, (T, D)), normal_bf16(rng, (E, D), 0.02)
    layer = MoeLayer(be, T, D, E, K, 256)
    L = layer.L
    d_X, d_out = be.upload(X), be.alloc(T * D * 2)
    d_logits = be.upload(np.full(T * E + 8, 0x1234, np.uint16))
    be.zero(L.slab, L.slab_bytes, CS)
    be.sync(CS)
    be.write(L.w_router, Wr)
    L.x_routed = d_logits.ptr + 2
    compare(be, L, layer, T, E, K, D, d_X, d_out, None)
    around = be.read(d_logits.ptr, (T * E + 8,), np.uint16)
    assert around[0] == 0x1234 and (around[T * E + 1:] == 0x1234).all()
    layer.free()


@pytest.mark.parametrize("T,E,K", [(64, 16, 1), (65, 16, 1), (127, 16, 2), (128, 16, 2), (129, 16, 2), (68, 38, 4), (32, 52, 2), (255, 32, 2), (256, 32, 2),
                                   (256, 33, 2), (256, 64, 2), (256, 100, 1)])
def test_few_tokens_at_the_edges_of_the_waves_that_add_up(backend, T, E, K):
    """256, 512 and 2048 quads of sums, where the single work-group gets more waves than its selection needs"""
    print("case routing waves T=%d E=%d K=%d" % (T, E, K), flush=True)
    be, D = backend, 512
    rng = np.random.default_rng(T + E + K)
    layer = MoeLayer(be, T, D, E, K, 256)
    L = layer.L
    X, Wr = normal_bf16(rng, (T, D)), normal_bf16(rng, (E, D), 0.02)
    d_X, d_out = be.upload(X), be.alloc(T * D * 2)
    be.write(L.w_router, Wr)
    be.zero(L.w1, E * L.expert_stride_bytes)
    compare(be, L, layer, T, E, K, D, d_X, d_out, None)
    layer.free()
    d_X.free(), d_out.free()
