"""Which ops the layer driver submits, on the CPU: a handle whose functions only note what they are given."""
import ctypes as C

import pytest

from ml_dataflow_amd import binding as B

T, D, E, K, H = 40, 64, 8, 2, 128
ROUTED_BY_OPS = ["default_matmul", "default_select_experts_BF16", "default_build_expert_mapping"]
HASH = C.CFUNCTYPE(C.c_uint64, C.POINTER(C.c_uint8), C.c_uint64)


class NotingHandle:
    """A Dataflow_Handle that notes the nicknames of the ops submitted to it and runs nothing; its op table is the library's."""

    def __init__(self, value_bytes=8):
        self.lib = B.load_library()
        self.h = B.DataflowHandle()
        self.names = []
        fields = dict(B.DataflowHandle._fields_)

        def note(handle, op, stream):
            self.names.append(op.contents.op_skeleton.header.op_nickname.decode())
            return 0

        self.kept = {"submit_op": fields["submit_op"](note), "set_mem": fields["set_mem"](lambda *a: 0), "get_num_procs": fields["get_num_procs"](lambda h: 256),
                     "get_stream_state": fields["get_stream_state"](lambda *a: 256), "submit_dependency": fields["submit_dependency"](lambda *a: 0),
                     "sync_stream": fields["sync_stream"](lambda *a: 0)}
        for name, fn in self.kept.items():
            setattr(self.h, name, fn)
        self.hash = HASH(lambda key, size: key[31] % size)
        assert self.lib.dataflow_init_table(C.byref(self.h.op_table), C.cast(self.hash, C.c_void_p), 32, value_bytes, 64, 256, 0.75, 0.1) == 0

    def forward(self, schedule, **changes):
        """the ops of one forward; no pointer of the layer is followed but that of the counts on the host"""
        layer = B.AmdMoeLayer(max_tokens=T, model_dim=D, num_experts=E, top_k=K, expert_dim=H, dt=B.DATAFLOW_BF16, expert_stride_bytes=3 * H * D * 2)
        for i, (name, kind) in enumerate(B.AmdMoeLayer._fields_):
            if kind is C.c_void_p:
                setattr(layer, name, (i + 1) << 24)
        layer.w3, layer.dw3 = layer.w1 + H * D * 2, layer.dw1 + H * D * 2
        layer.kernel_workspace_bytes = 1 << 23
        counts = (C.c_int * E)(*[T * K // E] * E)
        layer.host_expert_counts = C.addressof(counts)
        for name, value in changes.items():
            setattr(layer, name, value)
        self.names.clear()
        assert self.lib.amd_moe_layer_forward(C.pointer(self.h), 1, 2, C.byref(layer), T, 1 << 32, None, 2 << 32, schedule) == 0
        return list(self.names)


@pytest.mark.parametrize("schedule", [B.AMD_MOE_PER_EXPERT, B.AMD_MOE_GROUPED, B.AMD_MOE_FUSED])
def test_a_handle_without_the_routing_op_is_routed_op_by_op(schedule):
    names = NotingHandle().forward(schedule)
    assert names[:3] == ROUTED_BY_OPS
    assert not [name for name in names if name.startswith("amd_route_tokens")]
