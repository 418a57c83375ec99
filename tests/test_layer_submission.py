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

    def layer(self, **changes):
        """no pointer of it is followed but that of the counts on the host"""
        layer = B.AmdMoeLayer(max_tokens=T, model_dim=D, num_experts=E, top_k=K, expert_dim=H, dt=B.DATAFLOW_BF16, expert_stride_bytes=3 * H * D * 2)
        for i, (name, kind) in enumerate(B.AmdMoeLayer._fields_):
            if kind is C.c_void_p:
                setattr(layer, name, (i + 1) << 24)
        layer.w3, layer.dw3 = layer.w1 + H * D * 2, layer.dw1 + H * D * 2
        layer.kernel_workspace_bytes = 1 << 23
        self.counts = (C.c_int * E)(*[T * K // E] * E)
        layer.host_expert_counts = C.addressof(self.counts)
        for name, value in changes.items():
            setattr(layer, name, value)
        return layer

    def forward(self, schedule, **changes):
        """the ops of one forward"""
        layer = self.layer(**changes)
        self.names.clear()
        assert self.lib.amd_moe_layer_forward(C.pointer(self.h), 1, 2, C.byref(layer), T, 1 << 32, None, 2 << 32, schedule) == 0
        return list(self.names)


@pytest.mark.parametrize("schedule", [B.AMD_MOE_PER_EXPERT, B.AMD_MOE_GROUPED, B.AMD_MOE_FUSED])
def test_a_handle_without_the_routing_op_is_routed_op_by_op(schedule):
    names = NotingHandle().forward(schedule)
    assert names[:3] == ROUTED_BY_OPS
    assert not [name for name in names if name.startswith("amd_route_tokens")]


class HipFunction(C.Structure):
    """include/dataflow_amd.h: Hip_Function"""
    _fields_ = [("config", C.c_int * 2), ("is_native", C.c_bool), ("function_handle", C.c_void_p), ("set_launch_config", C.c_void_p),
                ("hip_external_func", C.c_void_p), ("op_extra", C.c_void_p), ("op_skeleton", B.OpSkeleton), ("stands_in_for", C.c_void_p * 3)]


def skeleton_of(lib, name):
    """the skeletons of the three ops that routing consists of, and of the op that stands in for them"""
    sk = B.OpSkeleton()
    if name == "matmul":
        lib.dataflow_set_matmul_skeleton(C.byref(sk))
    elif name == "select_experts":
        lib.dataflow_set_default_select_experts_skeleton(C.byref(sk), B.DATAFLOW_BF16)
    elif name == "build_expert_mapping":
        lib.dataflow_set_default_build_expert_mapping_skeleton(C.byref(sk))
    else:
        sk.header.op_nickname = b"amd_route_tokens_BF16"
        sk.header.num_args = 17
        tags = [B.DATAFLOW_INT_SCALAR] * 4 + [B.DATAFLOW_BF16] * 4 + [B.DATAFLOW_FP32, B.DATAFLOW_UINT16] + [B.DATAFLOW_INT] * 5 + [B.DATAFLOW_UINT64_SCALAR, B.DATAFLOW_VOID]
        sk.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*tags)
        assert lib.dataflow_do_fingerprinting(C.byref(sk.header), C.sizeof(sk.header), sk.fingerprint) == 0
    return sk


ROUTING_OPS = ("matmul", "select_experts", "build_expert_mapping")


class RegisteredHandle(NotingHandle):
    """with a table as registration leaves it: the three ops, and the one that stands in for them"""

    def __init__(self):
        super().__init__(C.sizeof(HipFunction))
        for i, name in enumerate(ROUTING_OPS):
            self.insert_op(name, 0x1000 * (i + 1))
        self.insert("route", hip_external_func=0x4000, stands_in_for=(C.c_void_p * 3)(0x1000, 0x2000, 0x3000))

    def insert(self, name, **fields):
        sk = skeleton_of(self.lib, name)
        fn = HipFunction(op_skeleton=sk, **fields)
        assert self.lib.dataflow_insert_table(C.byref(self.h.op_table), C.cast(sk.fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0

    def insert_op(self, name, implementation):
        self.insert(name, is_native=name != "matmul", **{"hip_external_func" if name == "matmul" else "function_handle": implementation})


@pytest.mark.parametrize("replaced", [None, *ROUTING_OPS])
def test_the_routing_op_gives_way_to_a_replaced_one(replaced):
    """a table as registration leaves it, then another implementation under one of the three skeletons"""
    noting = RegisteredHandle()
    lib, table = noting.lib, C.byref(noting.h.op_table)
    if replaced:
        assert lib.dataflow_remove_table(table, C.cast(skeleton_of(lib, replaced).fingerprint, C.c_void_p), None) == 0
        noting.insert_op(replaced, 0x5000)
    for schedule in (B.AMD_MOE_PER_EXPERT, B.AMD_MOE_GROUPED, B.AMD_MOE_FUSED):
        names = noting.forward(schedule)
        if replaced:
            assert names[:3] == ROUTED_BY_OPS
        else:
            assert names[0] == "amd_route_tokens_BF16" and not set(ROUTED_BY_OPS[1:]) & set(names)


@pytest.mark.parametrize("changes", [{"kernel_workspace": (9 << 24) + 8}, {"kernel_workspace_bytes": 256}, {"num_experts": 520}])
def test_the_routing_op_gives_way_where_its_limits_do_not_hold(changes):
    """a workspace off a 16-byte boundary, one too small for the counts, more experts than it takes: all of which the ops take"""
    names = RegisteredHandle().forward(B.AMD_MOE_FUSED, **changes)
    assert names[:3] == ROUTED_BY_OPS


@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("schedule", [B.AMD_MOE_GROUPED, B.AMD_MOE_FUSED])
def test_the_benchmark_times_the_ops_the_layer_submits(schedule, first):
    """bench.py's kernel table comes from a replay of the step op by op: the same ops in the same order as the layer's own"""
    import bench
    noting = RegisteredHandle()
    lib, hp, layer = noting.lib, C.pointer(noting.h), noting.layer()
    flag = B.AMD_MOE_FIRST_MICRO_BATCH if first else 0
    assert lib.amd_moe_layer_forward(hp, 1, 2, C.byref(layer), T, 1 << 32, None, 2 << 32, schedule) == 0
    assert lib.amd_moe_layer_backward(hp, 1, 2, C.byref(layer), T, 1 << 32, 3 << 32, 4 << 32, schedule | flag) == 0
    submitted = list(noting.names)
    noting.names.clear()

    class Stub:
        def __init__(self, **fields):
            self.__dict__.update(fields)

    be = Stub(lib=lib, h=noting.h, hp=hp, zero=lambda *a: None, sync=lambda *a: None)
    ev = Stub(new=lambda: None, record=lambda *a: None, elapsed_ms=lambda *a: 0.0)
    buffers = [Stub(ptr=n << 32) for n in (1, 2, 3, 4)]
    rows = bench.replay_step_with_events(be, Stub(L=layer, T=T, D=D, E=E, K=K, H=H), T, *buffers, None, True, ev, None, schedule == B.AMD_MOE_FUSED, first)
    assert noting.names == submitted
    work = bench.algorithmic_work(T, D, E, K, H, schedule == B.AMD_MOE_FUSED)
    assert len(rows) == len(submitted) and all(name in work for name, _ in rows)


GATHERING_OPS = ("amd_grouped_matmul_gathered", "amd_grouped_matmul", "default_prepare_experts_BF16_BF16")
ALIGNED_X = 1 << 32
AUTO, EIGHT_WAVES, FOUR_WAVES, FOUR_WAVES_384 = 0, 8, 4, 384          # include/amd_matmul.h


class AskingHandle(NotingHandle):
    """with the library's answer about gathered rows in the table, and under the three ops it speaks for what it was registered beside"""

    def __init__(self, matmul):
        super().__init__(C.sizeof(HipFunction))
        lib, self.skeletons = self.lib, {}
        setters = (lib.dataflow_set_amd_grouped_matmul_gathered_skeleton, lib.dataflow_set_amd_grouped_matmul_skeleton,
                   lambda sk: lib.dataflow_set_default_prepare_experts_skeleton(sk, B.DATAFLOW_BF16, B.DATAFLOW_BF16))
        for i, (name, setter) in enumerate(zip(GATHERING_OPS, setters)):
            self.skeletons[name] = B.OpSkeleton()
            setter(C.byref(self.skeletons[name]))
            self.insert(name, 0x1000 * (i + 1))
        answer = self.skeletons["answer"] = B.OpSkeleton()
        answer.header.op_nickname = b"amd_gathers_k_rows_BF16"
        answer.header.num_args = 10
        answer.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*([B.DATAFLOW_INT_SCALAR] * 4 + [B.DATAFLOW_BF16, B.DATAFLOW_INT_SCALAR] + [B.DATAFLOW_BF16] * 3 + [B.DATAFLOW_UINT64_SCALAR]))
        assert lib.dataflow_do_fingerprinting(C.byref(answer.header), C.sizeof(answer.header), answer.fingerprint) == 0
        self.insert("answer", C.cast(matmul.amd_gathers_k_rows, C.c_void_p).value, stands_in_for=(C.c_void_p * 3)(0x1000, 0x2000, 0x3000))

    def insert(self, name, implementation, **fields):
        native = "prepare" in name
        fn = HipFunction(op_skeleton=self.skeletons[name], is_native=native, **{"function_handle" if native else "hip_external_func": implementation}, **fields)
        assert self.lib.dataflow_insert_table(C.byref(self.h.op_table), C.cast(self.skeletons[name].fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0

    def replace(self, name):
        assert self.lib.dataflow_remove_table(C.byref(self.h.op_table), C.cast(self.skeletons[name].fingerprint, C.c_void_p), None) == 0
        self.insert(name, 0x5000)

    def gathers(self, layer, tokens, first, X=ALIGNED_X):
        return self.lib.amd_moe_layer_backward_gathers(C.pointer(self.h), C.byref(layer), tokens, X, first)


@pytest.fixture
def matmul():
    import os
    B.load_library()
    lib = C.CDLL(os.path.join(B.LIB_DIR, "libamd_matmul.so"))
    yield lib
    assert lib.amd_matmul_select_kernel(AUTO) == 0


def stacked_layer(dim, experts, top_k, hidden):
    up = 2 * dim * hidden
    return B.AmdMoeLayer(model_dim=dim, num_experts=experts, top_k=top_k, expert_dim=hidden, dx1=2 << 32, w1=3 << 32, w3=(3 << 32) + up, dw1=4 << 32, dw3=(4 << 32) + up,
                         expert_stride_bytes=3 * up)


@pytest.mark.parametrize("tokens,first,gathers", [(0, False, False), (2047, False, False), (2048, False, True), (2559, True, False), (2560, True, True)])
def test_the_backward_gathers_where_experts_have_the_rows(matmul, tokens, first, gathers):
    """dim 1280, 8 experts, top 2: the lines are 512 and 640 rows an expert; not with wide experts, narrow rows, w3 apart from w1, an X off a 16-byte boundary, one of
    4 GiB or an environment that forbids it"""
    handle, layer = AskingHandle(matmul), stacked_layer(1280, 8, 2, 1536)
    assert handle.gathers(layer, tokens, first) == gathers
    assert handle.gathers(layer, tokens, first, ALIGNED_X + 8) == 0
    apart = stacked_layer(1280, 8, 2, 1536)
    apart.w3 += 256
    for other in (stacked_layer(1272, 8, 2, 1536), stacked_layer(1280, 8, 2, 1544), apart):
        assert handle.gathers(other, tokens, first) == 0
    assert handle.gathers(layer, (1 << 32) // 2 // 1280 + 1, first) == 0


def test_the_backward_gathers_only_where_the_sliced_kernel_runs(matmul):
    """over drawn layers, with every kernel a program can name: the answer is that of the launch's own plan, within the layer's two lines"""
    import random
    rng, handle, told = random.Random(1), AskingHandle(matmul), {}
    for _ in range(4000):
        dim, hidden, experts, top_k = 64 * rng.randint(8, 64), 64 * rng.randint(8, 32), rng.randint(1, 64), rng.randint(1, 8)
        tokens, first = int(2 ** rng.uniform(8, 16)), rng.random() < 0.5
        if rng.random() < 0.3:                                          # about a round of tiles: where the lines of one and of more rounds meet
            experts = max(1, min(64, 256 // (-(-dim // 256) * -(-2 * hidden // 256)) + rng.randint(-1, 1)))
        if top_k > experts or tokens * dim * 2 > 0xFFFFFFFF:
            continue
        for kernel in (AUTO, EIGHT_WAVES, FOUR_WAVES, FOUR_WAVES_384):
            assert matmul.amd_matmul_select_kernel(kernel) == 0
            sliced = matmul.amd_matmul_planned_sliced(dim, tokens * top_k, 2 * hidden, experts, int(not first), 256)
            answer = handle.gathers(stacked_layer(dim, experts, top_k, hidden), tokens, first)
            assert answer == (sliced and dim >= 1280 and hidden <= 1536), (kernel, tokens, dim, experts, top_k, hidden, first)
            told[kernel] = told.get(kernel, 0) + answer
    assert told[AUTO] > 500 and told[FOUR_WAVES_384] > 500 and told[EIGHT_WAVES] == told[FOUR_WAVES] == 0


@pytest.mark.parametrize("replaced", [None, *GATHERING_OPS])
def test_the_gathered_gradient_gives_way_to_a_replaced_op(matmul, replaced):
    """the rows go through a copy where a program has put its own op in the place of one of the three, and where the table has no answer"""
    handle, layer = AskingHandle(matmul), stacked_layer(4096, 64, 8, 1024)
    if replaced:
        handle.replace(replaced)
    assert handle.gathers(layer, 8192, False) == (replaced is None)
    bare = NotingHandle(C.sizeof(HipFunction))
    assert bare.lib.amd_moe_layer_backward_gathers(C.pointer(bare.h), C.byref(layer), 8192, ALIGNED_X, False) == 0


@pytest.mark.parametrize("tokens,dim,streams", [(1024, 4096, {1}), (1025, 4096, {1, 2}), (2048, 2048, {1}), (2049, 1024, {1, 2})])
def test_small_grouped_passes_stay_on_one_stream(tokens, dim, streams):
    """the lines: 2^36 multiplies of the stacked up-projection, 2048 tokens; a layer whose w3 lies apart from w1 has a pair of matmuls in its forward"""
    noting, used, met = NotingHandle(), [], []
    fields = dict(B.DataflowHandle._fields_)
    on = fields["submit_op"](lambda handle, op, stream: used.append(stream) or 0)
    meet = fields["submit_dependency"](lambda *a: met.append(a[1]) or 0)
    noting.h.submit_op, noting.h.submit_dependency = on, meet
    layer = noting.layer(max_tokens=tokens, model_dim=dim, expert_dim=1024, num_experts=64, top_k=8, expert_stride_bytes=6 * dim * 1024)
    assert noting.lib.amd_moe_layer_forward(C.pointer(noting.h), 1, 2, C.byref(layer), tokens, 1 << 32, None, 2 << 32, B.AMD_MOE_GROUPED) == 0
    assert set(used) == streams and set(met) == (streams if len(streams) > 1 else set())
    used.clear()
    met.clear()
    assert noting.lib.amd_moe_layer_backward(C.pointer(noting.h), 1, 2, C.byref(layer), tokens, 1 << 32, 2 << 32, 3 << 32, B.AMD_MOE_GROUPED) == 0
    assert set(used) == streams and len(met) == (4 if len(streams) > 1 else 0)


def test_small_grouped_passes_refuse_a_secondary_stream_that_is_none():
    """they submit nothing to it, but an id the handle does not have stays an error, as in a large pass"""
    noting = NotingHandle()
    noting.h.num_streams = 3
    refuse = dict(B.DataflowHandle._fields_)["submit_dependency"](lambda handle, stream, state: 0 if 0 <= stream < 3 else -1)
    noting.h.submit_dependency = refuse
    for tokens in (16, 4096):
        layer = noting.layer(max_tokens=tokens, model_dim=4096, expert_dim=1024, num_experts=64, top_k=8, expert_stride_bytes=6 * 4096 * 1024)
        for secondary, answer in ((2, 0), (3, -1), (-1, -1)):
            args = (C.pointer(noting.h), 1, secondary, C.byref(layer), tokens, 1 << 32)
            assert noting.lib.amd_moe_layer_forward(*args, None, 2 << 32, B.AMD_MOE_GROUPED) == answer
            assert noting.lib.amd_moe_layer_backward(*args, 2 << 32, 3 << 32, B.AMD_MOE_GROUPED) == answer


UP_OPS = ["amd_grouped_matmul_gathered", "amd_swiglu_strided_BF16"]


@pytest.mark.parametrize("replaced", [None, *UP_OPS])
def test_the_up_projection_op_gives_way_to_a_replaced_one(replaced):
    """the fused schedule submits gather, GEMM and activation as one op where the table is as registration leaves it and the layer
    is small; as two where one of them has another implementation, or a limit of the op does not hold"""
    noting = NotingHandle(C.sizeof(HipFunction))
    lib, skeletons = noting.lib, {}
    for name, setter in zip(UP_OPS, (lib.dataflow_set_amd_grouped_matmul_gathered_skeleton, lambda sk: lib.dataflow_set_amd_swiglu_strided_skeleton(sk, B.DATAFLOW_BF16))):
        skeletons[name] = B.OpSkeleton()
        setter(C.byref(skeletons[name]))
    both = skeletons["amd_up_swiglu_BF16"] = B.OpSkeleton()
    both.header.op_nickname = b"amd_up_swiglu_BF16"
    both.header.num_args = 12
    both.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*([B.DATAFLOW_INT_SCALAR] * 4 + [B.DATAFLOW_INT, B.DATAFLOW_BF16, B.DATAFLOW_UINT64_SCALAR, B.DATAFLOW_BF16, B.DATAFLOW_INT,
                                                                                       B.DATAFLOW_INT_SCALAR, B.DATAFLOW_BF16, B.DATAFLOW_BF16]))
    assert lib.dataflow_do_fingerprinting(C.byref(both.header), C.sizeof(both.header), both.fingerprint) == 0

    def insert(name, implementation, **fields):
        fn = HipFunction(op_skeleton=skeletons[name], is_native="swiglu_strided" in name, **{"function_handle" if "swiglu_strided" in name else "hip_external_func": implementation}, **fields)
        assert lib.dataflow_insert_table(C.byref(noting.h.op_table), C.cast(skeletons[name].fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0

    def up(**changes):
        return [name for name in noting.forward(B.AMD_MOE_FUSED, **changes) if name in skeletons]

    for i, name in enumerate(UP_OPS):
        insert(name, 0x1000 * (i + 1))
    assert up() == UP_OPS
    insert("amd_up_swiglu_BF16", 0x4000, stands_in_for=(C.c_void_p * 3)(0x1000, 0x2000, None))
    if replaced:
        assert lib.dataflow_remove_table(C.byref(noting.h.op_table), C.cast(skeletons[replaced].fingerprint, C.c_void_p), None) == 0
        insert(replaced, 0x5000)
    assert up() == (UP_OPS if replaced else ["amd_up_swiglu_BF16"])
    assert up(x1=(7 << 24) + 8) == UP_OPS and up(kernel_workspace=(9 << 24) + 8) == UP_OPS     # off a 16-byte boundary
    large = 1 << 18                                                                            # T K 2 H = 42 M values
    assert up(expert_dim=large, w3=(2 << 24) + large * D * 2, w1=2 << 24, dw1=3 << 24, dw3=(3 << 24) + large * D * 2) == UP_OPS


UP_APART = {B.AMD_MOE_GROUPED: ("amd_up_swiglu_grouped_BF16", ("amd_grouped_matmul", "default_swiglu_BF16", "default_prepare_experts_BF16_BF16")),
            B.AMD_MOE_PER_EXPERT: ("amd_up_swiglu_expert_BF16", ("default_matmul", "default_swiglu_BF16"))}


@pytest.mark.parametrize("schedule,replaced", [(s, r) for s, (_, ops) in UP_APART.items() for r in (None, *ops)])
def test_the_up_projection_ops_with_results_apart_give_way_to_a_replaced_one(schedule, replaced):
    """as above for the schedules that keep x1 and x3 in arrays of their own"""
    noting = NotingHandle(C.sizeof(HipFunction))
    lib, skeletons = noting.lib, {}
    one_op, ops = UP_APART[schedule]
    setters = {"amd_grouped_matmul": lib.dataflow_set_amd_grouped_matmul_skeleton, "default_matmul": lib.dataflow_set_matmul_skeleton,
               "default_swiglu_BF16": lambda sk: lib.dataflow_set_default_swiglu_skeleton(sk, B.DATAFLOW_BF16),
               "default_prepare_experts_BF16_BF16": lambda sk: lib.dataflow_set_default_prepare_experts_skeleton(sk, B.DATAFLOW_BF16, B.DATAFLOW_BF16)}
    for name in ops:
        skeletons[name] = B.OpSkeleton()
        setters[name](C.byref(skeletons[name]))
    both = skeletons[one_op] = B.OpSkeleton()
    both.header.op_nickname = one_op.encode()
    both.header.num_args = 13
    both.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*([B.DATAFLOW_INT_SCALAR] * 4 + [B.DATAFLOW_INT, B.DATAFLOW_BF16, B.DATAFLOW_UINT64_SCALAR, B.DATAFLOW_BF16, B.DATAFLOW_INT,
                                                                                       B.DATAFLOW_INT_SCALAR] + [B.DATAFLOW_BF16] * 3))
    assert lib.dataflow_do_fingerprinting(C.byref(both.header), C.sizeof(both.header), both.fingerprint) == 0

    def insert(name, implementation, **fields):
        native = "matmul" not in name and name != one_op
        fn = HipFunction(op_skeleton=skeletons[name], is_native=native, **{"function_handle" if native else "hip_external_func": implementation}, **fields)
        assert lib.dataflow_insert_table(C.byref(noting.h.op_table), C.cast(skeletons[name].fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0

    def swiglus(**changes):
        return [name for name in noting.forward(schedule, **changes) if "swiglu" in name]

    times = E if schedule == B.AMD_MOE_PER_EXPERT else 1
    for i, name in enumerate(ops):
        insert(name, 0x1000 * (i + 1))
    assert swiglus() == ["default_swiglu_BF16"] * times
    table = {name: 0x1000 * (i + 1) for i, name in enumerate(ops)}
    order = [n for n in ("default_swiglu_BF16", "amd_grouped_matmul", "default_matmul", "default_prepare_experts_BF16_BF16") if n in table]
    insert(one_op, 0x7000, stands_in_for=(C.c_void_p * 3)(*[table[n] for n in order]))
    if replaced:
        assert lib.dataflow_remove_table(C.byref(noting.h.op_table), C.cast(skeletons[replaced].fingerprint, C.c_void_p), None) == 0
        insert(replaced, 0x6000)
    assert swiglus() == ([ops[1]] if replaced else [one_op]) * times
    assert swiglus(x1=(7 << 24) + 8) == swiglus(kernel_workspace=(9 << 24) + 8) == swiglus(w3=1 << 40) == [ops[1]] * times     # off a 16-byte boundary; not stacked


@pytest.mark.parametrize("replaced", [False, True])
def test_the_twin_matmul_gives_way_to_a_replaced_matmul(replaced):
    """an expert's dW1 and dW3 of the per-expert schedule: one op where the table is as registration leaves it"""
    noting = NotingHandle(C.sizeof(HipFunction))
    lib, hp, layer = noting.lib, C.pointer(noting.h), noting.layer()
    matmul, twin = B.OpSkeleton(), B.OpSkeleton()
    lib.dataflow_set_matmul_skeleton(C.byref(matmul))
    twin.header.op_nickname = b"amd_matmul_twin_BF16"
    twin.header.num_args = 11
    twin.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*([B.DATAFLOW_INT_SCALAR] * 3 + [B.DATAFLOW_FP32_SCALAR] + [B.DATAFLOW_BF16] * 7))
    assert lib.dataflow_do_fingerprinting(C.byref(twin.header), C.sizeof(twin.header), twin.fingerprint) == 0
    for sk, implementation, stands_in_for in ((matmul, 0x2000 if replaced else 0x1000, ()), (twin, 0x3000, (0x1000,))):
        fn = HipFunction(op_skeleton=sk, hip_external_func=implementation, stands_in_for=(C.c_void_p * 3)(*stands_in_for))
        assert lib.dataflow_insert_table(C.byref(noting.h.op_table), C.cast(sk.fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0
    assert lib.amd_moe_layer_forward(hp, 1, 2, C.byref(layer), T, 1 << 32, None, 2 << 32, B.AMD_MOE_PER_EXPERT) == 0
    noting.names.clear()
    assert lib.amd_moe_layer_backward(hp, 1, 2, C.byref(layer), T, 1 << 32, 3 << 32, 4 << 32, B.AMD_MOE_PER_EXPERT) == 0
    last = noting.names[noting.names.index("default_prepare_experts_BF16_BF16") + 1:]
    assert last == (["default_matmul"] * 2 * E if replaced else ["amd_matmul_twin_BF16"] * E) + ["default_matmul"]


NORM_OPS = ("default_rms_norm_bwd_w_BF16_BF16", "default_rms_norm_bwd_w_combine_BF16")
NORM_FEW_ROWS = "amd_rms_norm_bwd_w_few_rows_BF16_BF16"


@pytest.mark.parametrize("replaced", [None, *NORM_OPS])
def test_the_norms_weight_gradient_over_few_rows_gives_way_to_a_replaced_half(replaced):
    """one op where the table is as registration leaves it and the rows are few; two where they are not, where a half of it has
    another implementation, and (refused or not, as before) where the workspace is too small"""
    noting = NotingHandle(C.sizeof(HipFunction))
    lib, hp = noting.lib, C.pointer(noting.h)
    skeletons = {}
    for name, setter in zip(NORM_OPS, (lambda sk: lib.dataflow_set_default_rms_norm_bwd_w_skeleton(sk, B.DATAFLOW_BF16, B.DATAFLOW_BF16),
                                       lambda sk: lib.dataflow_set_default_rms_norm_bwd_w_combine_skeleton(sk, B.DATAFLOW_BF16))):
        skeletons[name] = B.OpSkeleton()
        setter(C.byref(skeletons[name]))
    few = skeletons[NORM_FEW_ROWS] = B.OpSkeleton()
    few.header.op_nickname = NORM_FEW_ROWS.encode()
    few.header.num_args = 8
    few.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*([B.DATAFLOW_INT_SCALAR] * 2 + [B.DATAFLOW_FP32] + [B.DATAFLOW_BF16] * 3 + [B.DATAFLOW_INT_SCALAR, B.DATAFLOW_INT]))
    assert lib.dataflow_do_fingerprinting(C.byref(few.header), C.sizeof(few.header), few.fingerprint) == 0

    def submit(rows, workspace_bytes=1 << 20):
        noting.names.clear()
        assert lib.dataflow_submit_default_rms_norm_bwd_w(hp, 1, B.DATAFLOW_BF16, B.DATAFLOW_BF16, rows, 64, 1e-5, 1 << 24, 2 << 24, 3 << 24, 4 << 24,
                                                          workspace_bytes, 5 << 24) == 0
        return tuple(noting.names)

    def insert(name, implementation, **fields):
        fn = HipFunction(op_skeleton=skeletons[name], is_native=True, function_handle=implementation, **fields)
        assert lib.dataflow_insert_table(C.byref(noting.h.op_table), C.cast(skeletons[name].fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0

    for i, name in enumerate(NORM_OPS):
        insert(name, 0x1000 * (i + 1))
    assert submit(16) == NORM_OPS                                   # ops registered one by one
    insert(NORM_FEW_ROWS, 0x4000, stands_in_for=(C.c_void_p * 3)(0x1000, 0x2000, None))
    if replaced:
        assert lib.dataflow_remove_table(C.byref(noting.h.op_table), C.cast(skeletons[replaced].fingerprint, C.c_void_p), None) == 0
        insert(replaced, 0x5000)
    expected = NORM_OPS if replaced else (NORM_FEW_ROWS,)
    assert submit(1) == expected and submit(1536) == expected
    assert submit(1537) == NORM_OPS and submit(0) == NORM_OPS and submit(16, 300) == NORM_OPS


NORM_FORMS = {"amd_rms_norm_wave_rows_BF16": [B.DATAFLOW_INT_SCALAR] * 2 + [B.DATAFLOW_FP32_SCALAR] + [B.DATAFLOW_BF16] * 3 + [B.DATAFLOW_FP32],
              "amd_rms_norm_bwd_x_wave_rows_BF16_BF16": [B.DATAFLOW_INT_SCALAR] * 2 + [B.DATAFLOW_FP32] + [B.DATAFLOW_BF16] * 5}
NORM_FORMS["amd_rms_norm_long_rows_BF16"] = NORM_FORMS["amd_rms_norm_wave_rows_BF16"]


@pytest.mark.parametrize("replaced", [False, True])
def test_the_norms_forms_by_rows_and_columns_and_only_beside_what_they_stand_in_for(replaced):
    """a row on a wave from 8192 rows of up to 1024 columns on, long rows from 2500 of over 4608 columns on (forward), the op itself elsewhere, in another
    type, and everywhere where the table has another implementation under it or none of the forms"""
    noting = NotingHandle(C.sizeof(HipFunction))
    lib, hp, forward, bwd_x = noting.lib, C.pointer(noting.h), B.OpSkeleton(), B.OpSkeleton()
    lib.dataflow_set_default_rms_norm_skeleton(C.byref(forward), B.DATAFLOW_BF16)
    lib.dataflow_set_default_rms_norm_bwd_x_skeleton(C.byref(bwd_x), B.DATAFLOW_BF16, B.DATAFLOW_BF16)

    def insert(skeleton, implementation, stands_in_for=None):
        fn = HipFunction(op_skeleton=skeleton, is_native=True, function_handle=implementation, stands_in_for=(C.c_void_p * 3)(stands_in_for, None, None))
        assert lib.dataflow_insert_table(C.byref(noting.h.op_table), C.cast(skeleton.fingerprint, C.c_void_p), C.cast(C.byref(fn), C.c_void_p)) == 0

    def submitted(rows, cols, dt=B.DATAFLOW_BF16):
        noting.names.clear()
        assert lib.dataflow_submit_default_rms_norm(hp, 1, dt, rows, cols, 1e-5, 1 << 24, 2 << 24, 3 << 24, 4 << 24) == 0
        assert lib.dataflow_submit_default_rms_norm_bwd_x(hp, 1, dt, dt, rows, cols, 1e-5, 4 << 24, 1 << 24, 2 << 24, 3 << 24, 5 << 24, None) == 0
        return tuple(noting.names)

    plain = ("default_rms_norm_BF16", "default_rms_norm_bwd_x_BF16_BF16")
    insert(forward, 0x1000)
    insert(bwd_x, 0x2000)
    assert submitted(8192, 1024) == submitted(2500, 4616) == plain
    for name, tags in NORM_FORMS.items():
        form = B.OpSkeleton()
        form.header.op_nickname, form.header.num_args = name.encode(), len(tags)
        form.header.arg_dtypes = (C.c_int * B.MAX_OP_ARGS)(*tags)
        assert lib.dataflow_do_fingerprinting(C.byref(form.header), C.sizeof(form.header), form.fingerprint) == 0
        insert(form, 0x3000, 0x2000 if "bwd_x" in name else 0x1000)
    if replaced:
        for skeleton in (forward, bwd_x):
            assert lib.dataflow_remove_table(C.byref(noting.h.op_table), C.cast(skeleton.fingerprint, C.c_void_p), None) == 0
            insert(skeleton, 0x5000)
    waves = plain if replaced else ("amd_rms_norm_wave_rows_BF16", "amd_rms_norm_bwd_x_wave_rows_BF16_BF16")
    long_rows = plain if replaced else ("amd_rms_norm_long_rows_BF16", plain[1])
    assert submitted(8192, 1024) == submitted(8192, 8) == submitted(1 << 20, 1024) == waves
    assert submitted(2500, 4616) == submitted(65536, 16384) == long_rows
    for rows, cols in ((8191, 1024), (8192, 1032), (0, 64), (1, 8), (2499, 4616), (2500, 4608), (8192, 4096)):
        assert submitted(rows, cols) == plain
    assert submitted(8192, 512, B.DATAFLOW_FP16)[0] == "default_rms_norm_FP16"


@pytest.mark.gpu
def test_gpu_replaced_select_experts_is_the_one_that_runs():
    """registration notes the real implementations; the op sequence takes over when one of them is exchanged for the same
    kernel out of a second load of the code object, with the same results"""
    import os

    import numpy as np

    from ml_dataflow_amd import Backend, MoeLayer
    from util import normal_bf16
    print("case replaced select_experts", flush=True)
    be = Backend(0)
    rng = np.random.default_rng(5)
    layer = MoeLayer(be, T, D, E, K, H)
    layer.load_weights(*(normal_bf16(rng, s, 0.02) for s in ((E, D), (E, H, D), (E, H, D), (E, D, H))))
    X, resid = normal_bf16(rng, (T, D)), normal_bf16(rng, (T, D))
    d_X = be.upload(X)
    names, kind = [], dict(B.DataflowHandle._fields_)["submit_op"]
    submit = kind(C.cast(be.h.submit_op, C.c_void_p).value)          # a pointer of its own, not the handle's field

    def note(handle, op, stream):
        names.append(op.contents.op_skeleton.header.op_nickname.decode())
        return submit(handle, op, stream)

    noting = kind(note)
    be.h.submit_op = noting

    def forward():
        names.clear()
        d_out = be.upload(resid)
        layer.forward(T, d_X.ptr, d_out.ptr, None, B.AMD_MOE_GROUPED)
        be.sync()
        return be.read(d_out.ptr, (T, D), np.uint16)

    first = forward()
    assert names[0] == "amd_route_tokens_BF16" and "default_select_experts_BF16" not in names
    hip = C.CDLL("libamdhip64.so")
    module, kernel = C.c_void_p(), C.c_void_p()
    assert hip.hipModuleLoad(C.byref(module), os.path.join(B.LIB_DIR, "hip_kernels_gfx950.hsaco").encode()) == 0
    assert hip.hipModuleGetFunction(C.byref(kernel), module, b"default_select_experts_bf16_kernel") == 0
    key = C.cast(skeleton_of(be.lib, "select_experts").fingerprint, C.c_void_p)
    entry = HipFunction()
    assert be.lib.dataflow_remove_table(C.byref(be.h.op_table), key, C.cast(C.byref(entry), C.c_void_p)) == 0
    assert entry.is_native and entry.function_handle != kernel.value
    entry.function_handle = kernel.value
    assert be.lib.dataflow_insert_table(C.byref(be.h.op_table), key, C.cast(C.byref(entry), C.c_void_p)) == 0
    second = forward()
    assert names[:3] == ROUTED_BY_OPS
    assert (first == second).all()
    be.h.submit_op = submit
    layer.free()
    be.close()
    assert hip.hipModuleUnload(module) == 0
