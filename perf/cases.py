"""Performance cases of the mixture-of-experts layer and the ops around it, on one GPU.

Each case is one pass of something a training or serving program has this library do, through the entry points such a
program calls: MoeLayer.forward / .backward and the submit wrappers, with caller-owned tensors in device memory and the
layer's weights laid out once.  Sizes are the benchmark's configurations and others of the same ranges.

  kind "layer"   a MoE layer: forward only (inference), or forward + backward (a training step)
  kind "norm"    the RMS norm in front of the layer and its backward passes
  kind "adamw"   the optimizer step over the expert weights of a layer
  kind "dense"   a dense projection of the transformer block (attention q / k / v / o) through the plain matmul: forward,
                 gradient of the input, accumulated gradient of the weight: the three operand layouts in use
"""
import math

import numpy as np
import torch

from ml_dataflow_amd import Backend, MoeLayer, binding as B
from ml_dataflow_amd.synthetic import SKEWED_ROUTING_BIAS_SCALE, zipf_bias

COMPUTE = 1                         # stream ids, as the drivers use them
BF, F32, NONE = B.DATAFLOW_BF16, B.DATAFLOW_FP32, B.DATAFLOW_NONE
SCHEDULES = {"per_expert": B.AMD_MOE_PER_EXPERT, "grouped": B.AMD_MOE_GROUPED, "fused": B.AMD_MOE_FUSED}
LARGEST_ROUTED_WORK = 65536 * 8 * 4096 * 1024      # tokens * top_k * model dim * expert dim of the largest listed case


def _layer(name, tokens, dim, experts, top_k, hidden, train, schedule="fused", skewed=False, first=False):
    case = {"kind": "layer", "tokens": tokens, "dim": dim, "experts": experts, "top_k": top_k, "hidden": hidden, "train": train,
            "schedule": schedule, "skewed": skewed, "first": first}
    return dict(case, name=name) if name else case


def listed():
    return [
        # a unit-test sized layer: nothing but launches and their latency
        _layer("fwd_256x512", 256, 512, 8, 2, 1024, False),
        # one generation step of a small batch: every token meets other experts, the weights are the traffic
        _layer("fwd_16x4096", 16, 4096, 64, 8, 1024, False),
        # prompt processing, or the forward of an evaluation run
        _layer("fwd_8192x2048", 8192, 2048, 32, 4, 1408, False),
        # the same with a router that prefers few experts: the largest takes almost eight times the mean
        _layer("fwd_8192x2048_skewed", 8192, 2048, 32, 4, 1408, False, skewed=True),
        # a training step on the benchmark's default configuration, weight gradients accumulated
        _layer("step_8192x4096", 8192, 4096, 64, 8, 1024, True),
        # the long-context training step
        _layer("step_65536x4096", 65536, 4096, 64, 8, 1024, True),
        # a ragged micro-batch that opens an accumulation: weight gradients written, not added to
        _layer("step_3001x2048_first", 3001, 2048, 32, 4, 1408, True, first=True),
        # the layer's default schedule, which keeps the reference's sequence of operations
        _layer("step_4096x2048_grouped", 4096, 2048, 32, 4, 1408, True, schedule="grouped"),
        # the reference's own schedule: the host waits for the routing and submits every expert by itself
        _layer("step_2048x2048_per_expert", 2048, 2048, 16, 2, 1408, True, schedule="per_expert"),
        # the norm around the layer of the default configuration
        {"name": "norm_8192x4096", "kind": "norm", "tokens": 8192, "dim": 4096},
        # the optimizer over the expert weights of the 32-expert configuration
        {"name": "adamw_277m", "kind": "adamw", "elements": 3 * 32 * 2048 * 1408, "step": 10},
        # the q / o projection of a block with the default configuration's model dim
        {"name": "dense_8192x4096x4096", "kind": "dense", "tokens": 8192, "dim_in": 4096, "dim_out": 4096},
    ]


def _spread(rng, lo, hi):
    """a whole number from lo to hi, spread over its logarithm"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "step", "step", "step", "norm", "adamw", "dense"])
    if kind == "norm":
        return {"kind": "norm", "tokens": _spread(rng, 16, 32768), "dim": 64 * rng.randint(8, 128)}
    if kind == "adamw":
        return {"kind": "adamw", "elements": _spread(rng, 4096, 3 * 64 * 4096 * 1024), "step": rng.randint(1, 1000)}
    if kind == "dense":
        return {"kind": "dense", "tokens": _spread(rng, 64, 32768), "dim_in": 64 * rng.randint(8, 64), "dim_out": 64 * rng.randint(8, 64)}
    dim, hidden, experts = 64 * rng.randint(8, 64), 64 * rng.randint(8, 32), rng.randint(8, 64)
    while experts * dim * hidden > 64 * 4096 * 1024:
        experts -= 1
    top_k = rng.randint(1, min(8, experts))
    most = min(65536, LARGEST_ROUTED_WORK // (top_k * dim * hidden))
    if kind == "forward":
        return _layer(None, _spread(rng, 1, most), dim, experts, top_k, hidden, False, skewed=rng.random() < 0.25)
    schedule = rng.choice(["fused", "fused", "fused", "grouped", "per_expert"])
    if schedule != "fused":
        most = min(16384, most)
    return _layer(None, _spread(rng, 256, most), dim, experts, top_k, hidden, True, schedule, rng.random() < 0.25, rng.random() < 0.5)


# ---------------------------------------------------------------- what a program has in hand

_handle = None


def _backend():
    """the process's handle on the GPU: opened once and kept, with its registered ops and streams"""
    global _handle
    if _handle is None:
        _handle = Backend(0)
    return _handle


class _OwnedLayer(MoeLayer):
    """a layer whose memory is given back with the last reference to it or to a tensor over one of its buffers"""

    def __del__(self):
        self.free()


class _Buffer:
    """one of a layer's buffers, described for torch.as_tensor; the tensor keeps this object and with it the layer"""

    def __init__(self, layer, ptr, shape, typestr):
        self.layer = layer
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False), "version": 2}


def _view(layer, ptr, shape, dtype):
    typestr = {torch.bfloat16: "<i2", torch.int16: "<i2", torch.float32: "<f4"}[dtype]
    return torch.as_tensor(_Buffer(layer, ptr, shape, typestr), device="cuda:0").view(dtype)


def _normal(gen, shape, std=1.0):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda:0").normal_(0.0, std, generator=gen)


class _LayerState:
    """a layer with its weights, the batch's tensors and views of what the passes leave in the layer's own buffers"""

    def __init__(self, case, seed):
        gen = torch.Generator(device="cuda:0").manual_seed(seed)
        T, D, E, K, H = (case[k] for k in ("tokens", "dim", "experts", "top_k", "hidden"))
        self.layer = layer = _OwnedLayer(_backend(), T, D, E, K, H)
        L = layer.L
        self.tokens, self.train, self.schedule, self.first = T, case["train"], SCHEDULES[case["schedule"]], case["first"]
        _view(layer, L.w_router, (E, D), torch.bfloat16).normal_(0.0, 0.02, generator=gen)
        _view(layer, L.w1, (E, L.expert_stride_bytes // 2), torch.bfloat16).normal_(0.0, 0.02, generator=gen)
        self.x, self.out = _normal(gen, (T, D)), _normal(gen, (T, D))         # normalised input; residual stream, updated in place
        self.dy = _normal(gen, (T, D)) if self.train else None
        self.dx = torch.empty_like(self.x) if self.train else None
        self.bias = None
        if case["skewed"]:
            row = torch.from_numpy(zipf_bias(np.random.default_rng(seed), E, SKEWED_ROUTING_BIAS_SCALE))
            self.bias = row.to("cuda:0", torch.bfloat16).expand(T, E).contiguous()
        self.results = {"out": self.out, "experts": _view(layer, L.chosen_experts, (T, K), torch.int16),
                        "weights": _view(layer, L.token_expert_weights, (T, K), torch.float32)}
        if self.train:
            self.results.update(dx=self.dx, dw_router=_view(layer, L.dw_router, (E, D), torch.bfloat16),
                                dw_experts=_view(layer, L.dw1, (E, L.expert_stride_bytes // 2), torch.bfloat16))

    def run(self):
        self.layer.forward(self.tokens, self.x.data_ptr(), self.out.data_ptr(), self.bias.data_ptr() if self.bias is not None else None, self.schedule)
        if self.train:
            self.layer.backward(self.tokens, self.x.data_ptr(), self.dy.data_ptr(), self.dx.data_ptr(), self.schedule, first_micro_batch=self.first)
        return self.results


class _NormState:
    def __init__(self, case, seed):
        gen = torch.Generator(device="cuda:0").manual_seed(seed)
        self.T, self.D = T, D = case["tokens"], case["dim"]
        self.be = _backend()
        self.x, self.dy = _normal(gen, (T, D)), _normal(gen, (T, D))
        self.scale = _normal(gen, (D,), 0.1).add_(1.0)
        self.normed, self.recomputed = torch.empty_like(self.x), torch.empty_like(self.x)
        self.rms = torch.empty(T, dtype=torch.float32, device="cuda:0")
        self.dx = _normal(gen, (T, D))                       # gradient that arrives over the residual stream, added to
        self.dscale = torch.zeros(D, dtype=torch.bfloat16, device="cuda:0")
        self.workspace = torch.empty(256 + 512 * D * 4, dtype=torch.uint8, device="cuda:0")

    def run(self):
        lib, hp = self.be.lib, self.be.hp
        ok = lib.dataflow_submit_default_rms_norm(hp, COMPUTE, BF, self.T, self.D, 1e-5, self.scale.data_ptr(), self.x.data_ptr(),
                                                  self.normed.data_ptr(), self.rms.data_ptr())
        ok |= lib.dataflow_submit_default_rms_norm_bwd_x(hp, COMPUTE, BF, BF, self.T, self.D, 1e-5, self.rms.data_ptr(), self.scale.data_ptr(),
                                                         self.x.data_ptr(), self.dy.data_ptr(), self.dx.data_ptr(), self.recomputed.data_ptr())
        ok |= lib.dataflow_submit_default_rms_norm_bwd_w(hp, COMPUTE, BF, BF, self.T, self.D, 1e-5, self.rms.data_ptr(), self.x.data_ptr(),
                                                         self.dy.data_ptr(), self.dscale.data_ptr(), self.workspace.numel(), self.workspace.data_ptr())
        if ok != 0:
            raise RuntimeError("a norm op was refused")
        return {"normed": self.normed, "rms": self.rms, "dx": self.dx, "recomputed": self.recomputed, "dscale": self.dscale}


class _AdamwState:
    def __init__(self, case, seed):
        gen = torch.Generator(device="cuda:0").manual_seed(seed)
        self.n, self.step = case["elements"], case["step"]
        self.be = _backend()
        self.param, self.grad = _normal(gen, (self.n,), 0.02), _normal(gen, (self.n,), 1e-3)
        self.mean, self.var = _normal(gen, (self.n,), 3e-4), _normal(gen, (self.n,), 1e-3).square_()

    def run(self):
        if self.be.lib.dataflow_submit_default_adamw_step(self.be.hp, COMPUTE, BF, BF, BF, BF, self.n, self.step, 1e-3, 0.9, 0.999, 0.1, 1e-8,
                                                          self.param.data_ptr(), self.grad.data_ptr(), self.mean.data_ptr(), self.var.data_ptr()) != 0:
            raise RuntimeError("the optimizer step was refused")
        return {"param": self.param, "mean": self.mean, "var": self.var}


class _DenseState:
    def __init__(self, case, seed):
        gen = torch.Generator(device="cuda:0").manual_seed(seed)
        self.T, self.I, self.O = case["tokens"], case["dim_in"], case["dim_out"]
        self.be = _backend()
        self.x, self.dy = _normal(gen, (self.T, self.I)), _normal(gen, (self.T, self.O))
        self.w, self.dw = _normal(gen, (self.O, self.I), 0.02), _normal(gen, (self.O, self.I))
        self.y, self.dx = torch.empty_like(self.dy), torch.empty_like(self.x)
        self.workspace = torch.empty(64 << 20, dtype=torch.uint8, device="cuda:0")

    def matmul(self, trans_a, trans_b, M, K, N, a, b, c, d):
        return self.be.lib.dataflow_submit_matmul(self.be.hp, COMPUTE, BF, BF, BF if c is not None else NONE, BF, F32, trans_a, trans_b, M, K, N,
                                                  1.0, 1.0 if c is not None else 0.0, a.data_ptr(), b.data_ptr(), c.data_ptr() if c is not None else None,
                                                  d.data_ptr(), self.workspace.numel(), self.workspace.data_ptr())

    def run(self):
        T, I, O = self.T, self.I, self.O
        ok = self.matmul(1, 0, O, I, T, self.w, self.x, None, self.y)            # y = x w^T
        ok |= self.matmul(0, 0, I, O, T, self.w, self.dy, None, self.dx)         # dx = dy w
        ok |= self.matmul(0, 1, I, T, O, self.x, self.dy, self.dw, self.dw)      # dw += dy^T x
        if ok != 0:
            raise RuntimeError("a matmul was refused")
        return {"y": self.y, "dx": self.dx, "dw": self.dw}


_STATES = {"layer": _LayerState, "norm": _NormState, "adamw": _AdamwState, "dense": _DenseState}


def prepare(case, seed):
    state = _STATES[case["kind"]](case, seed)
    torch.cuda.synchronize()            # the library's streams do not wait for torch's
    return state


def run(state):
    return state.run()


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: inputs read once, outputs written once (nothing that passes from one kernel of a pass to the next).  A layer
    reads the weights of the experts that its tokens are expected to meet."""
    if case["kind"] == "norm":
        n = case["tokens"] * case["dim"]
        return {"bytes": 2.0 * n * 6 + 4.0 * case["tokens"], "flops": 20.0 * n}      # x, dy, dx read; normed, recomputed, dx written
    if case["kind"] == "adamw":
        return {"bytes": 14.0 * case["elements"], "flops": 16.0 * case["elements"]}
    if case["kind"] == "dense":
        T, I, O = case["tokens"], case["dim_in"], case["dim_out"]
        return {"bytes": 2.0 * (2 * T * I + 2 * T * O + 3 * I * O), "flops": 6.0 * T * I * O}
    T, D, E, K, H = (case[k] for k in ("tokens", "dim", "experts", "top_k", "hidden"))
    met = E * (1.0 - (1.0 - K / E) ** T) if not case["skewed"] else min(E, T * K)
    weights = 3.0 * met * D * H + E * D
    values, flops = 3.0 * T * D + weights, 6.0 * T * K * D * H + 2.0 * T * D * E
    if case["train"]:
        values += 2.0 * T * D + (1.0 if case["first"] else 2.0) * (3.0 * E * D * H + E * D)
        flops *= 3.0
    return {"bytes": 2.0 * values, "flops": flops}


def tolerance(case):
    """bf16 results of fp32 sums.  A router logit next to a bf16 rounding boundary may fall to either side with another order
    of its sum, and at a tie for the last place that gives a token another expert: a few ids, and the rows of those tokens."""
    if case["kind"] == "layer":
        return {"rel": 1e-2, "max": 0.9, "differ": 1e-3}
    return {"rel": 1e-2}
