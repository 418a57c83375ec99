"""AdamW step of the layer's weights: the oracle pinned against the fp64 closed form, the HIP kernel against the
oracle through the C ABI.  Values: one bf16 rounding of the result plus the fp32 rounding of its terms (the moment update can cancel; powf, sqrtf,
the divisions and fused multiply-adds differ by an fp32 rounding between libm / the host compiler and the device)."""
import ctypes as C
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

import oracle_lib as O
from util import f32_to_bf16, bf16_to_f64, normal_bf16, bf16_ulp_diff

HP = dict(lr=1e-3, beta1=0.9, beta2=0.999, weight_decay=0.01, epsilon=1e-8)


def near(got_bits, want, scale, rel=2.0 ** -8):
    """one bf16 rounding of the result (2^-8 relative) plus fp32 rounding of the terms it is made of: the moment update
    beta * m + (1 - beta) * g can cancel, and then the fp32 rounding of its terms is what is left"""
    got, want = bf16_to_f64(got_bits), np.asarray(want, dtype=np.float64)
    assert (np.abs(got - want) <= rel * np.abs(want) + 4e-7 * scale).all()


def make(rng, n):
    param, grad, mean = normal_bf16(rng, (n,), 0.05), normal_bf16(rng, (n,), 0.01), normal_bf16(rng, (n,), 0.005)
    var = f32_to_bf16((rng.random(n).astype(np.float32) * 1e-4))
    return param, grad, mean, var


def closed_form(param, grad, mean, var, step, lr, beta1, beta2, weight_decay, epsilon):
    p, g, m, v = (bf16_to_f64(a) for a in (param, grad, mean, var))
    b1, b2 = np.float64(np.float32(beta1)), np.float64(np.float32(beta2))
    lr, wd, eps = (np.float64(np.float32(x)) for x in (lr, weight_decay, epsilon))
    m_t = b1 * m + (1 - b1) * g
    v_t = b2 * v + (1 - b2) * g * g
    m_hat, v_hat = m_t / (1 - b1 ** step), v_t / (1 - b2 ** step)
    return p - lr * (m_hat / (np.sqrt(v_hat) + eps) + wd * p), m_t, v_t


@pytest.mark.parametrize("n,step", [(1, 1), (1000, 1), (4099, 7), (65536, 1000)])
def test_oracle_is_the_closed_form(oracle, n, step):
    rng = np.random.default_rng(n + step)
    param, grad, mean, var = make(rng, n)
    want = closed_form(param, grad, mean, var, step, **HP)
    p, m, v = param.copy(), mean.copy(), var.copy()
    oracle.oracle_adamw_step(n, step, HP["lr"], HP["beta1"], HP["beta2"], HP["weight_decay"], HP["epsilon"], O.ptr(p), O.ptr(grad), O.ptr(m), O.ptr(v))
    scales = (np.abs(bf16_to_f64(param)).max(), max(np.abs(bf16_to_f64(mean)).max(), np.abs(bf16_to_f64(grad)).max()), np.abs(bf16_to_f64(var)).max())
    for got, w, sc in zip((p, m, v), want, scales):
        near(got, w, sc)


def test_oracle_fixed_points(oracle):
    n = 64
    zero = np.zeros(n, np.uint16)
    param = f32_to_bf16(np.linspace(-1, 1, n).astype(np.float32))
    p, m, v = param.copy(), zero.copy(), zero.copy()
    # zero gradient and zero moments: only the decoupled weight decay acts, the moments stay zero
    oracle.oracle_adamw_step(n, 3, 0.5, 0.9, 0.999, 0.25, 1e-8, O.ptr(p), O.ptr(zero), O.ptr(m), O.ptr(v))
    assert (m == 0).all() and (v == 0).all()
    np.testing.assert_allclose(bf16_to_f64(p), bf16_to_f64(param) * (1 - 0.5 * 0.25), rtol=2.0 ** -8)
    # first step from zero moments with no decay: the update is -lr * sign(g) (bias correction cancels beta)
    g = f32_to_bf16(np.where(np.arange(n) % 2, 0.01, -0.02).astype(np.float32))
    p, m, v = param.copy(), zero.copy(), zero.copy()
    oracle.oracle_adamw_step(n, 1, 0.125, 0.9, 0.999, 0.0, 1e-12, O.ptr(p), O.ptr(g), O.ptr(m), O.ptr(v))
    np.testing.assert_allclose(bf16_to_f64(p), bf16_to_f64(param) - 0.125 * np.sign(bf16_to_f64(g)), atol=2.0 ** -8)


@pytest.mark.gpu
@pytest.mark.parametrize("n,step,offset", [(8, 1, 0), (2048, 1, 0), (100003, 5, 0), (1 << 22, 300, 0), (5000, 2, 1)])
def test_gpu_matches_oracle(backend, oracle, n, step, offset):
    """offset 1: arrays that start 2 bytes off a 16-byte boundary take the element-wise path"""
    from ml_dataflow_amd import binding as B
    print("case adamw n=%d step=%d offset=%d" % (n, step, offset), flush=True)
    be = backend
    rng = np.random.default_rng(n)
    param, grad, mean, var = make(rng, n + offset)
    bufs = [be.upload(a) for a in (param, grad, mean, var)]
    ptrs = [b.ptr + 2 * offset for b in bufs]
    BF = B.DATAFLOW_BF16
    assert be.lib.dataflow_submit_default_adamw_step(be.hp, 1, BF, BF, BF, BF, n, step, HP["lr"], HP["beta1"], HP["beta2"], HP["weight_decay"],
                                                     HP["epsilon"], *ptrs) == 0
    be.sync(1)
    p, g, m, v = param[offset:].copy(), grad[offset:].copy(), mean[offset:].copy(), var[offset:].copy()
    oracle.oracle_adamw_step(n, step, HP["lr"], HP["beta1"], HP["beta2"], HP["weight_decay"], HP["epsilon"], O.ptr(p), O.ptr(g), O.ptr(m), O.ptr(v))
    got = [be.read(q, (n,), np.uint16) for q in (ptrs[0], ptrs[2], ptrs[3])]
    scales = (np.abs(bf16_to_f64(param)).max(), max(np.abs(bf16_to_f64(mean)).max(), np.abs(bf16_to_f64(grad)).max()), np.abs(bf16_to_f64(var)).max())
    for g_, w_, sc in zip(got, (p, m, v), scales):
        near(g_, bf16_to_f64(w_), sc, rel=2.0 ** -7)          # two rounded results: one bf16 step apart at most
        assert np.percentile(bf16_ulp_diff(g_, w_), 99.9) <= 1
    assert (be.read(ptrs[1], (n,), np.uint16) == grad[offset:]).all()           # the gradient is read only
    if offset:
        assert be.read(bufs[0].ptr, (1,), np.uint16)[0] == param[0]             # nothing written in front of the arrays
    # step numbers below 1 are rejected
    assert be.lib.dataflow_submit_default_adamw_step(be.hp, 1, BF, BF, BF, BF, n, 0, 1e-3, 0.9, 0.999, 0.0, 1e-8, *ptrs) == -1


@pytest.mark.gpu
def test_gpu_matches_oracle_beyond_the_caches(backend, oracle):
    """four arrays that the 256 MiB memory-side cache does not hold together, with a tail that is no whole vector"""
    test_gpu_matches_oracle(backend, oracle, (1 << 25) + 13, 3, 0)


def test_kernel_issues_its_loads_together_and_non_temporally(tmp_path):
    """The two things the kernel's speed rests on are the compiler's to undo, so they are read from the assembly of the
    kernel's own source: a lane's first four vector loads are in flight together, and every vector access carries nt."""
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ml_dataflow_amd", "csrc")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    flags = re.search(r"^HIPFLAGS = (.*)$", open(os.path.join(csrc, "Makefile")).read(), flags=re.M).group(1)
    flags = flags.replace("$(ARCH)", "gfx950").replace("$(INC)", "").split()
    source, asm = tmp_path / "adamw.hip", tmp_path / "adamw.s"
    source.write_text('#include "moe_common.h"\n#include "optimizer.hip"\n')
    subprocess.run([hipcc, *flags, "-I", os.path.join(csrc, "kernels"), "-S", "--cuda-device-only", "-o", str(asm), str(source)], check=True, capture_output=True)
    body = re.search(r"^default_adamw_step_bf16_bf16_bf16_bf16_kernel:(.*?)s_endpgm", asm.read_text(), flags=re.M | re.S).group(1)
    lines = [line.strip() for line in body.splitlines()]
    vector = [line for line in lines if re.match(r"global_(load|store)_dwordx4\b", line)]
    assert vector and all(re.search(r"\bnt\b", line) for line in vector), vector
    loads = [i for i, line in enumerate(lines) if line.startswith("global_load_dwordx4")]
    assert len(loads) >= 4
    assert not [line for line in lines[loads[0]:loads[3]] if line.startswith("s_waitcnt") and "vmcnt" in line]


@pytest.mark.gpu
def test_gpu_strides_beyond_the_lanes_of_a_launch(backend, oracle):
    """the kernel itself on a grid of fewer lanes than vectors, as a launch of more than 2^32 vectors would have: 3 groups
    for 8 groups' worth and a tail"""
    from ml_dataflow_amd import binding as B
    print("case adamw strided", flush=True)
    be, n, step = backend, 8 * 2048 + 13, 4
    param, grad, mean, var = make(np.random.default_rng(7), n)
    bufs = [be.upload(a) for a in (param, grad, mean, var)]
    hip = C.CDLL("libamdhip64.so")
    module, kernel = C.c_void_p(), C.c_void_p()
    assert hip.hipModuleLoad(C.byref(module), os.path.join(B.LIB_DIR, "hip_kernels_gfx950.hsaco").encode()) == 0
    assert hip.hipModuleGetFunction(C.byref(kernel), module, b"default_adamw_step_bf16_bf16_bf16_bf16_kernel") == 0
    args = [C.c_uint64(n), C.c_int(step)] + [C.c_float(HP[k]) for k in ("lr", "beta1", "beta2", "weight_decay", "epsilon")] + [C.c_void_p(b.ptr) for b in bufs]
    params = (C.c_void_p * len(args))(*[C.cast(C.byref(a), C.c_void_p) for a in args])
    assert hip.hipModuleLaunchKernel(kernel, 3, 1, 1, 256, 1, 1, 0, C.c_void_p(be.stream(1)), params, None) == 0
    be.sync(1)
    p, m, v = param.copy(), mean.copy(), var.copy()
    oracle.oracle_adamw_step(n, step, HP["lr"], HP["beta1"], HP["beta2"], HP["weight_decay"], HP["epsilon"], O.ptr(p), O.ptr(grad), O.ptr(m), O.ptr(v))
    scales = (np.abs(bf16_to_f64(param)).max(), max(np.abs(bf16_to_f64(mean)).max(), np.abs(bf16_to_f64(grad)).max()), np.abs(bf16_to_f64(var)).max())
    for buf, want, sc in zip((bufs[0], bufs[2], bufs[3]), (p, m, v), scales):
        near(be.read(buf.ptr, (n,), np.uint16), bf16_to_f64(want), sc, rel=2.0 ** -7)
    assert hip.hipModuleUnload(module) == 0
    for buf in bufs:
        buf.free()
