"""The optional outputs of sage_run in a caller's own layouts.

q is a slice of packed Q, K, V rows and q8 a buffer of its own, at shapes where
Q is quantized in the attention's prologue, in the pre-pass, and where the keys
are split or heads share a work-group: Q8 is the pre-pass's bit for bit in the
layout the options name (q's strides with fuse_q 1, q8_strides otherwise), and
not a byte beside its rows is written.  A call whose outputs are all the
caller's and that needs no other buffer runs without a workspace.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from test_run_routes import Q8_SHAPES

pytestmark = pytest.mark.gpu
CANARY = 77


def _strided_q8(shape, strides, dev):
    """An int8 buffer of canaries and the [B, H, N, D] view of it."""
    n = sum((a - 1) * b for a, b in zip(shape, strides)) + 1
    buf = torch.full((n + 256,), CANARY, dtype=torch.int8, device=dev)
    return buf, buf.as_strided(shape, strides)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape", Q8_SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_q8_layouts(shape, D, hip_impl, gpu_device):
    B, Hq, Hkv, Nq, Nkv = shape
    g = torch.Generator().manual_seed(Nq + Nkv)
    packed = torch.randn(B, Nq, 3, Hq, D, generator=g).to(torch.bfloat16).to(gpu_device)
    q = packed[:, :, 0].transpose(1, 2)  # rows 3 * Hq * D apart
    k, v = (torch.randn(B, Hkv, Nkv, D, generator=g).to(torch.bfloat16).to(gpu_device) for _ in range(2))
    lib = hip_impl._load()
    mul = float(np.float32(D ** -0.5 * hip_impl.LOG2E_REF))
    want = hip_impl.prepass(q, k, v)
    want_o = hip_impl.run(q, k, v)
    for fuse_q in (-1, 0, 1):
        print(f"[q8 layout] {shape} D{D} fuse_q {fuse_q}", flush=True)
        strides = q.stride() if fuse_q == 1 else (Hq * Nq * (D + 16) + 64, Nq * (D + 16), D + 16, 1)
        buf, q8 = _strided_q8(q.shape, strides, gpu_device)
        o = torch.empty(q.shape, dtype=q.dtype, device=gpu_device)
        qs = torch.empty((B, Hq, -(-Nq // 128)), dtype=torch.float32, device=gpu_device)
        hip_impl.whole_call(lib.sage_run, lib.sage_run_workspace_bytes, "sage_run", q, k, v, o, "HND",
                            (B, Hq, Hkv, Nq, Nkv, D), mul, False, 0, 128, 1, fuse_q, [q8, qs, None, None, None, None])
        torch.cuda.synchronize()
        assert torch.equal(q8, want["q8"]) and torch.equal(qs, want["q_scale"])
        assert torch.equal(o, want_o)
        q8.fill_(CANARY)
        assert (buf == CANARY).all()


@pytest.mark.parametrize("fuse_q", [None, True, False])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(4, 32, 32, 640, 128), (1, 2, 2, 256, 64), (16, 48, 12, 193, 64)],
                         ids=lambda s: "-".join(map(str, s)))
def test_intermediates_without_smoothing(shape, dtype, fuse_q, hip_impl, gpu_device):
    print(f"[no smoothing] {shape} {dtype} fuse_q {fuse_q}", flush=True)
    B, Hq, Hkv, N, D = shape
    dt = torch.float16 if dtype == "fp16" else torch.bfloat16
    g = torch.Generator().manual_seed(N)
    q, k, v = (torch.randn(B, h, N, D, generator=g).to(dt).to(gpu_device) for h in (Hq, Hkv, Hkv))
    o, pre = hip_impl.run(q, k, v, pv_dtype=dtype, smooth_k=False, fuse_q=fuse_q, return_intermediates=True)
    want = hip_impl.prepass(q, k, v, smooth_k=False)
    torch.cuda.synchronize()
    assert sorted(pre) == ["k8", "k_scale", "q8", "q_scale"]
    for key in pre:
        assert torch.equal(pre[key], want[key]), key
    assert torch.equal(o, hip_impl.run(q, k, v, pv_dtype=dtype, smooth_k=False))
    assert torch.equal(o, hip_impl.attention(q, k, v, want, pv_dtype=dtype))


# (B, Hq, Hkv, Nq, Nkv, D), dtype, pv, whether the pre-pass of the call has Q and V tiles
STAGES = [((1, 32, 32, 1100, 1100, 128), "bf16", "fp16", False, True),
          ((2, 24, 24, 900, 900, 64), "fp16", "fp16", False, False),
          ((1, 2, 2, 256, 256, 64), "bf16", "fp8", True, True),
          ((2, 8, 2, 32, 3000, 128), "bf16", "bf16", True, False)]


@pytest.mark.parametrize("case", STAGES, ids=lambda c: "-".join(map(str, c[0])))
def test_prepass_stage_is_runs(case, hip_impl, gpu_device):
    """The timed stage makes what run's own pre-pass makes, no more and no less."""
    (B, Hq, Hkv, Nq, Nkv, D), dtype, pv, has_q, has_vt = case
    dt = torch.float16 if dtype == "fp16" else torch.bfloat16
    g = torch.Generator().manual_seed(Nkv)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(dt).to(gpu_device) for h, n in ((Hq, Nq), (Hkv, Nkv), (Hkv, Nkv)))
    pre = hip_impl.prepass_stage(q, k, v, pv_dtype=pv)
    _, want = hip_impl.run(q, k, v, pv_dtype=pv, return_intermediates=True, fuse_q=False)
    torch.cuda.synchronize()
    assert ("q8" in pre, "vt" in pre) == (has_q, has_vt)
    for key in set(pre) & set(want):
        assert torch.equal(pre[key], want[key]), key
