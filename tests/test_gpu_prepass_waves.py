"""K quantized one block to a wave (1024 blocks or more, 2048 without V tiles; not
beside FP8 V tiles at head dim 128) against one to a work-group.

The same heads quantized sixteen at a time stay below that, so both
roles run on the same data; every output is equal bit for bit.  Lengths leave
one to four blocks to the last work-group and 1 to 64 rows to the last block;
blocks of zeros and scales outside the fast division's range are among them.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("N,smooth,pv,layout,pad", [(193, True, "fp16", "HND", 0), (257, True, "fp8", "NHD", 0),
                                                    (384, False, "fp8", "HND", 0), (447, True, "fp16", "HND", 24),
                                                    (449, True, None, "HND", 0), (512, True, "bf16", "NHD", 8)])
def test_wave_blocks_equal_work_group_blocks(N, smooth, pv, layout, pad, dtype, D, hip_impl, gpu_device):
    print(f"[k waves] N{N} D{D} {dtype} smooth={smooth} {pv} {layout} pad {pad}", flush=True)
    B = Hkv = 16
    g = torch.Generator().manual_seed(N)
    k = torch.randn(B, Hkv, N, D + pad, generator=g) + 2.0 * torch.randn(B, Hkv, 1, D + pad, generator=g)
    if not smooth:
        k[1, 2, 64:128] = 0  # scale 0
    k[3, 4] = 0
    if dtype == "bf16":
        k[5, 6] *= 2.0 ** -110  # scales below 2^-100: the general division
    k = k.to(DT[dtype]).to(gpu_device)
    v = torch.randn(k.shape, generator=g).to(DT[dtype]).to(gpu_device)
    k, v = (t[..., :D] for t in (k, v))
    q = torch.zeros(B, Hkv, 16, D, dtype=DT[dtype], device=gpu_device)
    if layout == "NHD":
        q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    kw = dict(smooth_k=smooth, pv_dtype=pv, quant_q=False, tensor_layout=layout)
    got = hip_impl.prepass(q, k, v, **kw)
    keys = ["k8", "k_scale"] + ["km"] * smooth + ["v_scale"] * (pv == "fp8")
    for b in range(B):
        want = hip_impl.prepass(q[b:b + 1], k[b:b + 1], v[b:b + 1], **kw)
        torch.cuda.synchronize()
        for key in keys:
            assert torch.equal(got[key][b:b + 1], want[key]), (b, key)
