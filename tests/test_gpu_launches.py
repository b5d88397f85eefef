"""Every launch a whole call chooses, in its own main loop, against float64.

Each entry names the kernel its shape takes (test_run_routes.py holds the C
ABI to that): 8 waves, 4 waves at two or three to a SIMD, Q from the pre-pass
or quantized in the prologue, V in place or in tiles.  Nothing here is split
over the keys, so the mask-free loop runs.  Non-causal sweeps of 64 * nkb keys
have nkb - 4 mask-free iterations, in trips of 4 at D = 64 (3 for the
unquantized kernel at three waves per SIMD; none unrolled for bf16 and FP8 P
there) and of 2 at D = 128 (with two S buffers): the lengths end the trips
without and with every leftover.  With rising scores the loop redoes blocks
whose P leaves the shortcut's bound and rescales O.

Sampled rows of three heads.  INT8 against the exact emulation of the same
codes, the unquantized kernel against attention in float64.  With e_p, e_o the
roundings of P (half an ulp: 2^-11 fp16, 2^-8 bf16, 2^-4 e4m3) and of the output, every
element is within e_p max|v| + (2 e_o + 5 * 2^-11) |o| (the last for the row
sums of fp16 P), and since the roundings of P are independent of V, the
relative 2-norm of all errors is within their rms, e_p / sqrt(3), plus
e_o + 5 * 2^-11.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import sage_oracle as O
from parity_util import sample_rows
from test_gpu_flash_vrow import _flash

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EP = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8, "fp8": 2.0 ** -4}
EO = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 2.0 ** -24}

# (kernel, waves, waves per SIMD), (B, Hq, Hkv, Nq, Nkv, D), causal, dtype, pv
LAUNCHES = []


def _add(kernels, shape, causal, *types):
    for k in kernels:
        for dtype, pv in types:
            LAUNCHES.append((k, shape, causal, dtype, pv))


PRE, PRO = "i8", "i8q"  # Q from the pre-pass, in the prologue
ALL_PV = [("bf16", "fp16"), ("fp16", "bf16"), ("bf16", "fp8")]
IN_PLACE = [("fp16", "fp16"), ("bf16", "bf16")]
# D = 64, two 4-wave work-groups to a CU: trips of 4, 3 .. 9 mask-free iterations
for nkb in (7, 8, 9, 10, 11, 13):
    _add([(PRE, 4, 2)], (3, 24, 8, 300, 64 * nkb, 64), False, ("bf16", "fp16"))
    _add([("flash", 4, 2)], (3, 24, 8, 300, 64 * nkb, 64), False, ("fp16", None))
_add([(PRE, 4, 2), (PRO, 4, 2)], (2, 24, 8, 961, 961, 64), False, *ALL_PV, *IN_PLACE)
_add([(PRE, 4, 2)], (2, 24, 8, 961, 961, 64), True, *ALL_PV, *IN_PLACE)
_add([("flash", 4, 2)], (2, 24, 8, 961, 961, 64), True, ("bf16", None))
# three to a CU
for nkb in (7, 8, 9, 10, 11):
    _add([(PRO, 4, 3)], (8, 48, 8, 130, 64 * nkb, 64), False, ("bf16", "fp16"))
    _add([("flash", 4, 3)], (8, 48, 8, 130, 64 * nkb, 64), False, ("fp16", None), ("bf16", None))
_add([(PRE, 4, 3), (PRO, 4, 3)], (8, 48, 8, 130, 577, 64), False, *ALL_PV, *IN_PLACE)
_add([(PRO, 4, 3)], (8, 48, 8, 577, 577, 64), True, *ALL_PV, *IN_PLACE)
_add([("flash", 4, 3)], (4, 48, 8, 705, 705, 64), True, ("fp16", None), ("bf16", None))
# 8 waves
_add([(PRE, 8, 2), (PRO, 8, 2)], (1, 24, 8, 2500, 20300, 64), False, *ALL_PV[:2], *IN_PLACE)
_add([(PRE, 8, 2), (PRO, 8, 2)], (1, 24, 8, 1333, 20300, 64), False, ALL_PV[2])
_add([("flash", 8, 2)], (1, 24, 8, 1333, 2500, 64), False, ("fp16", None), ("bf16", None))
_add([("flash", 8, 2)], (1, 24, 8, 2500, 2500, 64), True, ("fp16", None), ("bf16", None))
# D = 128
for nkb in (6, 7, 8, 9):
    _add([(PRO, 4, 2)], (3, 24, 8, 300, 64 * nkb, 128), False, ("bf16", "fp16"))
    _add([("flash", 4, 2)], (3, 24, 8, 300, 64 * nkb, 128), False, ("bf16", None))
_add([(PRE, 4, 2), (PRO, 4, 2)], (2, 24, 8, 705, 705, 128), False, *ALL_PV, *IN_PLACE)
_add([(PRE, 4, 2)], (2, 24, 8, 705, 705, 128), True, *ALL_PV, *IN_PLACE)
_add([(PRE, 8, 2), (PRO, 8, 2)], (1, 24, 8, 1333, 1333, 128), False, ("bf16", "fp16"), ("fp16", "fp16"))
_add([(PRO, 8, 2)], (1, 24, 8, 1472, 1472, 128), True, ("fp32", "fp16"), ("fp16", "fp16"))
_add([(PRE, 8, 2), (PRO, 8, 2)], (1, 24, 8, 1333, 7000, 128), False, ("bf16", "fp8"))
_add([("flash", 8, 2)], (1, 24, 8, 1333, 2500, 128), False, ("fp16", None), ("bf16", None))
_add([("flash", 8, 2)], (1, 24, 8, 2500, 2500, 128), True, ("fp16", None), ("bf16", None))


def _inputs(shape, dtype, rising, dev):
    """Normal q, k, v; rising: queries share a direction that the keys drift
    along, 2.5 log2 units per 64 keys (64 in all where the keys are many)."""
    B, Hq, Hkv, Nq, Nkv, D = shape
    g = torch.Generator().manual_seed(Nq + Nkv + D)
    q = torch.randn(B, Hq, Nq, D, generator=g)
    k = torch.randn(B, Hkv, Nkv, D, generator=g)
    v = torch.randn(B, Hkv, Nkv, D, generator=g)
    if rising:
        u = torch.randn(D, generator=g)
        u /= u.norm()
        drift = torch.arange(Nkv, dtype=torch.float32) / 64 * min(2.5, 64 * 64 / Nkv)
        q += 4.0 * u
        k += drift[:, None] * (D ** 0.5 / (4.0 * 1.4426950408889634)) * u
    return [t.to(DT[dtype]).to(dev) for t in (q, k, v)]


def _check(got, want, v, ep, eo):
    err = np.abs(got - want)
    bound = ep * np.abs(v).max() + (2 * eo + 5 * 2.0 ** -11) * np.abs(want)
    rel = np.linalg.norm(err) / np.linalg.norm(want)
    limit = ep / 3 ** 0.5 + eo + 5 * 2.0 ** -11
    print(f"  worst error/bound {(err / bound).max():.3f}, relative 2-norm {rel:.2e} of {limit:.2e}")
    assert np.isfinite(got).all() and (err <= bound).all() and rel <= limit


@pytest.mark.parametrize("rising", [False, True], ids=["normal", "rising"])
@pytest.mark.parametrize("case", LAUNCHES, ids=lambda c: f"{c[0][0]}-{c[0][1]}w{c[0][2]}-{'-'.join(map(str, c[1]))}-"
                                                         f"c{int(c[2])}-{c[3]}-{c[4]}")
def test_launch(case, rising, hip_impl, gpu_device):
    (kernel, _, _), shape, causal, dtype, pv = case
    print(f"[launch] {case} rising={rising}", flush=True)
    B, Hq, Hkv, Nq, Nkv, D = shape
    q, k, v = _inputs(shape, dtype, rising, gpu_device)
    if kernel == "flash":
        o = _flash().run(q, k, v, causal=causal)
    else:
        o = hip_impl.run(q, k, v, causal=causal, pv_dtype=pv, fuse_q=kernel == PRO)
        pre = hip_impl.prepass(q, k, v)
    torch.cuda.synchronize()
    rows = sample_rows(Nq, seed=Nkv, sample=16)
    got, want, vmax = [], [], []
    for b, h in {(0, 0), (B // 2, Hq // 2), (B - 1, Hq - 1)}:
        one, kv = (slice(b, b + 1), slice(h, h + 1)), (slice(b, b + 1), slice(h * Hkv // Hq, h * Hkv // Hq + 1))
        vn = v[kv].float().cpu().numpy()
        if kernel == "flash":
            qr, kn = q[one][0, 0, rows].double().cpu().numpy(), k[kv][0, 0].double().cpu().numpy()
            s = qr @ kn.T * D ** -0.5
            if causal:
                s = np.where(np.arange(Nkv)[None] > rows[:, None], -np.inf, s)
            p = np.exp(s - s.max(axis=1, keepdims=True))
            want.append(p @ vn[0, 0].astype(np.float64) / p.sum(axis=1, keepdims=True))
        else:
            codes, vs = O.quant_v_fp8(vn) if pv == "fp8" else (vn, None)
            q8, qs, k8, ks = (pre[key][sl].cpu().numpy() for key, sl in
                              (("q8", one), ("q_scale", one), ("k8", kv), ("k_scale", kv)))
            want.append(O.sage_emulate(q8, qs, k8, ks, codes, causal=causal, v_scale=vs, rows=rows)[0, 0])
        got.append(o[one][0, 0, rows].double().cpu().numpy())
        vmax.append(np.abs(vn).max())
    assert torch.isfinite(o).all()
    _check(np.concatenate(got), np.concatenate(want), np.array(vmax), EP[pv or dtype], EO[dtype])
