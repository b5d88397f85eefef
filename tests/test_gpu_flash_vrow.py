"""V read in place by the unquantized kernel (sage_flash_run) against the V tile path.

At lengths around the 64-key tile (one key, a tail of one, whole tiles, the
mask-free loop with and without leftovers), for both types and head dims,
causal and not, and with V rows that are slices of wider rows.  One sweep over
one tile of keys does the same arithmetic in the same order on the same V bits:
equal bit for bit.  With more keys the call may be split over them, so that P
and O are rounded against other maxima: with e the types' rounding (2^-11,
bf16 2^-9), P differs by e relative on either side, O by e |o|, and the fp16
row sums by 5 * 2^-11 each, hence |a - b| <= 2 e max|v| + (2 e + 10 * 2^-11) |o|.
V rows too far apart for the in-place loads take the tile path.
"""
from __future__ import annotations

import ctypes
import importlib.util
from pathlib import Path

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
FLASH = Path(__file__).resolve().parents[1] / "tribench_amd" / "kernels" / "flash_attn" / "hip_impl.py"


def _flash():
    spec = importlib.util.spec_from_file_location("flash_vrow_impl", FLASH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _tiles(H, q, k, v, causal, layout="HND"):
    """sage_vtiles + sage_flash_fwd, stage by stage."""
    lib = H._load()
    B, Hq, Hkv, Nq, Nkv, D = H._check_inputs(q, k, v, layout)
    vt = H.vtiles(v, {torch.float16: "fp16", torch.bfloat16: "bf16"}[q.dtype], tensor_layout=layout)
    o = torch.empty_like(q)
    mul = ctypes.c_float(float(np.float32(D ** -0.5 * H.LOG2E_REF)))
    rc = lib.sage_flash_fwd(H._ptr(q), H._strides(q, layout), H._ptr(k), H._strides(k, layout), H._ptr(vt),
                            H.DTYPE_VTILES, None, H._ptr(o), H._strides(o, layout), H._TORCH_CODES[q.dtype],
                            B, Hq, Hkv, Nq, Nkv, D, mul, int(causal), H._stream(q.device))
    H._check(rc, "sage_flash_fwd")
    return o


def _same(got, want, v, key_dim=2):
    torch.cuda.synchronize()
    if v.shape[key_dim] <= 64:
        assert torch.equal(got, want)
        return
    e = 2.0 ** -9 if v.dtype == torch.bfloat16 else 2.0 ** -11
    got, want = got.double(), want.double()
    bound = 2 * e * v.double().abs().max() + (2 * e + 10 * 2.0 ** -11) * want.abs()
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Nq,Nkv,causal", [(1, 1, False), (5, 63, False), (65, 65, True), (129, 128, False),
                                           (300, 257, False), (448, 448, True), (33, 705, False)])
def test_in_place_equals_tiles(D, dtype, Nq, Nkv, causal, gpu_device):
    print(f"[vrow] D{D} {dtype} {Nq}/{Nkv} causal={causal}", flush=True)
    F = _flash()
    g = torch.Generator().manual_seed(Nq * 1000 + Nkv)
    q = torch.randn(2, 4, Nq, D, generator=g).to(dtype).to(gpu_device)
    k = torch.randn(2, 2, Nkv, D, generator=g).to(dtype).to(gpu_device)
    wide = torch.randn(2, Nkv, 2, D + 8, generator=g).to(dtype).to(gpu_device)  # sequence-major, padded rows
    v = wide[..., :D].transpose(1, 2)
    _same(F.run(q, k, v, causal=causal), _tiles(F._H, q, k, v, causal), v)
    nhd = [t.transpose(1, 2).contiguous() for t in (q, k, v)]
    _same(F.run(*nhd, causal=causal, tensor_layout="NHD"), _tiles(F._H, *nhd, causal, "NHD"), nhd[2], key_dim=1)


def test_far_apart_rows_take_the_tile_path(gpu_device):
    F = _flash()
    base = torch.randn((1 << 25) + 64, device=gpu_device, dtype=torch.float16)
    v = base.as_strided((1, 1, 2, 64), (0, 0, 1 << 25, 1))
    q, k = (torch.randn(1, 1, 2, 64, device=gpu_device, dtype=torch.float16) for _ in range(2))
    got = F.run(q, k, v)
    torch.cuda.synchronize()
    assert torch.equal(got, F.run(q, k, v.contiguous()))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Nq,Nkv", [(1, 3, 1000), (1, 65, 65), (24, 300, 257)])
def test_infinite_last_v_row_stays_infinite(D, dtype, B, Nq, Nkv, hip_impl, gpu_device):
    """The keys that pad the last block weigh 0 times 0, not 0 times the last
    row's infinity: its channels are infinite and the others as without it."""
    print(f"[vrow inf] D{D} {dtype} {B}/{Nq}/{Nkv}", flush=True)
    g = torch.Generator().manual_seed(Nkv)
    q, k, v = (torch.randn(B, 4, n, D, generator=g).to(dtype).to(gpu_device) for n in (Nq, Nkv, Nkv))
    vi = v.clone()
    vi[:, :, -1, 5] = float("inf")
    vi[:, :, -1, 40] = float("-inf")
    pv = "fp16" if dtype == torch.float16 else "bf16"
    for run in (_flash().run, lambda *t: hip_impl.run(*t, pv_dtype=pv)):
        want, got = run(q, k, v).clone(), run(q, k, vi)
        want[..., 5], want[..., 40] = float("inf"), float("-inf")
        torch.cuda.synchronize()
        assert torch.equal(got, want)
