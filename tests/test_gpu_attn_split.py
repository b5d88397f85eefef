"""Attention split over the keys (partial kernels and merge) against one sweep.

``run`` chooses the split and the packing of grouped heads by the shape; the
stage entry points (``attention`` on the pre-pass's own outputs, sage_flash_fwd
on V tiles) always sweep all keys at once.  Q8, K8 and the scales are the same;
P is rounded to its type against another running max (e_p, relative: half an
ulp, 2^-11 fp16, 2^-8 bf16 with its 8 significant bits), the row sums of fp16 P
carry 5 * 2^-11 each, and O is rounded to its type (e_o), so
  |a - b| <= 2 e_p max|v| + (2 e_o + 10 * 2^-11) |o|.
The roundings of P are independent of V, so the relative 2-norm of a - b is
within their rms on both sides, 2 e_p / sqrt(3), plus 2 e_o + 10 * 2^-11.
FP8 P would move by 2^-4, the type's whole error, so its keys are not split; its
packed heads sweep the same blocks: equal bit for bit.  With integer scores P,
its sums and the merge's weights are exact: the exact result in every type.
Shapes: single rows, rows that fill a tile with packed heads and ones that end
in the middle of a head, keys that leave the last range short, causal rows that
see nothing of a range, every Q-scale granularity, both layouts.
"""
from __future__ import annotations

import pytest
import torch

from test_gpu_flash_vrow import _flash, _tiles

pytestmark = pytest.mark.gpu
E = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}
DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EO = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 2.0 ** -24}

# (B, Hq, Hkv, Nq, Nkv, causal)
SHAPES = [(1, 1, 1, 1, 65, False), (1, 4, 1, 1, 4097, False), (2, 6, 2, 37, 3000, False),
          (3, 8, 2, 32, 1000, False), (1, 12, 3, 127, 2111, False), (1, 2, 2, 130, 5000, False),
          (1, 2, 1, 1500, 1500, True), (1, 3, 3, 777, 777, True), (1, 1, 1, 3, 900, False),
          (16, 32, 4, 3, 777, False), (4, 24, 4, 37, 2000, False), (1, 3, 3, 1100, 1100, True)]
ONE_SWEEP = [SHAPES[0], SHAPES[7]]  # no gain from ranges (of SHAPES[7] at D = 64); the others are split
PACKED = [(64, 32, 8, 1, 200, False), (96, 18, 3, 5, 131, False), (64, 16, 2, 3, 700, False)]  # FP8 too


def _inputs(shape, D, dtype, dev, seed=3):
    B, Hq, Hkv, Nq, Nkv, _ = shape
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Hq, Nq, D, generator=g)
    k = torch.randn(B, Hkv, Nkv, D, generator=g) + 2.0 * torch.randn(B, Hkv, 1, D, generator=g)
    v = torch.randn(B, Hkv, Nkv, D, generator=g)
    return [t.to(DT[dtype]).to(dev) for t in (q, k, v)]


def _close(got, want, v, ep, eo):
    torch.cuda.synchronize()
    got, want = got.double(), want.double()
    assert torch.isfinite(got).all()
    bound = 2 * ep * v.double().abs().max() + (2 * eo + 10 * 2.0 ** -11) * want.abs()
    worst = ((got - want).abs() / bound).max().item()
    rel, limit = ((got - want).norm() / want.norm()).item(), 2 * ep / 3 ** 0.5 + 2 * eo + 10 * 2.0 ** -11
    print(f"  worst error/bound {worst:.3f}, relative 2-norm {rel:.2e} of {limit:.2e}")
    assert worst <= 1.0 and rel <= limit


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(str(int(x)) for x in s))
def test_int8_split_matches_one_sweep(shape, D, hip_impl, gpu_device):
    causal = shape[5]
    for i, (pv, gran, dtype) in enumerate([("fp16", "block", "bf16"), ("bf16", "wave", "fp16"),
                                           ("fp8", "thread", "fp32"), ("fp16", "wave", "fp16"),
                                           ("bf16", "thread", "bf16")]):  # the last two: V in place
        print(f"[split] {shape} D{D} {pv} {gran} {dtype}", flush=True)
        q, k, v = _inputs(shape, D, dtype, gpu_device)
        layout = "NHD" if i in (1, 4) else "HND"
        if i == 3:  # V rows that are slices of wider ones
            wide = torch.zeros(*v.shape[:3], D + 24, dtype=v.dtype, device=v.device)
            wide[..., :D] = v
            v = wide[..., :D]
        if layout == "NHD":
            q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
        o, pre = hip_impl.run(q, k, v, causal=causal, pv_dtype=pv, q_gran=gran, tensor_layout=layout, fuse_q=False,
                              return_intermediates=True)
        q_sub = hip_impl.q_sub_of(gran)
        stage = hip_impl.prepass(q, k, v, q_sub=q_sub, pv_dtype=pv, tensor_layout=layout)
        for key in ("q8", "q_scale", "k8", "k_scale", "km"):
            assert torch.equal(pre[key], stage[key]), key
        want = hip_impl.attention(q, k, v, stage, causal, pv_dtype=pv, q_sub=q_sub, tensor_layout=layout)
        if pv == "fp8":
            assert torch.equal(o, want)
        else:
            _close(o, want, v, E[pv], EO[dtype])
        fused = hip_impl.run(q, k, v, causal=causal, pv_dtype=pv, q_gran=gran, tensor_layout=layout, fuse_q=True)
        assert torch.equal(fused, o)  # where Q is quantized changes no bit


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape", SHAPES + PACKED, ids=lambda s: "-".join(str(int(x)) for x in s))
def test_fp8_rows_do_not_depend_on_the_call(shape, D, hip_impl, gpu_device):
    """FP8 P: the whole call gives one sweep's bits in every type, layout and
    Q granularity, heads packed or not, and so does a batch entry alone."""
    causal = shape[5]
    for gran, dtype, layout in [("block", "bf16", "HND"), ("wave", "fp16", "NHD"), ("thread", "fp32", "HND")]:
        print(f"[fp8 rows] {shape} D{D} {gran} {dtype} {layout}", flush=True)
        q, k, v = _inputs(shape, D, dtype, gpu_device)
        if layout == "NHD":
            q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
        kw = dict(pv_dtype="fp8", tensor_layout=layout)
        o = hip_impl.run(q, k, v, causal=causal, q_gran=gran, **kw)
        q_sub = hip_impl.q_sub_of(gran)
        stage = hip_impl.prepass(q, k, v, q_sub=q_sub, **kw)
        assert torch.equal(o, hip_impl.attention(q, k, v, stage, causal, q_sub=q_sub, **kw))
        one = hip_impl.run(*(t[-1:] for t in (q, k, v)), causal=causal, q_gran=gran, **kw)
        torch.cuda.synchronize()
        assert torch.equal(one, o[-1:])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(str(int(x)) for x in s))
def test_flash_split_matches_one_sweep(shape, dtype, D, gpu_device):
    print(f"[flash split] {shape} D{D} {dtype}", flush=True)
    F = _flash()
    q, k, v = _inputs(shape, D, dtype, gpu_device)
    _close(F.run(q, k, v, causal=shape[5]), _tiles(F._H, q, k, v, shape[5]), v, E[dtype], EO[dtype])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape", SHAPES + PACKED, ids=lambda s: "-".join(str(int(x)) for x in s))
def test_split_exact(shape, D, hip_impl, gpu_device):
    """Scores in -2 .. 2: every P is one of five consecutive powers of two, 32
    of which fp16 adds exactly, whatever maximum a range has.  A channel of 127
    that the other operand does not have makes the INT8 scales 1."""
    B, Hq, Hkv, Nq, Nkv, causal = shape
    g = torch.Generator().manual_seed(Nkv + D)
    q8, k8 = torch.zeros(B, Hq, Nq, D), torch.zeros(B, Hkv, Nkv, D)
    q8[..., :2] = torch.randint(-1, 2, (B, Hq, Nq, 2), generator=g).float()
    k8[..., :2] = torch.randint(-1, 2, (B, Hkv, Nkv, 2), generator=g).float()
    v = torch.randint(-1, 2, (B, Hkv, Nkv, D), generator=g) * 2.0 ** torch.randint(0, 4, (B, Hkv, Nkv, D), generator=g)
    v[:, :, 0] = 8.0  # FP8: every channel's scale is 8 / 448, its codes exact
    s = (q8[..., :2].double().reshape(B, Hkv, -1, 2) @ k8[..., :2].double().transpose(2, 3)).reshape(B, Hq, Nq, Nkv)
    if causal:
        s.masked_fill_(torch.arange(Nkv)[None] > torch.arange(Nq)[:, None], float("-inf"))
    p = torch.exp2(s).reshape(B, Hkv, -1, Nkv)
    want = ((p @ v.double()) / p.sum(dim=3, keepdim=True)).reshape(B, Hq, Nq, D)
    sm_scale = 1.0 / 1.44269504

    def check(o, dtype):
        torch.cuda.synchronize()
        err = (o.double().cpu() - want).abs()
        print(f"  max error {err.max():.2e}")
        assert (err <= 1e-5 * (1.0 + want.abs()) + EO[dtype] * want.abs()).all()

    F = _flash()
    for dtype in ("fp16", "bf16"):
        print(f"[split exact] {shape} D{D} flash {dtype}", flush=True)
        check(F.run(*(t.to(DT[dtype]).to(gpu_device) for t in (q8, k8, v)), causal=causal, sm_scale=sm_scale), dtype)
    q8[..., 2], k8[..., 3] = 127.0, 127.0
    for pv, dtype in [("fp16", "fp32"), ("bf16", "fp32"), ("fp8", "fp32"), ("fp16", "fp16"), ("bf16", "bf16")]:
        print(f"[split exact] {shape} D{D} {pv} {dtype}", flush=True)
        check(hip_impl.run(*(t.to(DT[dtype]).to(gpu_device) for t in (q8, k8, v)), causal=causal, sm_scale=sm_scale,
                           pv_dtype=pv, smooth_k=False), dtype)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("N,causal", [(1, False), (64, False), (193, True), (577, False)])
def test_int8_v_in_place_equals_tiles(N, causal, dtype, D, hip_impl, gpu_device):
    """Enough heads for one sweep per work-group: V in place and V tiles then
    do the same arithmetic, so the outputs are equal bit for bit."""
    print(f"[int8 vrow] N{N} D{D} {dtype} causal={causal}", flush=True)
    q, k, v = _inputs((16, 48, 48, N, N, causal), D, dtype, gpu_device)
    o = hip_impl.run(q, k, v, causal=causal, pv_dtype=dtype)
    stage = hip_impl.prepass(q, k, v, pv_dtype=dtype)
    assert torch.equal(o, hip_impl.attention(q, k, v, stage, causal, pv_dtype=dtype))


def test_int8_far_apart_v_rows_take_the_tile_path(hip_impl, gpu_device):
    base = torch.randn((1 << 25) + 64, device=gpu_device, dtype=torch.float16)
    v = base.as_strided((1, 1, 2, 64), (0, 0, 1 << 25, 1))
    q, k = (torch.randn(1, 1, 2, 64, device=gpu_device, dtype=torch.float16) for _ in range(2))
    assert torch.equal(hip_impl.run(q, k, v), hip_impl.run(q, k, v.contiguous()))


def test_split_handles_extreme_scores(gpu_device):
    """A range whose scores are all far below another's weighs nothing; NaN
    keys reach every row, as in one sweep."""
    F = _flash()
    q, k, v = _inputs((1, 1, 1, 3, 4096, False), 64, "fp16", gpu_device)
    k[:, :, :2048] = 0
    k[:, :, 2048:] = 200.0 * q[:, :, :1]
    _close(F.run(q, k, v), _tiles(F._H, q, k, v, False), v, E["fp16"], EO["fp16"])
    k[:, :, 4000] = float("nan")
    assert torch.isnan(F.run(q, k, v)).all()
