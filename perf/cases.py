"""The attention calls whose time is tracked, with their inputs and exact results.

Each case is one call of a pack's ``hip`` variant, looked up the way the
harness does: ``run(q, k, v, causal, ...)`` of sage_attn (INT8 QK^T with the
pre-pass inside the call) or of flash_attn (fp16/bf16 QK^T).  Together they
cover what the two packs are called for: whole-sequence attention from the
smallest benchmark configuration to the largest, causal and not, attention
over another sequence (short text keys, few or single query rows over a long
context), grouped KV heads, both layouts, both head dims, all input types,
P.V types and Q-scale granularities.

``exact`` restates each path in float64.  For sage_attn the INT8 codes (and
the e4m3 codes of V) are part of the operation's definition, so the codes are
formed as the pre-pass defines them and everything else is float64.
"""
from __future__ import annotations

import functools
import math

import torch

from tribench_amd.harness.packs import PackIndex

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BLKQ, BLKK = 128, 64  # rows per Q / K quantization block
Q_ROWS = {"block": BLKQ, "wave": 32, "thread": 1}  # rows per Q scale
LARGEST_FLOPS = 7.0e12  # a drawn case's limit (the largest listed ones do 7.8e12 and 8.8e12)


def _case(pack, dtype, B, Hq, Hkv, Nq, Nkv, D, causal=False, layout="HND", pv="fp16", q_gran="block",
          v_dist="normal", name=None):
    c = dict(pack=pack, dtype=dtype, B=B, Hq=Hq, Hkv=Hkv, Nq=Nq, Nkv=Nkv, D=D, causal=causal, layout=layout,
             pv=pv, q_gran=q_gran, v_dist=v_dist)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest benchmark configuration: latency and launches
        _case("sage_attn", "bf16", 1, 2, 2, 256, 256, 64, name="sage_small"),
        # one ragged sequence of ordinary length, sequence-major layout, per-row Q scales
        _case("sage_attn", "fp16", 1, 24, 24, 1333, 1333, 128, layout="NHD", q_gran="thread", name="sage_ragged_mid"),
        # the pack's first case in the harness's default type: a training-size batch at head dim 64
        _case("sage_attn", "fp16", 8, 16, 16, 4096, 4096, 64, name="sage_s4k_d64"),
        # the headline benchmark configuration
        _case("sage_attn", "bf16", 4, 32, 32, 4096, 4096, 128, name="sage_s4k_d128"),
        # prefill of a short batch from a model kept in fp32, bf16 P.V
        _case("sage_attn", "fp32", 2, 32, 32, 2048, 2048, 128, causal=True, pv="bf16", name="sage_causal_2k_fp32"),
        # the GQA benchmark configuration: long ragged video-length sequence, head dim 64
        _case("sage_attn", "bf16", 2, 48, 8, 17776, 17776, 64, name="sage_gqa_ragged_d64"),
        # the FP8 benchmark configuration: long causal prefill, heavy-tailed V, per-wave Q scales
        _case("sage_attn", "bf16", 1, 32, 32, 32768, 32768, 128, causal=True, pv="fp8", q_gran="wave",
              v_dist="student_t", name="sage_causal_fp8"),
        # cross attention of that video-length sequence over a short text
        _case("sage_attn", "bf16", 2, 48, 48, 17776, 226, 64, name="sage_cross_text"),
        # a few new query tokens over a long context
        _case("sage_attn", "fp16", 2, 32, 8, 32, 16384, 128, name="sage_few_queries"),
        # the flash pack's own case at head dim 128
        _case("flash_attn", "bf16", 4, 32, 32, 4096, 4096, 128, name="flash_s4k_d128"),
        # a small causal prefill
        _case("flash_attn", "fp16", 1, 16, 16, 512, 512, 64, causal=True, name="flash_small_causal"),
        # decode: one query row per sequence over a long context, grouped KV heads
        _case("flash_attn", "bf16", 8, 32, 8, 1, 8192, 128, name="flash_decode"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: self attention, attention over another sequence, or a
    few query rows, of either pack; lengths log-uniform (so mostly odd)."""
    while True:
        pack = rng.choice(["sage_attn", "sage_attn", "flash_attn"])
        dtype = rng.choice(["bf16", "bf16", "fp16"] if pack == "flash_attn" else ["bf16", "bf16", "fp16", "fp32"])
        D = rng.choice([64, 128])
        kind = rng.choice(["self", "self", "cross", "few"])
        B = rng.choice([1, 1, 2, 3, 4, 8])
        Hkv = rng.choice([1, 2, 3, 4, 8, 12, 16])
        Hq = Hkv * rng.choice([1, 1, 2, 4, 6])
        causal = False
        if kind == "self":
            Nq = Nkv = _log_int(rng, 128, 24000)
            causal = rng.random() < 0.5
        elif kind == "cross":
            Nq, Nkv = _log_int(rng, 256, 18000), _log_int(rng, 64, 2048)
        else:
            Nq, Nkv = _log_int(rng, 1, 64), _log_int(rng, 512, 32768)
        sage = pack == "sage_attn"
        c = _case(pack, dtype, B, Hq, Hkv, Nq, Nkv, D, causal=causal, layout=rng.choice(["HND", "NHD"]),
                  pv=rng.choice(["fp16", "fp16", "bf16", "fp8"]) if sage else "fp16",
                  q_gran=rng.choice(["block", "wave", "thread"]) if sage else "block",
                  v_dist=rng.choice(["normal", "normal", "student_t"]))
        if work(c)["flops"] <= (LARGEST_FLOPS if sage else LARGEST_FLOPS / 4):
            return c


# --------------------------------------------------------------------------
# inputs and the call
# --------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _variant(pack):
    return PackIndex().pack(pack).variant("hip")


def _hnd(case, seed):
    """q, k, v as [B, H, N, D] views in the case's layout, seeded on the GPU:
    unit-variance rows, a constant per-channel offset of K (what K smoothing
    removes), V normal or Student-t with 3 degrees of freedom."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    B, D, nhd = case["B"], case["D"], case["layout"] == "NHD"

    def randn(h, n):
        shape = (B, n, h, D) if nhd else (B, h, n, D)
        t = torch.randn(shape, generator=g, device=dev)
        return t.transpose(1, 2) if nhd else t

    q = randn(case["Hq"], case["Nq"])
    k = randn(case["Hkv"], case["Nkv"])
    k += 2.0 * randn(case["Hkv"], 1)
    v = randn(case["Hkv"], case["Nkv"])
    if case["v_dist"] == "student_t":
        chi2 = sum(randn(case["Hkv"], case["Nkv"]).square_() for _ in range(3))
        v /= (chi2 / 3).sqrt_()
    dt = DTYPES[case["dtype"]]
    return q.to(dt), k.to(dt), v.to(dt)


def prepare(case, seed):
    q, k, v = _hnd(case, seed)
    if case["layout"] == "NHD":
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    kw = {"causal": case["causal"], "tensor_layout": case["layout"]}
    if case["pack"] == "sage_attn":
        kw.update(pv_dtype=case["pv"], q_gran=case["q_gran"])
    return {"fn": _variant(case["pack"]), "q": q, "k": k, "v": v, "kw": kw}


def run(state):
    return state["fn"](state["q"], state["k"], state["v"], **state["kw"])


def work(case):
    """Q, K, V read once and O written once; 4*D operations per unmasked pair."""
    es = 4 if case["dtype"] == "fp32" else 2
    B, Hq, Hkv, Nq, Nkv, D = (case[x] for x in ("B", "Hq", "Hkv", "Nq", "Nkv", "D"))
    pairs = Nq * (Nq + 1) // 2 if case["causal"] else Nq * Nkv
    return {"bytes": es * B * D * (2 * Hq * Nq + 2 * Hkv * Nkv), "flops": 4 * B * Hq * D * pairs}


def tolerance(case):
    """About four times the distance of the outputs from ``exact`` (measured
    1.8e-3 to 2.4e-3 with bf16 outputs or bf16 P, 2.8e-4 to 4.6e-4 with fp16,
    2.1e-2 with FP8 P.V): the rounding of the output and of P to their types."""
    if case["pv"] == "fp8" and case["pack"] == "sage_attn":
        return {"rel": 8e-2}
    if case["dtype"] == "bf16" or case["pv"] == "bf16":
        return {"rel": 8e-3}
    return {"rel": 1.6e-3}


# --------------------------------------------------------------------------
# float64 results
# --------------------------------------------------------------------------
def _int8(x, rows):
    """INT8 codes times scale of x [N, D] in groups of ``rows`` rows: scale =
    max|x| / 127, codes rounded half away from zero; float64."""
    n, d = x.shape
    pad = -n % rows
    xp = torch.cat([x, x.new_zeros(pad, d)]) if pad else x
    xg = xp.view(-1, rows * d)
    scale = xg.abs().amax(dim=1, keepdim=True) / 127.0
    t = torch.where(scale > 0, xg / scale, torch.zeros_like(xg))
    codes = torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t))
    return (codes * scale).view(-1, d)[:n]


def _e4m3(v):
    """V through per-channel e4m3: scale = max|v| / 448 over the tokens."""
    scale = (v.abs().amax(dim=0, keepdim=True) / 448.0).float()
    codes = torch.where(scale > 0, v.float() / scale, torch.zeros_like(v, dtype=torch.float32))
    return codes.to(torch.float8_e4m3fn).double() * scale.double()


def exact(case, seed):
    q, k, v = _hnd(case, seed)
    B, Hq, Hkv, Nq, Nkv, D = (case[x] for x in ("B", "Hq", "Hkv", "Nq", "Nkv", "D"))
    sage, causal = case["pack"] == "sage_attn", case["causal"]
    mul = float(torch.tensor(D ** -0.5 * 1.44269504, dtype=torch.float32))  # scores in log2 units
    out = torch.empty((B, Hq, Nq, D), dtype=torch.float64, device=q.device)
    step = max(1, min(Nq, (1 << 28) // Nkv))  # 2 GiB of scores at a time
    cols = torch.arange(Nkv, device=q.device)
    for b in range(B):
        for hk in range(Hkv):
            kk, vv = k[b, hk].double(), v[b, hk].double()
            if sage:
                kk = _int8(kk - kk.mean(dim=0, keepdim=True), BLKK)
                if case["pv"] == "fp8":
                    vv = _e4m3(vv)
            kt = kk.t().contiguous()
            for h in range(hk * (Hq // Hkv), (hk + 1) * (Hq // Hkv)):
                qq = q[b, h].double() * mul
                if sage:
                    qq = _int8(qq, Q_ROWS[case["q_gran"]])
                for i0 in range(0, Nq, step):
                    i1 = min(i0 + step, Nq)
                    n1 = min(i1, Nkv) if causal else Nkv
                    s = qq[i0:i1] @ kt[:, :n1]
                    if causal:
                        rows = torch.arange(i0, i1, device=q.device)
                        s.masked_fill_(cols[None, :n1] > rows[:, None], float("-inf"))
                    s -= s.amax(dim=1, keepdim=True)
                    s.exp2_()
                    den = s.sum(dim=1, keepdim=True)
                    out[b, h, i0:i1] = (s @ vv[:n1]) / den
    return out.transpose(1, 2) if case["layout"] == "NHD" else out
