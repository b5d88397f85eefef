"""Which launches sage_run and sage_flash_run take, and with which layouts, on
a host without a GPU: the C ABI's own source with recording stand-ins for the
pre-pass and the kernel launches (tests/native/run_routes.cpp)."""
from __future__ import annotations

import ctypes
import json
import random
import shutil
import subprocess
from pathlib import Path

import pytest

from tribench_amd import build as hip_build

HERE = Path(__file__).resolve().parent
PV = {"fp16": 0, "bf16": 1, "fp8": 2}
DT = {"fp32": 0, "fp16": 1, "bf16": 2}
BUF, Q8 = 1 << 20, 1 << 21  # addresses nothing reads


def _build_routes(out, hip_impl, *flags):
    if not (shutil.which("hipcc") or Path("/opt/rocm/bin/hipcc").exists()):
        pytest.skip("hipcc not available")
    hip_impl._load()  # (first: as a dependency of the stand-ins it would bind to them)
    so = hip_impl.library_path()
    subprocess.run([hip_build.hipcc(), *hip_build.COMMON, *flags, "-O0", "-w", "-shared", "-x", "hip",
                    str(HERE / "native" / "run_routes.cpp"), "-x", "none", str(so), f"-Wl,-rpath,{so.parent}",
                    "-Wl,-Bsymbolic", "-o", str(out)], check=True, capture_output=True)
    lib = ctypes.CDLL(str(out))
    lib.take_routes.restype = lib.sage_last_error.restype = ctypes.c_char_p
    for name in ("sage_run", "sage_flash_run"):
        getattr(lib, name).argtypes = [ctypes.c_char_p, ctypes.c_void_p]
        getattr(lib, name + "_workspace_bytes").restype = ctypes.c_size_t
        getattr(lib, name + "_workspace_bytes").argtypes = [ctypes.c_char_p]
    return lib


@pytest.fixture(scope="module")
def routes(tmp_path_factory, hip_impl):
    return _build_routes(tmp_path_factory.mktemp("routes") / "run_routes.so", hip_impl)


def dense(H, N, D):
    return [H * N * D, N * D, D]


def run_call(lib, hip_impl, B, Hq, Hkv, Nq, Nkv, D, *, flash=False, dtype="bf16", causal=False, pv="fp16", q_sub=128,
             smooth_k=1, fuse_q=-1, q_strides=None, outs=None, q8_strides=None, k8_strides=None):
    """(status, routes or message) of one call with the workspace it asks for;
    outs: addresses of q8, q_scale, k8, k_scale, km, v_scale."""
    sq, sk = dense(Hq, Nq, D), dense(Hkv, Nkv, D)
    name = "sage_flash_run" if flash else "sage_run"

    def pack(ws, n):
        return hip_impl._CALL.pack(hip_impl._CALL_SIZE, BUF, BUF, BUF, BUF, ws, n, *(q_strides or sq), *sk, *sk, *sq,
                                   B, Hq, Hkv, Nq, Nkv, D, 0.1, DT[dtype], int(causal), PV[pv], q_sub, smooth_k,
                                   fuse_q, *(outs or [0] * 6), *(q8_strides or [0] * 3), *(k8_strides or [0] * 3))

    if not flash:
        quant_q, v_tiles = ctypes.c_int(-1), ctypes.c_int(-1)
        assert lib.sage_run_stages(pack(0, 0), ctypes.byref(quant_q), ctypes.byref(v_tiles)) == 0
    n = getattr(lib, name + "_workspace_bytes")(pack(0, 0))
    lib.take_routes()
    rc = getattr(lib, name)(pack(BUF if n else 0, n), None)
    if rc:
        return rc, lib.sage_last_error().decode()
    got = [json.loads(line) for line in lib.take_routes().decode().splitlines()]
    if not flash:  # sage_run_stages says what the call then does
        assert (quant_q.value, v_tiles.value) == (got[0]["quant_q"], got[0]["v"]) == (got[0]["quant_q"], 1 - got[1]["vrow"])
    return 0, got


def test_fp8_keys_stay_in_one_sweep(routes, hip_impl):
    """FP8 P is rounded against the sweep's running max, so ranges would give
    other codes: whatever the shape, one range; rows of few heads may still
    share a work-group.  The same shapes with fp16 P do split."""
    rng = random.Random(1)
    split = packed = 0
    for _ in range(400):
        Hkv, G = rng.choice([1, 2, 3, 8, 16]), rng.choice([1, 2, 4, 6])
        shape = (rng.choice([1, 2, 8, 64, 200]), Hkv * G, Hkv, int(2 ** rng.uniform(0, 11)), int(2 ** rng.uniform(6, 15)),
                 rng.choice([64, 128]))
        kw = dict(dtype=rng.choice(list(DT)), causal=rng.random() < 0.3, fuse_q=rng.choice([-1, 0, 1]))
        rc, got = run_call(routes, hip_impl, *shape, pv="fp8", **kw)
        assert rc == 0, got
        assert got[-1]["nsplit"] == 1, (shape, kw, got)
        packed += got[-1]["grp"] > 1
        split += run_call(routes, hip_impl, *shape, pv="fp16", **kw)[1][-1]["nsplit"] > 1
    assert split > 50 and packed > 5


def test_gpu_packed_shapes_pack(routes, hip_impl):
    """The shapes that test_gpu_attn_split.py means to pack heads with FP8 P do."""
    from test_gpu_attn_split import PACKED

    for *shape, causal in PACKED:
        for D in (64, 128):
            rc, got = run_call(routes, hip_impl, *shape, D, causal=causal, pv="fp8")
            assert rc == 0 and got[-1]["launch"] == "i8 part" and got[-1]["grp"] > 1, got


# (B, Hq, Hkv, Nq, Nkv): Q in the prologue when left to choose; two that split the keys; packed heads
Q8_SHAPES = [(4, 32, 8, 512, 512), (1, 4, 2, 300, 4096), (2, 8, 2, 5, 3000), (64, 32, 8, 1, 200)]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape", Q8_SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_q8_layout_follows_the_options(routes, hip_impl, shape, D):
    """A caller's q8 has q's strides with fuse_q 1 and q8_strides otherwise,
    whatever launches the shape takes; q is a slice of packed Q, K, V rows."""
    B, Hq, Hkv, Nq, Nkv = shape
    q_strides = [Nq * 3 * Hq * D, D, 3 * Hq * D]
    q8_strides = [Hq * Nq * D + 64, Nq * D, D]
    outs = [Q8, BUF, 0, 0, 0, 0]
    seen = set()
    for fuse_q in (-1, 0, 1):
        # (with fuse_q 1 the caller need not fill q8_strides)
        rc, got = run_call(routes, hip_impl, *shape, D, fuse_q=fuse_q, q_strides=q_strides, outs=outs,
                           q8_strides=None if fuse_q == 1 else q8_strides)
        assert rc == 0, got
        pre, attn = got
        want = q_strides if fuse_q == 1 else q8_strides
        if pre["quant_q"]:
            assert pre["q8"] == Q8 and pre["q8_strides"] == want and attn["q_strides"] == want, got
        else:
            assert attn["q8_out"] == Q8 and attn["q_strides"] == q_strides == want, got
        seen.add(attn["launch"])
    assert ("i8 part" in seen) == (shape != Q8_SHAPES[0]), seen


def test_q8_rows_stay_aligned(routes, hip_impl):
    """q8 with q's strides is refused by those strides, not by the launch."""
    for shape in Q8_SHAPES:
        D = 64
        q_strides = [shape[1] * shape[3] * 72, shape[3] * 72, 72]
        kw = dict(q_strides=q_strides, outs=[Q8, BUF, 0, 0, 0, 0])
        rc, msg = run_call(routes, hip_impl, *shape, D, fuse_q=1, **kw)
        assert rc != 0 and "invalid argument" in msg and "q8" in msg, msg
        for fuse_q in (-1, 0):
            assert run_call(routes, hip_impl, *shape, D, fuse_q=fuse_q, q8_strides=dense(shape[1], shape[3], D), **kw)[0] == 0


@pytest.mark.parametrize("fuse_q", [0, 1])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(4, 32, 32, 1024, 1024, 128), (1, 2, 2, 256, 256, 64)],
                         ids=lambda s: "-".join(map(str, s)))
def test_no_workspace_needed(routes, hip_impl, shape, dtype, fuse_q):
    """Every output given, no K smoothing, V in place and one sweep: nothing to
    keep in a workspace, and the call runs without one."""
    B, Hq, Hkv, Nq, Nkv, D = shape
    kw = dict(dtype=dtype, pv=dtype, fuse_q=fuse_q, smooth_k=0, outs=[BUF] * 4 + [0, 0], q8_strides=dense(Hq, Nq, D),
              k8_strides=dense(Hkv, Nkv, D))
    rc, got = run_call(routes, hip_impl, *shape, **kw)
    assert rc == 0, got
    pre, attn = got
    assert attn["vrow"] == 1 and attn["nsplit"] == 1 and pre["quant_q"] == 1 - fuse_q
    assert run_call(routes, hip_impl, *shape, **{**kw, "smooth_k": 1})[0] == 0  # (a workspace for the sums)


def test_stages_of_typical_calls(routes, hip_impl):
    """What the harness times as run's pre-pass: Q where few blocks or a split
    want it there, V tiles where V is not of the P.V type."""
    for shape, kw, quant_q, v in [
        ((4, 32, 32, 4096, 4096, 128), dict(dtype="bf16"), 0, 1),
        ((8, 16, 16, 4096, 4096, 64), dict(dtype="fp16"), 0, 0),
        ((1, 2, 2, 256, 256, 64), dict(dtype="bf16"), 1, 1),
        ((2, 32, 8, 32, 16384, 128), dict(dtype="fp16"), 1, 0),
        ((2, 32, 8, 32, 16384, 128), dict(dtype="fp16", fuse_q=1), 1, 0),  # split: Q8 comes from the pre-pass
        ((1, 8, 8, 512, 512, 128), dict(dtype="bf16", pv="fp8", fuse_q=1), 0, 1),
    ]:
        rc, got = run_call(routes, hip_impl, *shape, **kw)
        assert rc == 0 and (got[0]["quant_q"], got[0]["v"]) == (quant_q, v), (shape, kw, got)


def test_gpu_launch_shapes_take_the_launch_they_name(routes, hip_impl):
    from test_gpu_launches import LAUNCHES

    for launch, shape, causal, dtype, pv in LAUNCHES:
        flash = launch[0] == "flash"
        kw = dict(flash=True) if flash else dict(pv=pv, fuse_q=int(launch[0] == "i8q"))
        rc, got = run_call(routes, hip_impl, *shape, dtype=dtype, causal=causal, **kw)
        assert rc == 0 and (got[-1]["launch"], got[-1]["nw"], got[-1]["wpe"]) == launch, (launch, shape, dtype, pv, got)
        assert got[-1]["vrow"] == int(flash or dtype == pv), got


def test_gpu_split_shapes_split(routes, hip_impl):
    """The shapes that test_gpu_attn_split.py compares with one sweep are split, in both packs."""
    from test_gpu_attn_split import ONE_SWEEP, SHAPES

    packed = set()
    for shape in SHAPES:
        for D in (64, 128):
            for kw in [dict(flash=True, dtype="fp16"), dict(flash=True), dict(dtype="bf16"), dict(dtype="fp32", pv="bf16"),
                       dict(dtype="fp16", fuse_q=1)]:
                rc, got = run_call(routes, hip_impl, *shape[:5], D, causal=shape[5], **kw)
                assert rc == 0 and (got[-1]["nsplit"] > 1 or shape in ONE_SWEEP), (shape, D, kw, got)
                if got[-1]["grp"] > 1:
                    packed.add(shape)
    assert len(packed) >= 3, packed


def test_trace_build_launches_once_unless_traced(routes, hip_impl, tmp_path):
    """The trace build times as the product does; only with a trace attached,
    and where the product's launch is not of 8 waves, one of 8 waves is added."""
    traced = _build_routes(tmp_path / "trace_routes.so", hip_impl, "-DSAGE_TRACE=2")
    traced.sage_trace_attach.argtypes = [ctypes.c_void_p, ctypes.c_int64]
    eight = (1, 24, 8, 1333, 1333, 128)
    for shape, kw in [(eight, {}), ((2, 24, 8, 961, 961, 64), {}), ((2, 8, 2, 32, 3000, 128), {}),
                      ((1, 24, 8, 1333, 2500, 128), dict(flash=True)), ((8, 32, 8, 1, 8192, 128), dict(flash=True))]:
        want = run_call(routes, hip_impl, *shape, **kw)[1]
        assert run_call(traced, hip_impl, *shape, **kw)[1] == want
        assert traced.sage_trace_attach(BUF, 1 << 30) == 0
        got = run_call(traced, hip_impl, *shape, **kw)[1]
        assert traced.sage_trace_attach(None, 0) == 0
        if want[-1]["nw"] == 8:
            assert got == want
        else:
            assert got[:-2] == want[:-1] and got[-1] == want[-1] and got[-2]["nw"] == 8, got
    assert run_call(routes, hip_impl, *eight)[1][-1]["nw"] == 8


def test_k_blocks_by_wave_only_where_that_is_faster(routes):
    """At head dim 128 the wave role takes its launch's other roles the registers:
    FP8 V tiles there, and long calls, keep a work-group to a K block."""
    def pay(nblk, D, vt_in_b, pv):
        return bool(routes.k_waves_pay(ctypes.c_int64(nblk), ctypes.c_int64(D), vt_in_b, PV[pv]))

    for nblk in (1024, 2048, 4448, 8192, 16384):
        for pv in PV:
            assert pay(nblk, 64, 1, pv) and pay(nblk, 64, 0, pv) == (nblk >= 2048)
            assert pay(nblk, 128, 1, pv) == (pv != "fp8" and nblk < 8192)
            assert pay(nblk, 128, 0, pv) == (2048 <= nblk < 8192)
    assert not pay(1023, 64, 1, "fp16") and not pay(1023, 128, 1, "fp16")


def test_stage_calls_keep_8_waves_for_few_rows(routes, hip_impl):
    """The stage calls cannot split keys; with a head's rows in one work-group
    and a CU to each, head dim 128 keeps 8 waves (they share the tile loads)."""
    i3 = ctypes.c_int64 * 3
    p = ctypes.c_void_p(BUF)
    routes.sage_attn_fwd.argtypes = hip_impl._load().sage_attn_fwd.argtypes
    for (B, Hq, Hkv, Nq, Nkv, D), pv, nw in [
        ((4, 6, 3, 58, 9570, 128), "fp16", 8), ((4, 6, 3, 128, 9570, 128), "bf16", 8), ((1, 2, 2, 1, 200, 128), "fp16", 8),
        ((4, 6, 3, 58, 9570, 128), "fp8", 4), ((4, 6, 3, 58, 9570, 64), "fp16", 4), ((4, 6, 3, 129, 9570, 128), "fp16", 4),
        ((16, 32, 8, 58, 4000, 128), "fp16", 4),
    ]:
        sq, sk = i3(*dense(Hq, Nq, D)), i3(*dense(Hkv, Nkv, D))
        routes.take_routes()
        assert routes.sage_attn_fwd(p, sq, p, p, sk, p, p, hip_impl.DTYPE_VTILES, None, p, p, DT["fp32"], sq, B, Hq, Hkv,
                                    Nq, Nkv, D, 0, 128, 64, 128, PV[pv], None) == 0
        got = json.loads(routes.take_routes())
        assert got["nw"] == nw, (B, Hq, Nq, Nkv, D, pv, got)
