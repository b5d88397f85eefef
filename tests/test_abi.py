"""The C-ABI library on a host without a GPU: it loads, exports every symbol
of include/sage_attn.h and sage_attn_run.h, and rejects bad arguments before
touching a device."""
from __future__ import annotations

import ctypes
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "sage_attn.h"
RUN_HEADER = ROOT / "include" / "sage_attn_run.h"


def _declared_functions(header=HEADER):
    text = header.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sage_[a-z_0-9]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib(hip_impl):
    return hip_impl._load()


def test_header_declares_the_entry_points():
    assert _declared_functions() == ["sage_abi_version", "sage_attn_fwd", "sage_attn_fwd_q", "sage_flash_fwd",
                                     "sage_last_error", "sage_prepass", "sage_prepass_vt",
                                     "sage_prepass_vt_noalloc", "sage_prepass_workspace_bytes",
                                     "sage_vtile_bytes", "sage_vtiles"]


def _declared_arg_counts(header=HEADER):
    """Parameter count of every function declared in the header."""
    text = re.sub(r"/\*.*?\*/", "", header.read_text(), flags=re.S)
    out = {}
    for name, params in re.findall(r"\b(sage_[a-z_0-9]+)\s*\(([^;{]*?)\)\s*;", text, flags=re.S):
        params = params.strip()
        out[name] = 0 if params in ("", "void") else params.count(",") + 1
    return out


def test_bindings_match_the_header_argument_counts(lib):
    """hip_impl binds every entry point with exactly the header's number of
    parameters: a signature change on one side without the other fails here
    instead of passing garbage through ctypes."""
    counts = _declared_arg_counts()
    assert set(counts) == set(_declared_functions())
    for name, n in counts.items():
        fn = getattr(lib, name)
        assert fn.argtypes is not None, name
        assert len(fn.argtypes) == n, f"{name}: header {n} parameters, binding {len(fn.argtypes)}"


def test_library_exports_every_declared_symbol(lib):
    for name in _declared_functions():
        assert hasattr(lib, name), name


def test_abi_version_matches_header(lib, hip_impl):
    m = re.search(r"#define SAGE_ABI_VERSION (\d+)", HEADER.read_text())
    assert lib.sage_abi_version() == int(m.group(1)) == hip_impl.ABI_VERSION


def test_workspace_bytes(lib):
    # smooth_k: B*Hkv*nch*D fp32 partial sums; FP8 V adds as many channel maxima
    nch = 16  # N = 4096 -> 16 chunks of 256 tokens
    assert lib.sage_prepass_workspace_bytes(4, 32, 4096, 128, 1, 0) == 4 * 32 * nch * 128 * 4
    assert lib.sage_prepass_workspace_bytes(4, 32, 4096, 128, 1, 1) == 2 * 4 * 32 * nch * 128 * 4
    assert lib.sage_prepass_workspace_bytes(4, 32, 4096, 128, 0, 0) == 0


def test_noalloc_prepass_rejects_before_touching_a_device(lib):
    """The fixed-scratch pre-pass checks its size limit (and a null V tile
    buffer) before any HIP call."""
    m = re.search(r"#define SAGE_SCRATCH_BYTES \((\d+)u << (\d+)\)", HEADER.read_text())
    limit = int(m.group(1)) << int(m.group(2))
    assert limit == 4 << 20
    a = _prepass_args(B=16, Hq=64, Hkv=64, Nq=4096, Nkv=4096, D=128, smooth=1, km=ctypes.c_void_p(16))
    assert lib.sage_prepass_workspace_bytes(16, 64, 4096, 128, 1, 0) > limit
    fn = lib.sage_prepass_vt_noalloc
    rc = fn(*a[:-3], 0, ctypes.c_void_p(16), ctypes.c_size_t(1 << 30), None)
    msg = lib.sage_last_error().decode()
    assert rc != 0 and "invalid argument" in msg and "scratch" in msg, msg
    rc = fn(*_prepass_args()[:-3], 0, None, ctypes.c_size_t(0), None)
    msg = lib.sage_last_error().decode()
    assert rc != 0 and "invalid argument" in msg and "vtiles" in msg, msg


def _prepass_args(**over):
    s3 = (ctypes.c_int64 * 3)(0, 0, 0)
    a = dict(q=ctypes.c_void_p(16), k=ctypes.c_void_p(16), v=None, in_dtype=2, B=1, Hq=2, Hkv=2, Nq=64, Nkv=64,
             D=64, qs=s3, ks=s3, vs=None, mul=0.18, blkq=128, blkk=64, q_sub=128, smooth=0, vmode=0,
             q8=ctypes.c_void_p(16), q8s=s3, qsc=ctypes.c_void_p(16), k8=ctypes.c_void_p(16), k8s=s3,
             ksc=ctypes.c_void_p(16), km=None, v8=None, v8s=None, vsc=None, ws=None, wsb=0, st=None)
    a.update(over)
    return list(a.values())


@pytest.mark.parametrize("over,needle", [
    (dict(D=96), "head_dim"),
    (dict(Hq=3, Hkv=2), "multiple"),
    (dict(B=0), "empty shape"),
    (dict(blkq=100), "blkq"),
    (dict(q_sub=48), "q_sub"),
    (dict(q_sub=2), "q_sub"),
    (dict(q_sub=0), "q_sub"),
    (dict(in_dtype=7), "in_dtype"),
    (dict(smooth=1), "km is null"),
    (dict(q=None), "null pointer"),
    (dict(q=ctypes.c_void_p(8)), "aligned"),
    (dict(q=None, qs=None, q8s=None, qsc=None), "null pointer"),  # q8 given without q
])
def test_prepass_rejects_bad_arguments(lib, over, needle):
    rc = lib.sage_prepass(*_prepass_args(**over))
    msg = lib.sage_last_error().decode()
    assert rc != 0 and "invalid argument" in msg and needle in msg, msg


@pytest.mark.parametrize("over,vt_over,needle", [
    ({}, dict(pv=7), "pv_mode"),
    ({}, dict(pv=2), "FP8 V tiles need v_mode"),          # FP8 tiles without v_scale
    ({}, dict(vt=None), "null pointer"),
    (dict(v=None), {}, "null V pointer"),
    ({}, dict(vtb=1000), "vtiles"),                       # 1000 < 2*64*64*2 bytes
    ({}, dict(vt=ctypes.c_void_p(24)), "aligned"),
    (dict(q_sub=2), {}, "q_sub"),                         # the pre-pass's own checks still apply
])
def test_prepass_vt_rejects_bad_arguments(lib, over, vt_over, needle):
    s3 = (ctypes.c_int64 * 3)(0, 0, 0)
    base = dict(v=ctypes.c_void_p(16), vs=s3)
    base.update(over)
    tail = dict(pv=0, vt=ctypes.c_void_p(16), vtb=1 << 20, st=None)
    tail.update(vt_over)
    args = _prepass_args(**base)[:-1] + list(tail.values())
    rc = lib.sage_prepass_vt(*args)
    msg = lib.sage_last_error().decode()
    assert rc != 0 and "invalid argument" in msg and needle in msg and "sage_prepass_vt" in msg, msg


def test_attn_rejects_bad_arguments(lib):
    s3 = (ctypes.c_int64 * 3)(0, 0, 0)
    p = ctypes.c_void_p(16)
    rc = lib.sage_attn_fwd(p, s3, p, p, s3, p, p, 2, s3, None, p, 2, s3, 1, 2, 2, 64, 64, 64, 0, 128, 32, 128, 0,
                           None)
    assert rc != 0 and "blkk" in lib.sage_last_error().decode()
    rc = lib.sage_attn_fwd(p, s3, p, p, s3, p, p, 2, s3, None, p, 1, s3, 1, 2, 2, 64, 64, 64, 0, 128, 64, 128, 0,
                           None)
    assert rc != 0 and "v_dtype" in lib.sage_last_error().decode()


def test_vtile_bytes_and_rejections(lib):
    # tiles of 64 keys (ragged N rounded up), 2 bytes per element for fp16/bf16, 1 for e4m3
    assert lib.sage_vtile_bytes(4, 32, 4096, 128, 0) == 4 * 32 * 64 * 128 * 64 * 2
    assert lib.sage_vtile_bytes(2, 8, 17776, 64, 1) == 2 * 8 * 278 * 64 * 64 * 2
    assert lib.sage_vtile_bytes(1, 32, 32768, 128, 2) == 32 * 512 * 128 * 64
    assert lib.sage_prepass_workspace_bytes(4, 32, 4096, 128, 0, 2) == 4 * 32 * 16 * 128 * 4
    s3 = (ctypes.c_int64 * 3)(0, 0, 0)
    p = ctypes.c_void_p(16)
    big = ctypes.c_size_t(1 << 40)
    for args, needle in [
        ((p, 2, 1, 2, 64, 96, s3, 0, None, p, big, None), "head_dim"),
        ((p, 2, 1, 2, 64, 64, s3, 2, None, p, big, None), "null"),
        ((p, 2, 1, 2, 64, 64, s3, 5, None, p, big, None), "pv_mode"),
        ((p, 2, 1, 2, 64, 64, s3, 0, None, p, ctypes.c_size_t(64), None), "out"),
    ]:
        rc = lib.sage_vtiles(*args)
        msg = lib.sage_last_error().decode()
        assert rc != 0 and "invalid argument" in msg and needle in msg, msg


def test_library_override_must_exist(hip_impl, monkeypatch, tmp_path):
    """$TRIBENCH_SAGE_HIP_LIB naming no file is an error, not a silent fall
    back to the in-tree library; naming a file selects it."""
    missing = tmp_path / "no_such_lib.so"
    monkeypatch.setenv("TRIBENCH_SAGE_HIP_LIB", str(missing))
    with pytest.raises(RuntimeError, match="is not a file"):
        hip_impl.library_path()
    monkeypatch.delenv("TRIBENCH_SAGE_HIP_LIB")
    default = hip_impl.library_path()
    monkeypatch.setenv("TRIBENCH_SAGE_HIP_LIB", str(default))
    assert hip_impl.library_path() == default


def test_hip_variant_refuses_cpu_tensors(hip_impl):
    import torch

    q = torch.zeros(1, 2, 16, 64)
    with pytest.raises(RuntimeError, match="ROCm GPU device"):
        hip_impl.run(q, q, q)


def test_flash_rejects_bad_arguments(lib):
    s3 = (ctypes.c_int64 * 3)(0, 0, 0)
    p = ctypes.c_void_p(16)
    for args, needle in [
        ((p, s3, p, s3, p, 4, None, p, s3, 1, 1, 2, 2, 64, 64, 96, 0.18, 0, None), "head_dim"),
        ((p, s3, p, s3, p, 4, None, p, s3, 0, 1, 2, 2, 64, 64, 64, 0.18, 0, None), "in_dtype"),
        ((p, s3, p, s3, p, 2, None, p, s3, 2, 1, 2, 2, 64, 64, 64, 0.18, 0, None), "v_dtype"),
        ((p, s3, p, s3, p, 4, None, p, s3, 2, 1, 3, 2, 64, 64, 64, 0.18, 0, None), "Hq"),
        ((p, s3, p, s3, p, 4, None, p, s3, 2, 1, 2, 2, 64, 64, 64, 0.0, 0, None), "qk_mul"),
        ((None, s3, p, s3, p, 4, None, p, s3, 2, 1, 2, 2, 64, 64, 64, 0.18, 0, None), "null"),
        ((ctypes.c_void_p(8), s3, p, s3, p, 4, None, p, s3, 2, 1, 2, 2, 64, 64, 64, 0.18, 0, None), "aligned"),
    ]:
        rc = lib.sage_flash_fwd(*args)
        msg = lib.sage_last_error().decode()
        assert rc != 0 and "invalid argument" in msg and needle in msg, msg


def test_attn_fwd_q_rejects_bad_arguments(lib):
    s3 = (ctypes.c_int64 * 3)(0, 0, 0)
    p = ctypes.c_void_p(16)
    base = dict(q=p, qs=s3, qdt=2, qmul=0.18, q8o=None, qso=None, k8=p, k8s=s3, ksc=p, v=p, vdt=4, vs=None,
                vsc=None, o=p, os=s3, B=1, Hq=2, Hkv=2, Nq=64, Nkv=64, D=64, causal=0, blkq=128, blkk=64,
                q_sub=128, pv=0, st=None)
    for over, needle in [
        (dict(blkq=64, q_sub=64), "blkq"),
        (dict(q_sub=48), "q_sub"),
        (dict(q_sub=2), "q_sub"),
        (dict(qdt=9), "q_dtype"),
        (dict(qmul=-1.0), "q_mul"),
        (dict(vdt=2), "v_dtype"),
        (dict(q=None), "null"),
        (dict(D=96), "head_dim"),
        (dict(q8o=ctypes.c_void_p(8)), "aligned"),
    ]:
        a = dict(base)
        a.update(over)
        rc = lib.sage_attn_fwd_q(*a.values())
        msg = lib.sage_last_error().decode()
        assert rc != 0 and "invalid argument" in msg and needle in msg, msg


def _sage_call(hip_impl, **over):
    """A packed sage_call of one 64-row head; every buffer at address 256."""
    c = dict(B=1, Hq=1, Hkv=1, Nq=64, Nkv=64, D=128, mul=0.1, dtype=2, fuse_q=-1, q_row=128, ws=1 << 40)
    c.update(over)
    rows = [64 * 128, 64 * 128, 128]
    return hip_impl._CALL.pack(hip_impl._CALL_SIZE, 256, 256, 256, 256, 256, c["ws"], rows[0], rows[1], c["q_row"],
                               *rows, *rows, *rows, c["B"], c["Hq"], c["Hkv"], c["Nq"], c["Nkv"], c["D"], c["mul"],
                               c["dtype"], 0, 0, 128, 1, c["fuse_q"], *hip_impl._NO_OUTS)


@pytest.mark.parametrize("Hq", [1, 512])  # by size, Q is quantized in the pre-pass or in the prologue
def test_sage_run_limits_do_not_depend_on_the_shape(lib, hip_impl, Hq):
    import torch

    for over, needle in [
        (dict(mul=0.0), "mul"),
        (dict(mul=-1.0), "mul"),
        (dict(mul=float("inf")), "mul"),
        (dict(mul=-1.0, D=64, fuse_q=1), "mul"),
        (dict(q_row=1 << 25), "2^31 bytes"),
    ]:
        assert lib.sage_run(_sage_call(hip_impl, Hq=Hq, **over), None) != 0
        msg = lib.sage_last_error().decode()
        assert "invalid argument" in msg and needle in msg, msg
    if torch.cuda.is_available():  # what is not refused would launch on these addresses
        return
    for over in [dict(mul=-1.0, D=64), dict(mul=-1.0, fuse_q=0), dict(q_row=1 << 25, D=64)]:
        assert lib.sage_run(_sage_call(hip_impl, Hq=Hq, **over), None) != 0  # no device: the launch fails
        msg = lib.sage_last_error().decode()
        assert "invalid argument" not in msg, msg


@pytest.mark.parametrize("pack", ["sage_attn", "flash_attn"])
def test_packs_load_on_a_torch_without_a_gpu_backend(pack, hip_impl, monkeypatch):
    """Such a build has no raw stream query; the packs load and the call names
    the missing device."""
    import importlib.util

    import torch

    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    path = ROOT / "tribench_amd" / "kernels" / pack / "hip_impl.py"
    spec = importlib.util.spec_from_file_location(f"no_backend_{pack}", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    q = torch.zeros(1, 2, 16, 64, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="ROCm GPU device"):
        mod.run(q, q, q)


def test_run_header_declares_what_the_binding_calls(lib):
    counts = _declared_arg_counts(RUN_HEADER)
    assert sorted(counts) == _declared_functions(RUN_HEADER) == [
        "sage_flash_run", "sage_flash_run_workspace_bytes", "sage_run", "sage_run_stages", "sage_run_workspace_bytes"]
    for name, n in counts.items():
        assert len(getattr(lib, name).argtypes) == n, name


def test_sage_call_layout_matches_the_header(hip_impl, tmp_path):
    """The binding packs sage_call field by field where the C compiler puts them."""
    text = re.sub(r"/\*.*?\*/", "", RUN_HEADER.read_text(), flags=re.S)
    body = re.search(r"typedef struct sage_call \{(.*?)\} sage_call;", text, flags=re.S).group(1)
    fields = []  # (name, struct code, count)
    for ctype, names in re.findall(r"(const void\s*\*|void\s*\*|int64_t|double)\s*([^;]+);", body):
        for name in names.split(","):
            m = re.fullmatch(r"\s*(\w+)(?:\[(\d+)\])?\s*", name)
            fields.append((m.group(1), "P" if "*" in ctype else {"int64_t": "q", "double": "d"}[ctype],
                           int(m.group(2) or 1)))
    assert "".join(code * n for _, code, n in fields) == "".join(
        code * int(n or 1) for n, code in re.findall(r"(\d*)([qPd])", hip_impl._CALL.format))
    src = tmp_path / "layout.c"
    src.write_text('#include <stddef.h>\n#include <stdio.h>\n#include "sage_attn_run.h"\nint main(void) {\n'
                   + "".join(f'  printf("%zu\\n", offsetof(sage_call, {name}));\n' for name, _, _ in fields)
                   + '  printf("%zu\\n", sizeof(sage_call));\n  return 0;\n}\n')
    exe = tmp_path / "layout"
    subprocess.run(["gcc", f"-I{RUN_HEADER.parent}", "-o", str(exe), str(src)], check=True)
    got = [int(x) for x in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]
    want, at = [], 0
    for _, _, n in fields:
        want.append(at)
        at += 8 * n
    assert got == want + [hip_impl._CALL_SIZE]
    assert dict(zip((f[0] for f in fields), got))["workspace"] == hip_impl._CALL_WS_AT


def test_a_library_without_the_whole_call_is_refused_by_version(monkeypatch, tmp_path):
    """A library of the ABI before sage_attn_run.h is told to rebuild, not
    tripped over by its missing symbols."""
    import importlib.util

    src, so = tmp_path / "old.c", tmp_path / "old.so"
    src.write_text("int sage_abi_version(void) { return 6; }\n"
                   + "".join(f"void {n}(void) {{}}\n" for n in _declared_functions() if n != "sage_abi_version"))
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    monkeypatch.setenv("TRIBENCH_SAGE_HIP_LIB", str(so))
    spec = importlib.util.spec_from_file_location("old_lib_impl", ROOT / "tribench_amd" / "kernels" / "sage_attn" /
                                                  "hip_impl.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    with pytest.raises(RuntimeError, match="ABI 6.*rebuild"):
        mod._load()
