"""The tensor checks of k3h.py's typed calls (extension _k3h_py): what a kernel argument is
rejected for, on the CPU where the device decides first and on the GPU for the rest, and
that a call runs on the stream current at that moment."""
import importlib.util
import os
import shutil
import subprocess
import sys

import pytest
import torch

import k3h

PKG = os.path.dirname(os.path.abspath(k3h.__file__))


def test_rejects_host_tensors_and_other_objects():
    t = torch.zeros(64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match=r"x: must be a GPU tensor \(got cpu\)"):
        k3h._dev(t, "x", k3h.BF16, 64)
    for bad in (3, None, [t]):
        with pytest.raises(ValueError, match="x: expected a torch tensor"):
            k3h._dev(bad, "x", k3h.BF16)
    for args, kw in (((t, "x"), {}), ((t, "x", k3h.BF16, 1, 16, 1), {}), ((t, "x", k3h.BF16), {"size": 1}),
                     ((t, "x", "bf16"), {}), ((t, "x", k3h.BF16, 1.5), {})):
        with pytest.raises(TypeError):
            k3h._dev(*args, **kw)
    assert k3h._ptr(None) is None and k3h._ptr(t) == t.data_ptr()
    with pytest.raises(ValueError):
        k3h._ptr(3)


def test_import_without_a_build(tmp_path):
    """k3h.py imports where nothing is built; what needs the library or the extension names
    the missing file, and the extension is picked up once it is there."""
    shutil.copy(os.path.join(PKG, "k3h.py"), tmp_path)
    code = f"""
import os, shutil
import k3h, torch
assert os.path.dirname(os.path.abspath(k3h.__file__)) == {str(tmp_path)!r}
assert k3h.pack_args(["i32"], [3]) == b"\\x03\\x00\\x00\\x00"
for call in (k3h.Ctx, lambda: k3h._ptr(None), lambda: k3h._dev(torch.zeros(1), "x", k3h.F32)):
    try:
        call()
    except FileNotFoundError as e:
        assert "build.py" in str(e)
    else:
        raise SystemExit("no error without a build")
os.makedirs(k3h.BUILD)
shutil.copy({os.path.join(k3h.BUILD, "_k3h_py.so")!r}, k3h.BUILD)
assert k3h._ptr(None) is None
try:
    k3h._dev(torch.zeros(1), "x", k3h.F32)
except ValueError as e:
    assert "must be a GPU tensor" in str(e)
"""
    env = dict(os.environ, PYTHONPATH=str(tmp_path))
    r = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, env=env, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_library_builds_without_torch_headers(tmp_path, monkeypatch):
    """The code objects and libk3h.so need no torch: `only=` leaves the extension alone, and a
    whole build does without it where torch's C++ headers are missing."""
    spec = importlib.util.spec_from_file_location("k3_build_headers", os.path.join(PKG, "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    from torch.utils import cpp_extension
    monkeypatch.setattr(b, "OUT", str(tmp_path))
    monkeypatch.setattr(b, "MODULES", ["k3h_fused"])
    ran = []
    monkeypatch.setattr(b, "_run", lambda cmd, what: (ran.append(what), open(cmd[cmd.index("-o") + 1], "w").close()))
    b.build(only=["k3h_fused"], oracle=False)
    assert sorted(ran) == ["k3h_fused", "libk3h.so"]
    ran.clear()
    monkeypatch.setattr(cpp_extension, "include_paths", lambda *a, **k: [str(tmp_path)])
    b.build(oracle=False)
    assert sorted(ran) == ["k3h_fused", "libk3h.so"]


@pytest.mark.gpu
def test_rejects_wrong_gpu_tensors():
    t = torch.zeros(64, 2, dtype=torch.bfloat16, device="cuda")
    assert k3h._dev(t, "x", k3h.BF16, 128) is None
    assert k3h._dev(t, "x", k3h.BF16 + k3h.F32, numel=1, align=2) is None
    assert k3h._dev(t[1:], "x", k3h.BF16, align=4) is None
    assert k3h._dev(t.view(torch.uint8).view(torch.float8_e4m3fn), "x", k3h.U8) is None
    assert k3h._dev(t, "x", k3h.ANY) is None
    for bad, mask, numel, align, why in (
            (t, k3h.F32, 1, 16, r"dtype torch.bfloat16 not in \[torch.float32\]"),
            (t, k3h.I32 + k3h.I64, 1, 16, r"not in \[torch.int32, torch.int64\]"),
            (t.t(), k3h.BF16, 1, 16, "must be contiguous"),
            (t, k3h.BF16, 129, 16, "needs at least 129 elements, has 128"),
            (t[1:], k3h.BF16, 1, 16, "must be 16-byte aligned")):
        with pytest.raises(ValueError, match="x: .*" + why):
            k3h._dev(bad, "x", mask, numel, align)


@pytest.mark.gpu
def test_default_stream_is_the_current_one(ctx):
    assert k3h._stream(None) == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert k3h._stream(None) == s.cuda_stream
    assert k3h._stream(s) == s.cuda_stream and k3h._stream(7) == 7
