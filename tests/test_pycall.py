"""The native launch calls of btf_hip.py (csrc/pycall.c) hand the C ABI the
same arguments as its ctypes path, over the forms that they read; every other
form is left to the ctypes path. Host only: the calls are bound to recording
callbacks instead of the launchers."""
import ctypes as C
import os
import shutil
import subprocess
import sys
import types

import numpy as np
import pytest
import torch

import btf_hip as hip

native = pytest.mark.skipif(not os.path.exists(hip.CALL_PATH), reason="native launch calls not built")
vp = C.c_void_p
Q8P, HXP, SEGP = C.POINTER(hip._Q8Act), C.POINTER(hip._Hx), C.POINTER(hip._GemvSeg)
ARGS = {"prep": [vp, C.c_int, C.c_int, C.c_int, vp, C.c_float, HXP, vp, C.c_int, Q8P, vp],
        "gemv": [SEGP, C.c_int, C.c_int, C.c_int, Q8P, C.c_int, vp],
        "gemv_ptq1_0": [SEGP, C.c_int, C.c_int, C.c_int, Q8P, C.c_int, vp],
        "gemv_ex": [SEGP, C.c_int, C.c_int, C.c_int, Q8P, vp, C.c_int, C.c_int, Q8P, vp]}


def plain(v, nseg):
    if isinstance(v, SEGP):
        return [plain(v[i], 0) for i in range(nseg)]
    if isinstance(v, (Q8P, HXP)):
        return plain(v[0], 0) if v else None
    if isinstance(v, C.Structure):
        return tuple(getattr(v, f) for f, _ in v._fields_)
    return v


@pytest.fixture
def seen():
    """The native calls bound to recorders: seen[-1] = (name, arguments)."""
    got, keep = [], []

    def recorder(name):
        def f(*a):
            nseg = a[1] if name != "prep" else 0
            got.append((name, [plain(v, nseg) for v in a]))
            return 0
        keep.append(C.CFUNCTYPE(C.c_int, *ARGS[name])(f))
        return C.cast(keep[-1], vp).value
    hip._call.bind(*[recorder(n) for n in ("prep", "gemv", "gemv_ptq1_0", "gemv_ex")], hip.Q8Act, hip.Hx, hip.GemvSeg)
    yield got
    hip._call.bind(*[C.cast(f, vp).value for f in (hip._launch_prep, hip._launch_gemv, hip._launch_gemv_ptq1_0,
                                                   hip._launch_gemv_ex)], hip.Q8Act, hip.Hx, hip.GemvSeg)


T = [torch.zeros(8 + i) for i in range(8)]
ACTS = [hip.Q8Act(T[0], T[1], T[2]), hip.Q8Act(16, None, T[2]), hip.Q8Act()]
STREAMS = [None, 0, 1 << 45, types.SimpleNamespace(cuda_stream=77)]


@native
@pytest.mark.parametrize("stream", STREAMS, ids=str)
@pytest.mark.parametrize("a", ACTS, ids=["tensors", "mixed", "empty"])
@pytest.mark.parametrize("hx", [None, hip.Hx(), hip.Hx(1024, 32, 2, 4, T[5]), hip.Hx(block=64, signs=4096)],
                         ids=["none", "zero", "perm", "address"])
def test_prep_arguments(seen, stream, a, hx):
    hip.launch_prep(T[3], 5120, -1, 1 << 30, T[4], 1e-6, hx, None, True, a, stream)
    name, v = seen[-1]
    h = (hx or hip.Hx())._c()
    assert name == "prep"
    assert v == [T[3].data_ptr(), 5120, -1, 1 << 30, T[4].data_ptr(), C.c_float(1e-6).value, plain(h, 0), None, 1,
                 plain(a._c(), 0), hip._stream(stream) or None]


@native
@pytest.mark.parametrize("stream", STREAMS, ids=str)
@pytest.mark.parametrize("nseg", [1, 2, 3])
@pytest.mark.parametrize("kind", [list, tuple])
def test_gemv_arguments(seen, stream, nseg, kind):
    segs = kind([hip.GemvSeg(T[0], T[1], 5, T[2], 7), hip.GemvSeg(64, None, 6), hip.GemvSeg()][:nseg])
    want = [plain(s._c(), 0) for s in segs]
    st = hip._stream(stream) or None
    for f, name in ((hip.launch_gemv, "gemv"), (hip.launch_gemv_ptq1_0, "gemv_ptq1_0")):
        for mode in (hip.GemvMode.kSwiglu, 1):
            f(segs, 128, 3, ACTS[0], mode, stream)
            assert seen[-1] == (name, [want, nseg, 128, 3, plain(ACTS[0]._c(), 0), int(mode), st])
    for a, x, out in ((ACTS[0], None, None), (None, T[6], ACTS[1]), (None, 256, None)):
        hip.launch_gemv_ex(segs, 128, 3, a, x, 9, hip.GemvMode.kAdd, out, stream)
        assert seen[-1] == ("gemv_ex", [want, nseg, 128, 3, a and plain(a._c(), 0), hip._addr(x), 9, 1,
                                        out and plain(out._c(), 0), st])


class SubAct(hip.Q8Act):
    pass


def test_other_forms_take_the_ctypes_path(seen):
    """Forms that the native calls do not read reach the library itself
    (here: its argument checks, or ctypes' own refusals), never the recorder."""
    S, A = [hip.GemvSeg(T[0], T[1], 5, T[2], 7)], ACTS[0]
    for args in [([], 128, 3, A, 0), (S * 4, 128, 3, A, 0), (S, 127, 3, SubAct(16, 16, 16), 0)]:
        with pytest.raises(RuntimeError):
            hip.launch_gemv(*args)
    hip.launch_gemv(S, np.int64(128), 0, A, 0)  # no rows: nothing to do
    with pytest.raises(C.ArgumentError):
        hip.launch_gemv(S, 128.0, 0, A, 0)
    hip.launch_prep(T[3], 8, 0, 8, None, np.float64(1e-6), None, None, 0, A)
    with pytest.raises(AttributeError):
        hip.launch_prep(np.zeros(8), 8, 0, 8, None, 0.0, None, None, 0, A)
    with pytest.raises(AttributeError):
        hip.launch_gemv(S, 128, 3, A, 0, object())
    assert not seen


def test_errors_raise_the_library_message():
    with pytest.raises(RuntimeError, match="multiple of 128"):
        hip.launch_gemv([hip.GemvSeg(T[0], T[1], 5, T[2], 7)], 100, 1, ACTS[0])
    with pytest.raises(RuntimeError, match="multiple of 32"):
        hip.launch_prep(T[3], 33, 1, 33, None, 0.0, None, None, 0, ACTS[0])


def test_bindings_work_without_the_native_calls(tmp_path):
    """A tree with the library alone imports, and its launches take the ctypes
    path; native calls built for another Python are not loaded."""
    shutil.copy(os.path.join(hip.HERE, "btf_hip.py"), tmp_path)
    os.symlink(hip.LIB_PATH, tmp_path / "libbtf_hip.so")
    for name in ("_btf_call.so", "_btf_call.cpython-39-x86_64-linux-gnu.so"):
        (tmp_path / name).write_bytes(b"not for this Python")
    code = """
import btf_hip as h
for f in (lambda: h.launch_prep(16, 33, 1, 33, None, 0.0, None, None, 0, h.Q8Act(16, 16, 16)),
          lambda: h.launch_gemv([h.GemvSeg(16, 16, 5, 16, 5)], 100, 1, h.Q8Act(16, 16, 16)),
          lambda: h.launch_gemv_ptq1_0([h.GemvSeg(16, None, 5, 16, 5)], 100, 1, h.Q8Act(16, 16, 16)),
          lambda: h.launch_gemv_ex([h.GemvSeg(16, 16, 5, 16, 5)], 100, 1, h.Q8Act(16, 16, 16))):
    try:
        f()
    except RuntimeError as e:
        print(e)
"""
    out = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    assert out.stdout.count("multiple of") == 4, out.stdout


def test_library_builds_without_python():
    """`make` needs neither a Python nor its headers for the library itself."""
    def targets(*args):
        out = subprocess.run(["make", "-n", "-B", "-C", hip.HERE, "all", *args], capture_output=True, text=True)
        assert out.returncode == 0, out.stderr
        return out.stdout
    assert "pycall.c" not in targets("PYTHON=/nonexistent/python3")
    assert "pycall.c" not in targets("CC=/nonexistent/cc")
    assert "libbtf_hip.so" in targets("PYTHON=/nonexistent/python3")
    if os.path.exists(hip.CALL_PATH):
        assert os.path.basename(hip.CALL_PATH) in targets(f"PYTHON={sys.executable}")
