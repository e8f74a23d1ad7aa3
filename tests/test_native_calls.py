"""The compiled launch calls of reinstinct_amd.runtime: what they take as arguments and how they fail (CPU: every call here is
refused by the library's or the wrapper's own checks)."""
import ctypes as C
import inspect
import json
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip, runtime

PKG = os.path.dirname(os.path.abspath(rein.__file__))


class Buf:
    _as_parameter_ = 64


@pytest.mark.parametrize("x", [64, True, None, Buf(), C.c_void_p(64)])
def test_pointer_arguments(x):
    with pytest.raises(rein.ReinError) as e:                  # in_dim 31: the shape is checked before any pointer is used
        runtime.quantize_q8(x, 64, 31)
    assert e.value.code == -3
    with pytest.raises(rein.ReinError) as e:
        runtime.quantize_q8(x, xq=64, in_dim=31, n_vec=2, stream=None)
    assert e.value.code == -3


class OnStream:
    raw = 64


@pytest.mark.parametrize("call", [lambda s: runtime.quantize_q8(64, 64, 31, 1, s), lambda s: runtime.quantize_q8(64, 64, 31, stream=s),
                                  lambda s: runtime.matvec_multi_xq8([12], [64], [64], [32], 64, 255, 1, s),
                                  lambda s: runtime.moe_ffn(runtime.moe_shape(0, 256, 8, 2, 256, 12, 12), 64, 64, 64, 64, 64, 64, 64, 64, s)])
def test_a_stream_is_a_stream(call):
    """None or an object whose `raw` is the handle; a number, a pointer or a buffer in its place is a mistake"""
    for stream in (None, OnStream()):
        with pytest.raises(rein.ReinError) as e:
            call(stream)
        assert e.value.code == -3
    for stream in (64, True, Buf(), C.c_void_p(64), "s"):
        with pytest.raises(TypeError):
            call(stream)


def test_a_stream_is_no_pointer():
    with pytest.raises(TypeError):
        runtime.quantize_q8(hip.Stream.__new__(hip.Stream), 64, 31)


def test_wrong_arguments():
    for call in (lambda: runtime.quantize_q8(1.5, 64, 32), lambda: runtime.quantize_q8(64, 64, "32"), lambda: runtime.quantize_q8(64, 64),
                 lambda: runtime.quantize_q8(64, 64, 32, 1, None, 0), lambda: runtime.quantize_q8(64, 64, 32, x=64),
                 lambda: runtime.quantize_q8(64, 64, 32, rows=1), lambda: runtime.add_rmsnorm_q8(64, None, 64, None, 64, 32, 1, "eps"),
                 lambda: runtime.moe_ffn(b"short", 64, 64, 64, 64, 64, 64, 64, 64)):
        with pytest.raises(TypeError):
            call()


class Four:
    def __index__(self):
        return 4


COUNTS = (32, True, np.int64(32), np.uint8(32), Four(), C.c_uint(32))
POINTERS = (64, None, Buf(), C.c_void_p(64), C.c_void_p(None), C.create_string_buffer(64), C.pointer(C.c_int(1)), C.byref(C.c_int(1)), b"host", C.c_char_p(b"host"))
NUMBERS = (1e-6, 1, np.float32(1e-6), np.int32(1), C.c_float(1e-6))
NEITHER = (1.5, "32", C.c_int(32), C.c_long(32), C.c_float(1.0), [32], object(), np.float32(4.0), np.zeros(4))


@pytest.mark.parametrize("o", [*COUNTS, *POINTERS, *NUMBERS, *NEITHER], ids=repr)
def test_arguments_are_those_of_ctypes(o):
    """what ctypes takes for an unsigned, a pointer and a float parameter is taken, what it refuses is refused"""
    def taken(ctype):
        try:
            ctype.from_param(o)
            return True
        except (TypeError, C.ArgumentError):
            return False

    def called(call):
        try:
            call()
        except rein.ReinError:                                # the library's own refusal: every argument was converted
            return True
        except TypeError:
            return False

    assert called(lambda: runtime.quantize_q8(64, 64, 31, o)) == taken(C.c_uint)
    assert called(lambda: runtime.quantize_q8(o, 64, 31)) == taken(C.c_void_p)
    assert called(lambda: runtime.rmsnorm_q8(64, 64, 64, 31, 1, o)) == taken(C.c_float)
    assert called(lambda: runtime.matmul_ws(12, 64, 64, 64, 31, 32, 40, 64, o)) == taken(C.c_size_t)
    assert called(lambda: runtime.matvec_xq8(o, 64, 64, 64, 0, 32)) == taken(C.c_int)


def test_the_shape_of_moe_ffn():
    with pytest.raises(TypeError):
        runtime.moe_ffn(bytes(C.sizeof(runtime.MoeShape)), 64, 64, 64, 64, 64, 64, 64, 64)


def test_multi_tables():
    with pytest.raises(rein.ReinError) as e:                  # five matrices: refused by the library
        runtime.matvec_multi_xq8([12] * 5, [64] * 5, [64] * 5, [32] * 5, 64, 256)
    assert e.value.code == -3
    with pytest.raises(ValueError):
        runtime.matvec_multi_xq8([12, 12], [64], [64, 64], [32, 32], 64, 256)
    with pytest.raises(rein.ReinError) as e:
        runtime.matvec_multi_xq8((12, 12), (Buf(), 64), [64, 64], [32, 32], Buf(), 255)
    assert e.value.code == -3


def test_signatures_are_visible():
    assert str(inspect.signature(runtime.rmsnorm_q8)) == "(x, w, xq, n, n_vec=1, eps=1e-06, stream=None)"
    assert "quantize_q8" in runtime.quantize_q8.__doc__


def child(code, root):
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120, cwd=root,
                          env=dict(os.environ, PYTHONPATH=str(root)))


def package(root, *built):
    """a copy of the package's Python files, with these of the built ones"""
    there = root / "reinstinct_amd"
    there.mkdir()
    for f in os.listdir(PKG):
        if f.endswith(".py") or f in built:
            os.symlink(os.path.join(PKG, f), there / f)
    return root


def test_import_and_calls_without_anything_built(tmp_path):
    run = child("from reinstinct_amd import runtime, hip, quant, gguf, ReinError\n"
                "try: runtime.quantize_q8(64, 64, 32)\n"
                "except ReinError as e: print(e.code, e)\n", package(tmp_path))
    assert run.returncode == 0, run.stderr
    assert run.stdout.startswith("-1 ") and "librein.so is not built" in run.stdout


def test_the_extension_is_the_one_in_use():
    assert inspect.isbuiltin(runtime.quantize_q8) and inspect.isbuiltin(runtime.moe_ffn)


def test_calls_by_ctypes_are_the_same(tmp_path):
    """without the compiled extension: every launch call is there, with its parameters and defaults, and reaches the library"""
    names = [n for n in dir(runtime) if inspect.isbuiltin(getattr(runtime, n))]
    assert len(names) == 32
    run = child("import inspect, json\n"
                "from reinstinct_amd import runtime, ReinError\n"
                f"names = {names!r}\n"
                "assert not any(inspect.isbuiltin(getattr(runtime, n)) for n in names)\n"
                "codes = []\n"
                "for call in (lambda: runtime.quantize_q8(64, 64, 31), lambda: runtime.matvec_multi_xq8([12] * 5, [64] * 5, [64] * 5, [32] * 5, 64, 256),\n"
                "             lambda: runtime.moe_ffn(runtime.moe_shape(0, 256, 8, 2, 256, 12, 12), 64, 64, 64, 64, 64, 64, 256, 64),\n"
                "             lambda: runtime.matmul_ws(12, 64, 64, 64, 256, 32, 40, 64, n_scratch)):\n"
                "    n_scratch = 8\n"
                "    try: call()\n"
                "    except ReinError as e: codes.append(e.code)\n"
                "print(json.dumps([codes, [str(inspect.signature(getattr(runtime, n))) for n in names]]))\n", package(tmp_path, "librein.so"))
    assert run.returncode == 0, run.stderr
    codes, signatures = json.loads(run.stdout)
    assert codes == [-3, -3, -3, -3]
    assert signatures == [str(inspect.signature(getattr(runtime, n))) for n in names]


@pytest.mark.skipif(shutil.which("make") is None, reason="no make")
def test_the_library_builds_without_pythons_headers(tmp_path):
    csrc = os.path.join(PKG, "csrc")
    for setting in (f"PY_INC={tmp_path}", "PYTHON=/nonexistent/python"):
        plan = subprocess.run(["make", "-n", "-B", "-C", csrc, setting], capture_output=True, text=True)
        assert plan.returncode == 0, plan.stderr
        assert "rein_api.cpp" in plan.stdout and "rein_kernels.hip" in plan.stdout and "native.cpp" not in plan.stdout
