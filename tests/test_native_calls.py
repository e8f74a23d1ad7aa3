"""The compiled launch calls of reinstinct_amd.runtime: what they take as arguments and how they fail (CPU: every call here is
refused by the library's or the wrapper's own checks)."""
import ctypes as C
import inspect

import pytest

import reinstinct_amd as rein
from reinstinct_amd import runtime


class Buf:
    _as_parameter_ = 64


@pytest.mark.parametrize("x", [64, True, None, Buf(), C.c_void_p(64)])
def test_pointer_arguments(x):
    with pytest.raises(rein.ReinError) as e:                  # in_dim 31: the shape is checked before any pointer is used
        runtime.quantize_q8(x, 64, 31)
    assert e.value.code == -3
    with pytest.raises(rein.ReinError) as e:
        runtime.quantize_q8(x, xq=64, in_dim=31, n_vec=2, stream=x)
    assert e.value.code == -3


def test_wrong_arguments():
    for call in (lambda: runtime.quantize_q8(1.5, 64, 32), lambda: runtime.quantize_q8(64, 64, "32"), lambda: runtime.quantize_q8(64, 64),
                 lambda: runtime.quantize_q8(64, 64, 32, 1, None, 0), lambda: runtime.quantize_q8(64, 64, 32, x=64),
                 lambda: runtime.quantize_q8(64, 64, 32, rows=1), lambda: runtime.add_rmsnorm_q8(64, None, 64, None, 64, 32, 1, "eps"),
                 lambda: runtime.moe_ffn(b"short", 64, 64, 64, 64, 64, 64, 64, 64)):
        with pytest.raises(TypeError):
            call()


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
