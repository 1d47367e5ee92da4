"""The extension between the Python modules and the C ABI (csrc/host.cpp): what it takes as an argument, what it refuses, and that
the library sees the same values as through ctypes.  No launch: every call is refused by the library's own checks."""
import ctypes as C

import numpy as np
import pytest
import torch

from ml import _lib as L


def refused(fn, *args):
    """Status and message of a call, through `fn` of the extension's functions or of ctypes."""
    rc = fn(*args)
    return rc, L.lib.sp_last_error_string().decode()


P = 0x6000


@pytest.mark.parametrize("w", [[P, P], (P, None), [C.c_void_p(P), P + 4], (C.c_void_p * 2)(P, P), None])
@pytest.mark.parametrize("dims", [[32, 64, 65], (C.c_int32 * 3)(32, 64, 65), (32, 60, 3), [32, 64, 3], None])
@pytest.mark.parametrize("x", [P, C.c_void_p(P), P + 8, None])
def test_calls_reach_the_library_as_through_ctypes(w, dims, x):
    as_array = lambda v, t: v if v is None or isinstance(v, C.Array) else (t * len(v))(*v)
    rest = (None, None, P, None, None, 16, 1, 5, None)      # a mask wider than a head of 3
    mine = refused(L.lib.sp_mlp_forward, 1, x, 2, w, None, dims, *rest)
    theirs = refused(L.lib._cdll.sp_mlp_forward, 1, x, 2, as_array(w, C.c_void_p), None, as_array(dims, C.c_int32), *rest)
    assert mine == theirs and mine[0] < 0


def test_structures_and_numbers():
    ph = L.PhiloxConfig(1, 0, 17, 256, 24, 0, 0, 0)          # no such mode
    for given in (ph, C.byref(ph)):
        assert refused(L.lib.sp_row_sample, L.ROW_SOFTMAX, P, None, given, None, None, None, P, None, 8, 64, 0, None)[0] == -5
    assert refused(L.lib.sp_map_f32, 1, P, P, -(1 << 40), None)[0] == -2                 # 64 bits arrive whole
    for wrong in ((1, P, P, 4), (1, P, P, 4.5, None), (1, P, P, "4", None), (1, "P", P, 4, None), (1, object(), P, 4, None),
                  (1, bytearray(8), P, 4, None), (1, np.zeros(2), P, 4, None), (1, torch.zeros(2), P, 4, None)):
        with pytest.raises(TypeError):
            L.lib.sp_map_f32(*wrong)
    for layers in (8, 16, 17, 40):                           # more than a stack may have
        assert refused(L.lib.sp_mlp_forward, 1, P, layers, [P] * layers, None, [32] * layers + [65], None, None, P, None, None, 16, 1, 0, None) == refused(
            L.lib._cdll.sp_mlp_forward, 1, P, layers, (C.c_void_p * layers)(*[P] * layers), None, (C.c_int32 * (layers + 1))(*[32] * layers, 65), None, None, P,
            None, None, 16, 1, 0, None)


def test_pointers_of_tensors():
    assert L.ptr(None) is None and L.ptr(None, torch.float32, "x") is None
    with pytest.raises(TypeError, match="x must be a torch.Tensor"):
        L.ptr(3, name="x")
    with pytest.raises(ValueError, match=r"x must live on the GPU \(got cpu\)"):
        L.ptr(torch.zeros(3), torch.float32, "x")
    with pytest.raises(ValueError, match="tensor must live on the GPU"):
        torch.func.vmap(lambda t: L.ptr(t) or t)(torch.zeros(2, 3))
    with pytest.raises(TypeError):
        L.ptr()
