"""The extension between the Python modules and the C ABI (csrc/host.cpp): what it takes as an argument, what it refuses, and that
the library sees the same values as through ctypes.  No launch: every call is refused by the library's own checks."""
import ctypes as C
import subprocess

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


def bad_stream():
    return L.PhiloxConfig(1, 0, 17, 256, 24, 0, 0, 0)        # no such mode: looked at behind widths and weights


def stack(dims=(32, 64, 4), w=(P, P), rng=None, fn=None, biases=None, x=P):
    """Status and message of a two-layer stack that the library's checks refuse at its random stream, if at nothing before."""
    stream = bad_stream() if rng is None else rng
    return refused(fn or L.lib.sp_mlp_forward, 1, x, 2, w, biases, dims, None, stream, P, P, None, 16, 1, 0, None)


AT_THE_STREAM = (-5, "philox mode")


def reaches(result, expected):
    return result[0] == expected[0] and expected[1] in result[1]


def test_elements_of_lists_arrive_as_addresses():
    arrays = lambda *v: (C.c_void_p * len(v))(*v)
    for make in (list, tuple, lambda v: arrays(*v)):
        assert reaches(stack(w=make((P, P + 16))), AT_THE_STREAM)
        assert reaches(stack(w=make((P, None))), (-1, "weights[1] is NULL"))
        assert reaches(stack(w=make((P + 4, P))), (-3, "weights[0] is not 16-byte aligned"))
        assert reaches(stack(w=make((P, P + 4))), (-3, "weights[1] is not 16-byte aligned"))
        assert reaches(stack(w=make((P,))), (-1, "weights[1] is NULL"))                   # too short: nothing behind the last
    for dims in ([32, 64], (32, 64), (C.c_int32 * 2)(32, 64)):
        assert reaches(stack(dims=dims), (-2, "dims[2] must be positive"))
    assert reaches(stack(w=[C.c_void_p(P), P], dims=(C.c_int32 * 40)(32, 64, 4)), AT_THE_STREAM)


def test_pointers_of_ctypes_mean_what_they_point_to():
    three, two, stream = (C.c_int32 * 3)(32, 64, 4), (C.c_void_p * 2)(P, P + 4), bad_stream()
    for fn in (L.lib.sp_mlp_forward, L.lib._cdll.sp_mlp_forward):
        ok = dict(fn=fn, dims=three, w=(C.c_void_p * 2)(P, P))
        assert reaches(stack(**dict(ok, dims=C.cast(three, C.POINTER(C.c_int32)))), AT_THE_STREAM)
        assert reaches(stack(**dict(ok, dims=C.POINTER(C.c_int32)())), (-1, "weights/dims is NULL"))
        assert reaches(stack(**dict(ok, w=C.cast(two, C.POINTER(C.c_void_p)))), (-3, "weights[1]"))
        assert reaches(stack(**dict(ok, rng=C.pointer(stream))), AT_THE_STREAM)
        assert reaches(stack(**dict(ok, rng=C.byref(stream))), AT_THE_STREAM)
        assert reaches(stack(**dict(ok, rng=stream)), AT_THE_STREAM)
        assert reaches(stack(**dict(ok, rng=(L.PhiloxConfig * 2)(stream, stream))), AT_THE_STREAM)
        assert reaches(stack(**dict(ok, x=C.cast(P + 8, C.POINTER(C.c_float)))), (-3, "x is not 16-byte aligned"))


WRONG = (TypeError, C.ArgumentError)


@pytest.mark.parametrize("rng", [1234, 0, C.c_void_p(P), C.c_int(5), C.byref(C.c_int(5)), C.pointer(C.c_int(5)), (C.c_int32 * 64)(), (1, 2), "seed",
                                 L.DeviceInfo(), C.byref(bad_stream(), 8), (L.PhiloxConfig * 0)(), np.zeros(64), torch.zeros(64)])
def test_a_random_stream_is_a_structure_of_its_type(rng):
    """A seed given for the stream was read as the address of one."""
    with pytest.raises(WRONG):
        stack(rng=rng)
    with pytest.raises(WRONG):
        L.lib.sp_philox_uniforms(rng, P, 8, 8, None)


@pytest.mark.parametrize("dims", [1234, C.c_void_p(P), (C.c_float * 3)(32, 64, 4), (C.c_int64 * 3)(32, 64, 4), (C.c_void_p * 3)(32, 64, 4), C.c_int64(5),
                                  C.byref(C.c_float(1)), C.pointer(C.c_int64(5)), C.byref((C.c_int32 * 3)(32, 64, 4)), C.byref(C.c_int32(32), 4),
                                  bad_stream(), np.zeros(3, np.int32), torch.zeros(3, dtype=torch.int32), [32.0, 64, 4], b"abcdefghijkl"])
def test_widths_are_integers_of_32_bits(dims):
    with pytest.raises(WRONG):
        stack(dims=dims)


@pytest.mark.parametrize("w", [P, C.c_void_p(P), (C.c_int64 * 2)(P, P), (C.c_int32 * 4)(), C.byref((C.c_void_p * 2)(P, P)), C.pointer(C.c_int64(P)),
                               bad_stream(), np.zeros(2, np.int64), [P, 0.5], ["P", P], [(C.c_int32 * 4)(), P]])
def test_weights_are_an_array_of_addresses(w):
    with pytest.raises(WRONG):
        stack(w=w)


@pytest.mark.parametrize("x", [C.c_int(5), C.c_float(5), C.byref(C.c_int(5)), (C.c_float * 4)(), bad_stream(), [P], 1.5, np.zeros(4)])
def test_device_memory_is_an_address(x):
    """The memory of an object of the host is none that a kernel may read; nor is a list, for a const int32_t* of the device."""
    with pytest.raises(WRONG):
        stack(x=x)
    with pytest.raises(WRONG):
        L.lib.sp_row_map_i32(6, x, P, 8, 8, None)
    assert refused(L.lib.sp_row_map_i32, 6, P + 4, P, 8, 8, None)[0] == -3


@pytest.mark.parametrize("name", [None, 5, ("a", "b"), b"x"])
def test_names_of_pointers_are_any_object(name):
    for make in (lambda: L.ptr(3, None, name), lambda: L.ptr(3, name=name)):
        with pytest.raises(TypeError) as err:
            make()
        assert str(err.value) == str(name) + " must be a torch.Tensor"
    with pytest.raises(ValueError, match="must live on the GPU"):
        L.ptr(torch.zeros(3), None, name)


def test_scalars_may_be_of_ctypes():
    """Of the parameter's own type, as through ctypes; every call is refused at a size or a misaligned address."""
    for fn in (L.lib.sp_map_f32, L.lib._cdll.sp_map_f32):
        assert refused(fn, C.c_int(1), P, P, C.c_int64(-(1 << 40)), None)[0] == -2
        for wrong in ((C.c_int64(1), P, P, 4, None), (1, P, P, C.c_int32(4), None), (1, P, P, C.c_float(4), None)):
            with pytest.raises(WRONG):
                fn(*wrong)
    for fn in (L.lib.sp_row_l1_normalize, L.lib._cdll.sp_row_l1_normalize):
        got = [refused(fn, P + 4, P, 8, 8, t, None) for t in (C.c_float(0.5), 0.5, 1, True)]
        assert got[0][0] == -3 and all(g == got[0] for g in got)
        for wrong in (C.c_double(0.5), C.c_int(1), "1"):
            with pytest.raises(WRONG):
                fn(P + 4, P, 8, 8, wrong, None)
    for fn in (L.lib.sp_row_binarize, L.lib._cdll.sp_row_binarize):
        assert refused(fn, P, P, 8, 8, C.c_uint32(0), None)[0] == -5
    for fn in (L.lib.sp_cem_resample_philox, L.lib._cdll.sp_cem_resample_philox):
        assert refused(fn, P, P, C.c_uint64(1), C.c_uint64(2), P, 0, 8, 0.5, 0.5, None)[0] == -2


def test_refused_arguments_raise_what_ctypes_raises():
    for args, number in (((1, "P", P, 4, None), None), ((1, P, object(), 4, None), 3), ((1, P, P, 4.5, None), 4), ((C.c_float(1), P, P, 4, None), 1)):
        with pytest.raises(C.ArgumentError) as err:
            L.lib.sp_map_f32(*args)
        assert isinstance(err.value, TypeError) and (number is None or str(err.value).startswith("argument %d: " % number))
        if number is not None:
            with pytest.raises(C.ArgumentError, match="argument %d: " % number):
                L.lib._cdll.sp_map_f32(*args)
    with pytest.raises(C.ArgumentError, match="argument 8: a random stream is None or a PhiloxConfig, not int"):
        stack(rng=1234)


def test_each_library_keeps_its_own_functions(tmp_path):
    """Functions bound to a second library leave those of the first as they are."""
    names = [n for n in L.SIGNATURES if L.SIGNATURES[n][1][-1:] == [L._P]]
    (tmp_path / "other.c").write_text("".join("int %s() { return -42; }\n" % n for n in names))
    other = str(tmp_path / "libother.so")
    subprocess.run(["gcc", "-w", "-shared", "-fPIC", str(tmp_path / "other.c"), "-o", other], check=True)
    refused_before = L.lib.sp_map_f32(1, P, P, -1, None)
    functions = L._host.bind(other, L.PhiloxConfig)
    assert refused_before == -2 and functions["sp_map_f32"](1, P, P, -1, None) == -42
    assert L.lib.sp_map_f32(1, P, P, -1, None) == -2 and functions["sp_row_map_i32"](6, P, P, 8, 8, None) == -42


def test_each_library_keeps_its_own_structure():
    """A second module with a structure of its own for random streams, or this one loaded again, leaves the first one's as it was."""
    class Other(C.Structure):
        _fields_ = L.PhiloxConfig._fields_
    functions = L._host.bind(L.lib._cdll._name, Other)
    assert reaches(stack(rng=bad_stream()), AT_THE_STREAM)
    other = Other.from_buffer_copy(bad_stream())
    assert reaches(stack(fn=functions["sp_mlp_forward"], rng=other), AT_THE_STREAM)
    for fn, rng in ((L.lib.sp_mlp_forward, other), (functions["sp_mlp_forward"], bad_stream())):
        with pytest.raises(WRONG):
            stack(fn=fn, rng=rng)


def test_lists_may_change_while_they_are_read():
    class Shortens:
        def __index__(self):
            dims.clear()
            return 64
    dims = [32]
    dims += [Shortens(), 4]
    with pytest.raises(RuntimeError, match="changed its size"):
        stack(dims=dims)
