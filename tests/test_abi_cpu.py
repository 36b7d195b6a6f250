"""CPU-side checks of the boundary: the shared library loads and exports every symbol the
header declares, and argument errors come back as status codes without a GPU."""
import ctypes as C
import os
import re
import time
import types

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_symbols():
    text = open(os.path.join(ROOT, "include", "autograph_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(agh_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from autograph_amd import _ffi
    syms = header_symbols()
    assert len(syms) >= 30
    for s in syms:
        assert hasattr(_ffi.lib, s), f"{s} declared in the header but not exported"
    # and the ctypes table covers the header exactly
    assert sorted(_ffi.SIGNATURES) == syms


def test_calls_before_init_fail_with_status_not_crash():
    from autograph_amd import _ffi
    p = C.c_void_p()
    rc = _ffi.lib.agh_malloc(C.byref(p), 16)
    if rc == 0:  # a GPU is present and another test initialised the library
        _ffi.lib.agh_free(p)
        return
    assert rc == -2  # AGH_ENOINIT
    assert b"agh_init" in _ffi.lib.agh_last_error_string()
    assert _ffi.lib.agh_gemm_f32(1, 1, 1, 1.0, None, 0, 1, 1, None, 0, 1, 1, 0.0, None, 0, 1, 1) == -2


def test_calls_that_read_no_variable_do_not_walk_the_environment(monkeypatch):
    """An entry point that no AGH_* variable concerns costs the same whatever the environment's size (a walk through 8000 variables
    takes about 5 us, the call itself 0.3)."""
    from autograph_amd import _ffi

    def us():
        best = float("inf")
        for _ in range(20):
            t0 = time.perf_counter()
            for _ in range(50):
                _ffi.lib.agh_branch_join()
            best = min(best, time.perf_counter() - t0)
        return best / 50 * 1e6
    few = us()
    for i in range(8000):
        monkeypatch.setenv(f"FILLER_{i}", "1")
    assert us() < 2 * few + 2


def test_option_shape_formulas():
    from autograph_amd import Col2ImConv2Options, Im2ColConv2Options, MaxPool2Options
    import oracle as orc
    o = Im2ColConv2Options(filter=(3, 5), padding=(1, 0), stride=(2, 1), dilation=(1, 2))
    assert o.output_shape((9, 14)) == (orc.conv_out(9, 3, 1, 2, 1), orc.conv_out(14, 5, 0, 1, 2))
    c = Col2ImConv2Options(shape=(5, 6), filter=(3, 5), padding=(1, 0), stride=(2, 1), dilation=(1, 2))
    assert c.output_shape() == (orc.col2im_out(5, 3, 1, 2, 1), orc.col2im_out(6, 5, 0, 1, 2))
    assert MaxPool2Options((2, 3), (2, 2)).output_shape((9, 8)) == (orc.pool_out(9, 2, 2), orc.pool_out(8, 3, 2))


@pytest.mark.parametrize("shape", [(np.int16(300), np.int16(300)), (np.uint8(28), np.uint8(28)), (100, np.int16(1000)),
                                   (np.int32(802816), np.int32(3200)), (np.int8(100),) * 3, (np.int16(100),) * 4, np.array([200, 200], np.uint8)])
def test_narrow_integers_as_dimensions(monkeypatch, shape):
    """8-, 16- and 32-bit numpy integers as dimensions: allocated size, length, strides and reshapes are those of the same Python integers
    (products of such numbers wrap; no device: the allocation is only recorded)."""
    from autograph_amd import tensor
    sizes = []
    monkeypatch.setattr(tensor, "Buffer", lambda nbytes: sizes.append(nbytes) or types.SimpleNamespace(ptr=0, nbytes=nbytes))
    dims = tuple(int(d) for d in shape)
    want = 1
    for d in dims:
        want *= d
    for dtype, size in (("f32", 4), ("bf16", 2)):
        t = tensor.Tensor.uninit(shape, dtype)
        assert sizes.pop() == size * want and t.shape == dims and all(type(d) is int for d in t.shape)
        assert len(t) == want and t.strides == tensor._std_strides(dims) and t.is_standard_layout()
        assert t.into_shape((want,)).into_shape(shape).strides == t.strides
        assert len(tensor.Tensor(t.buffer, shape, t.strides, 0, dtype)) == want
    with pytest.raises(tensor.AghError):
        t.into_shape((want + 1,))


@pytest.mark.parametrize("shape", [(2.5, 4), ("2", 4), ("24",), (np.float32(2.5), 4)])
def test_dimensions_that_are_no_whole_numbers_are_refused(monkeypatch, shape):
    """Not cut down to whole ones: 2.5 x 4 is no shape of the eight elements of 2 x 4.  (Whole floats count as the integers they are.)"""
    from autograph_amd import tensor
    monkeypatch.setattr(tensor, "Buffer", lambda nbytes: types.SimpleNamespace(ptr=0, nbytes=nbytes))
    t = tensor.Tensor.uninit((2, 4), "f32")
    with pytest.raises(tensor.AghError):
        t.into_shape(shape)
    with pytest.raises(tensor.AghError):
        tensor.Tensor.uninit(shape, "f32")
    assert t.into_shape((4.0, np.int8(2))).shape == (4, 2)


_C_TO_RUST = {"int": "c_int", "int64_t": "i64", "float": "f32", "size_t": "usize", "char": "c_char", "void": "c_void"}


def _rust_type_of(ctype):
    """The Rust FFI spelling of a C parameter type: pointers keep their depth and the constness of the pointee."""
    const = re.search(r"\bconst\b", ctype) is not None
    base = re.sub(r"\bconst\b|\*", " ", ctype).split()
    assert len(base) == 1, ctype
    out = _C_TO_RUST[base[0]]
    for level in range(ctype.count("*")):
        out = ("*const " if const and level == 0 else "*mut ") + out
    return out


def test_rust_sys_crate_declares_the_header():
    """rust/autograph-hip-sys/src/lib.rs (source only, no Rust toolchain here) must declare every entry
    point of the header with the same argument TYPES in the same order (int64_t <-> i64, int <-> c_int,
    float <-> f32, size_t <-> usize, pointers with their constness and depth) and the same return type."""
    text = open(os.path.join(ROOT, "include", "autograph_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    c_decls = {}
    for ret, name, args in re.findall(r"^\s*([a-z_0-9 ]+?\s*\**)\s*\b(agh_[a-z0-9_]+)\s*\(([^)]*)\)\s*;", text, flags=re.M):
        types = []
        if args.strip() not in ("", "void"):
            for a in args.split(","):
                a = " ".join(a.split())
                types.append(_rust_type_of(re.sub(r"[A-Za-z_][A-Za-z_0-9]*$", "", a)))  # drop the parameter name
        c_decls[name] = (types, _rust_type_of(ret))
    rs = open(os.path.join(ROOT, "rust", "autograph-hip-sys", "src", "lib.rs")).read()
    rs_decls = {}
    for name, args, ret in re.findall(r"pub fn (agh_[a-z0-9_]+)\(([^)]*)\) -> ([^;]+);", rs):
        types = [a.split(":", 1)[1].strip() for a in args.split(",")] if args.strip() else []
        rs_decls[name] = (types, ret.strip())
    assert sorted(rs_decls) == sorted(c_decls)
    for name in c_decls:
        assert rs_decls[name] == c_decls[name], name
    assert sorted(c_decls) == header_symbols()
    # the ctypes table agrees too (same width and kind per argument)
    from autograph_amd import _ffi
    kind = {"c_int": C.c_int, "i64": C.c_int64, "f32": C.c_float, "usize": C.c_size_t}
    for name, (types, _) in c_decls.items():
        argtypes = _ffi.SIGNATURES[name][0]
        assert len(argtypes) == len(types), name
        for t, ct in zip(types, argtypes):
            if t.startswith("*"):
                assert C.sizeof(ct) == C.sizeof(C.c_void_p) and not issubclass(ct, (C.c_int64, C.c_size_t, C.c_float)) or ct is C.c_void_p, (name, t, ct)
            else:
                assert ct is kind[t] or (C.sizeof(ct) == C.sizeof(kind[t]) and ct._type_ == kind[t]._type_), (name, t, ct)


def test_native_calls_mean_what_the_ctypes_calls_mean():
    """The calls without ctypes: errors carry the entry's code and message, arguments that are no plain numbers (a ctypes pointer, a bool, a
    numpy integer, too few) do what ctypes makes of them, integers wrap to their width; a Buffer owns what its `ptr` says."""
    from autograph_amd import AghError, Buffer, _ffi
    gemm = _ffi.calls.agh_gemm_f32
    args = [1, 1, 1, 1.0, None, 0, 1, 1, None, 0, 1, 1, 0.0, None, 0, 1, 1]
    for a in (args, args[:4] + [C.c_void_p(None)] + args[5:], [True] + args[1:], [np.int64(1)] + args[1:]):
        with pytest.raises(AghError) as e:
            gemm(*a)
        assert e.value.code == -2 and "agh_init" in str(e.value)  # no device here
    for a in (args[:-1], args[:3] + ["1.0"] + args[4:], [1.0] + args[1:]):
        with pytest.raises((TypeError, C.ArgumentError)):
            gemm(*a)
    for a in (args[:3] + [10**400] + args[4:], args[:3] + [10**400, C.c_void_p(None)] + args[5:]):  # an integer that no float holds
        with pytest.raises(C.ArgumentError):
            gemm(*a)
    with pytest.raises(AghError):
        gemm(*args[:3], 10**300, *args[4:])
    with pytest.raises(AghError):
        gemm(2**64 + 1, *args[1:])
    for size in (16, np.int64(16), True):
        with pytest.raises(AghError):
            Buffer(size)
    for size in (1.5, "16", None):
        with pytest.raises((TypeError, C.ArgumentError)):
            Buffer(size)
    b = Buffer.__new__(Buffer)  # what a failed allocation leaves: nothing is owned, dropping it frees nothing
    b.ptr = None
    b.note = "instances take attributes"
    del b


def test_one_instance_of_the_library(tmp_path):
    """The calls without ctypes reach the library that ctypes has opened, not another one that the loader's search path holds."""
    import shutil
    import subprocess
    import sys

    from autograph_amd import _ffi
    shutil.copy(_ffi.LIB_PATH, tmp_path / os.path.basename(_ffi.LIB_PATH))
    program = ("import autograph_amd\n"
               "print(len({line.split()[-1] for line in open('/proc/self/maps') if line.rstrip().endswith('/libautograph_hip.so')}))\n")
    env = dict(os.environ, LD_LIBRARY_PATH=os.pathsep.join(filter(None, (str(tmp_path), os.environ.get("LD_LIBRARY_PATH")))))
    out = subprocess.run([sys.executable, "-c", program], env=env, cwd=ROOT, check=True,
                         capture_output=True, text=True).stdout
    assert out.strip() == "1"


def test_library_is_built_without_python():
    """`make lib`, and `make` where there are no Python headers, build the library and not the package's extension."""
    import subprocess

    def commands(*args):
        return subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "autograph_amd", "csrc"), *args], check=True, capture_output=True, text=True).stdout
    for args in (("lib",), ("PYTHON=false",)):
        text = commands(*args)
        assert "-o ../lib/libautograph_hip.so" in text and "agh_calls.cpp -o" not in text, args
    assert "agh_calls.cpp -o ../_calls." in commands()
