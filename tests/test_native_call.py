"""Calls of C functions by address (``ops.native_call``): every argument arrives where the function looks for it, as
through ctypes, and what is no number is refused."""
import ctypes
import os
import platform
import shutil
import subprocess
import sysconfig

import pytest

from minivllm_amd import build
from minivllm_amd.ops import native_call

SOURCE = r"""
#include <stdint.h>
int none(void) { return -7; }
long many(void* a, long b, int c, void* d, float e, int f, int g, long h, void* i, int j, float k, int l, void* m, long n,
          int o, int p, float q, int r, int s, void* t, int u, float v, uint64_t w, int x, float y, float z, float aa, float ab, long ac) {
    return 3 * (long)a + 5 * b + 7 * c + 11 * (long)d + (long)(e * 16) + 13 * f + 17 * g + 19 * h + 23 * (long)i + 29 * j +
           (long)(k * 32) + 31 * l + 37 * (long)m + 41 * n + 43 * o + 47 * p + (long)(q * 64) + 53 * r + 59 * s + 61 * (long)t +
           67 * u + (long)(v * 128) + (long)(w >> 60) + 71 * x + (long)(y * 256) + (long)(z * 512) + (long)(aa * 1024) +
           (long)(ab * 2048) + 73 * ac;
}
"""
P, L, I, F, U = ctypes.c_void_p, ctypes.c_long, ctypes.c_int, ctypes.c_float, ctypes.c_uint64
MANY = [P, L, I, P, F, I, I, L, P, I, F, I, P, L, I, I, F, I, I, P, I, F, U, I, F, F, F, F, L]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None or native_call._native is None:
        pytest.skip("no C compiler, or no native calls")
    d = tmp_path_factory.mktemp("call")
    (d / "f.c").write_text(SOURCE)
    subprocess.run([cc, "-O1", "-shared", "-fPIC", "-o", str(d / "f.so"), str(d / "f.c")], check=True)
    return ctypes.CDLL(str(d / "f.so"))


def test_arguments(lib):
    f = native_call.bind(lib, "many", MANY, L)
    args = [1 << 46, -5, -(1 << 31), None, -1.5, 7, -1, -(1 << 50), 77, True, 2.25, -2, 12345678901, 1 << 40, 1, -2, 3, 4, 5, 6,
            False, 7.0, (1 << 64) - 1, 9, 0.5, -0.25, 8, 1e3, -1]
    assert f is not lib.many and f(*args) == lib.many(*args)
    assert native_call.bind(lib, "none", [])() == -7


def test_what_is_refused(lib):
    f = native_call.bind(lib, "many", MANY, L)
    args = [0] * len(MANY)
    for bad in (args[:-1], args + [0], [1.0] + args[1:], ["x"] + args[1:], args[:4] + ["x"] + args[5:], args[:4] + [None] + args[5:]):
        with pytest.raises(TypeError):
            f(*bad)
    # None is a pointer and no number; a pointer is an int and nothing that stands for one (a tensor's item would be waited for)
    class Index:
        def __index__(self):
            return 5
    for i, t in enumerate(MANY):
        bad = args[:i] + [Index() if t is P else None] + args[i + 1:]
        with pytest.raises(TypeError):
            f(*bad)
        with pytest.raises(ctypes.ArgumentError):
            lib.many(*bad)
    assert f(*[None if t is P else Index() if t is not F else 0 for t in MANY]) == \
        lib.many(*[None if t is P else Index() if t is not F else 0 for t in MANY])
    for types in ("", "i", "iX", "f" * 9 + "I", "i" * 47 + "I"):
        with pytest.raises(ValueError):
            native_call._native.bind(1, types)


def test_without_it(lib, monkeypatch):
    """ctypes takes the calls where the module is not there."""
    monkeypatch.setattr(native_call, "_native", None)
    f = native_call.bind(lib, "many", MANY, L)
    assert f(*[1] * len(MANY)) == lib.many(*[1] * len(MANY))


@pytest.fixture
def empty_package(monkeypatch, tmp_path):
    """The builder with a package folder of its own, and a source in it."""
    (tmp_path / "launch.cpp").write_bytes(open(build.LAUNCH_SRC, "rb").read())
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "LAUNCH_SRC", str(tmp_path / "launch.cpp"))
    return tmp_path


@pytest.mark.parametrize("lack", ["machine", "headers", "compiler"])
def test_done_without_where_it_cannot_be_built(empty_package, monkeypatch, lack):
    if lack == "machine":
        monkeypatch.setattr(platform, "machine", lambda: "aarch64")
    elif lack == "headers":
        monkeypatch.setattr(sysconfig, "get_paths", lambda: {"include": str(empty_package)})
    else:
        monkeypatch.setattr(shutil, "which", lambda name: None)
    assert build.build_launch(verbose=False) == "" and build.build_launch(force=True) == ""
    with pytest.warns(UserWarning, match="ctypes"):
        assert native_call._load() is None


def test_named_by_source_and_interpreter(lib, empty_package):
    first = build.build_launch(verbose=False)
    assert first.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and os.path.exists(first)
    stamp = os.stat(first).st_mtime_ns
    assert build.build_launch(verbose=False) == first and os.stat(first).st_mtime_ns == stamp
    (empty_package / "launch.cpp").open("a").write("// another source\n")
    second = build.build_launch(verbose=False)
    assert second != first and os.listdir(empty_package).count(os.path.basename(first)) == 0
    assert native_call._load() is not None
    (empty_package / "launch.cpp").write_text("no C++\n")
    with pytest.warns(UserWarning, match="command failed"):
        assert native_call._load() is None
