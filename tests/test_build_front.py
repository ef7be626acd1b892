"""libm5k.so builds without the headers of the native front (Python's and torch's), and is in place
also where the front does not compile.  A small source tree stands for csrc/ and diag/."""

import ctypes
import shutil

import pytest

from m5kernels_amd import build

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")


@pytest.fixture
def tree(monkeypatch, tmp_path):
    for folder in ("csrc", "diag", "lib"):
        (tmp_path / folder).mkdir()
    (tmp_path / "csrc" / "one.cpp").write_text('extern "C" int answer() { return 42; }\n')
    (tmp_path / "diag" / "two.hip").write_text("#include <hip/hip_runtime.h>\n__global__ void nothing() {}\n")
    (tmp_path / "front.cpp").write_text("#error does not compile\n")
    (tmp_path / "lib" / "m5k_fast.so").write_text("of an older build")
    for name, value in dict(CSRC="csrc", DIAG_DIR="diag", BUILD_DIR="objects", LIB_PATH="lib/libm5k.so",
                            DIAG_LIB_PATH="lib/libm5k_diag.so", FAST_SRC="front.cpp",
                            FAST_PATH="lib/m5k_fast.so").items():
        monkeypatch.setattr(build, name, tmp_path / value)
    return tmp_path


def _built(tree):
    assert (tree / "lib" / "libm5k_diag.so").exists()
    assert not (tree / "lib" / "m5k_fast.so").exists()
    return ctypes.CDLL(str(tree / "lib" / "libm5k.so")).answer() == 42


def test_without_the_headers_of_the_front(tree, monkeypatch):
    monkeypatch.setattr(build, "_front_includes", lambda: [])
    with pytest.warns(RuntimeWarning, match="m5k_fast.so is not built"):
        build.build()
    assert _built(tree)


def test_a_front_that_does_not_compile_is_an_error_beside_a_built_library(tree):
    with pytest.raises(RuntimeError, match="front.cpp"):
        build.build()
    assert _built(tree)


def test_headers_are_looked_for(monkeypatch, tmp_path):
    assert build._front_includes()
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build._front_includes() == []
