"""When the libraries are mapped into the process (host only; no GPU).

The dynamic loader keeps a mapped file for its path, so a process that maps libm5k.so on import and
then builds the package would run the library that its build replaced."""

import subprocess
import sys
from pathlib import Path

import pytest
import torch

from m5kernels_amd import _lib, hip, quantize

PACKAGE = Path(__file__).resolve().parent.parent / "m5-max-kernels_amd"

MAPPED = "sorted({l.split()[-1] for l in open('/proc/self/maps') if '/m5k' in l or 'libm5k' in l})"


def test_importing_the_package_maps_no_library():
    code = f"import m5kernels_amd, m5kernels_amd.build, m5kernels_amd.harness.cli; print({MAPPED})"
    out = subprocess.run([sys.executable, "-c", code], cwd=PACKAGE, capture_output=True, text=True, check=True).stdout
    assert out.strip() == "[]"


def test_the_first_call_loads_the_native_front_once(monkeypatch):
    loads = []

    class Front:
        bind = staticmethod(lambda *args: loads.append("bind"))
        quantize = staticmethod(lambda *args: "codes")

    monkeypatch.setattr(_lib, "load_fast", lambda: loads.append("load") or Front)
    monkeypatch.setattr(hip, "_fast", hip._NativeFront())
    held = hip._fast
    assert quantize(None, "int8") == "codes" and hip._fast is Front
    assert quantize(None, "int8") == "codes" and held.quantize(None, "int8") == "codes"
    assert loads == ["load", "bind"]


def test_without_the_native_front_the_python_one_takes_the_call(monkeypatch):
    monkeypatch.setattr(_lib, "load_fast", lambda: None)
    monkeypatch.setattr(hip, "_fast", hip._NativeFront())
    with pytest.raises(ValueError, match="unknown quantization mode"):
        quantize(torch.zeros(2, 2), "int9")
    assert hip._fast is None


@pytest.fixture
def older_abi(monkeypatch):
    """The loaded library, with another ABI version than m5k_fast.so was compiled for."""
    lib = _lib.load()

    class Other:
        m5k_abi_version = staticmethod(lambda: lib.m5k_abi_version() + 100)

    monkeypatch.setattr(_lib, "load", lambda: Other)


def test_a_front_of_another_abi_is_refused(older_abi):
    with pytest.warns(RuntimeWarning, match="compiled for"):
        assert _lib.load_fast() is None


def test_a_front_of_another_torch_is_refused(monkeypatch):
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    with pytest.warns(RuntimeWarning, match="compiled for"):
        assert _lib.load_fast() is None


def test_the_built_front_matches_the_library():
    front = _lib.load_fast()
    assert front.abi_version == _lib.load().m5k_abi_version() and front.torch_version == torch.__version__
