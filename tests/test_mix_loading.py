"""How libhydra_mix.so and the module beside it are opened, and what is said when they do not fit."""
import ctypes
import subprocess

import pytest

from hydrainfer_amd import _lib


@pytest.fixture
def fresh(monkeypatch):
    """Nothing opened yet."""
    for name in ("_mix", "_front", "_front_of"):
        monkeypatch.setattr(_lib, name, None)


def _library(tmp_path, name, text):
    source, out = tmp_path / "x.c", tmp_path / name
    source.write_text(text)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(out), str(source)], check=True)
    return str(out)


@pytest.mark.parametrize("version", [_lib.HXM_ABI_VERSION - 1, _lib.HXM_ABI_VERSION + 1])
def test_a_library_of_another_version_is_named_as_such(fresh, monkeypatch, tmp_path, version):
    # (without the entry points that came with this version)
    monkeypatch.setattr(_lib, "MIX_LIB_PATH", _library(tmp_path, "libother.so", f"int hxm_abi_version(void) {{ return {version}; }}"))
    with pytest.raises(_lib.HydraHipError, match=f"ABI version {version} != .*rebuild"):
        _lib.mix_lib()


def test_the_version_with_the_key_splits_of_biased_attention():
    assert "hxm_biased_attention_plan" in _lib._MIX_SIGNATURES and _lib.HXM_ABI_VERSION >= 8
    assert isinstance(_lib.mix_lib(), ctypes.CDLL)


def test_the_module_fits_this_torch_and_python(fresh):
    front = _lib.front()
    assert front is not None and front is _lib._front and _lib._front_of is _lib.mix_lib()


def _no_module(tmp_path):
    return str(tmp_path / "nothing.so")


def _not_a_library(tmp_path):
    path = tmp_path / "text.so"
    path.write_text("not a library")
    return str(path)


def _other_torch(tmp_path):
    return _library(tmp_path, "libfront.so", 'const char* hydra_front_built_for(void) { return "ABI 8, torch 1.0, Python 3.0"; }')


def _without_a_version(tmp_path):
    return _library(tmp_path, "libfront.so", "int x;")


def _missing_symbol(tmp_path):
    return _library(tmp_path, "libfront.so", "int gone(void); int hydra_front_built_for(void) { return gone(); }")


@pytest.mark.parametrize("path", [_no_module, _not_a_library, _other_torch, _without_a_version, _missing_symbol])
def test_without_a_module_that_fits_calls_go_on_in_python(fresh, monkeypatch, tmp_path, path):
    """Said once, with what to build; the library itself is open, and nobody is refused."""
    monkeypatch.setattr(_lib, "FRONT_PATH", path(tmp_path))
    with pytest.warns(UserWarning, match="make -C hydrainfer_amd/csrc front") as said:
        lib = _lib.mix_lib()
        assert _lib.front() is None and _lib.mix_lib() is lib
    assert len(said) == 1 and lib.hxm_abi_version() == _lib.HXM_ABI_VERSION


def test_a_stand_in_for_the_library_goes_through_python(fresh, monkeypatch):
    lib = _lib.mix_lib()

    class StandIn:
        def __getattr__(self, name):
            return getattr(lib, name)

    monkeypatch.setattr(_lib, "_mix", StandIn())
    assert _lib.front() is None
    monkeypatch.setattr(_lib, "_mix", lib)
    assert _lib.front() is not None
