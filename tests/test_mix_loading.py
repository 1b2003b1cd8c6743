"""How libhydra_mix.so and the module beside it are opened, and what is said when they do not fit."""
import ctypes
import subprocess

import pytest

from hydrainfer_amd import _lib


@pytest.fixture
def fresh(monkeypatch):
    """Nothing opened yet."""
    for name, value in (("_mix", None), ("_front", None), ("_front_of", None), ("_front_tried", False)):
        monkeypatch.setattr(_lib, name, value, raising=False)


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
