"""The compiled operator call is a shorter way to the library, not a part of it: the package loads without it, or beside one
that was made for something else."""
import os
import subprocess
import sys
import types
import warnings

import pytest

import patrickstar_amd as ps
from patrickstar_amd import _lib, build


@pytest.fixture
def fresh(monkeypatch):
    """The library as a process finds it that has not loaded it yet."""
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.delattr(ps, "_binding", raising=False)
    return monkeypatch


def test_the_library_loads_without_the_binding(fresh):
    fresh.setitem(sys.modules, "patrickstar_amd._binding", None)
    with pytest.warns(RuntimeWarning, match="without its compiled call"):
        lib = _lib.load()
    assert lib.ps_abi_version() == _lib.PS_ABI_VERSION
    assert lib.adam_update(*range(13)) is None  # "not of the ordinary form": the caller goes on to the general path


def test_without_the_binding_no_step_asks_the_library_for_it(fresh):
    """ctypes looks a name up in the library and all that it needs, again every time."""
    fresh.setitem(sys.modules, "patrickstar_amd._binding", None)
    with pytest.warns(RuntimeWarning):
        lib = _lib.load()
    assert vars(lib)["compiled"] is None


@pytest.mark.parametrize("source,says", [
    ("int ps_abi_version(void) { return %d; }" % (_lib.PS_ABI_VERSION - 1), f"has ABI version {_lib.PS_ABI_VERSION - 1}, expected {_lib.PS_ABI_VERSION}; rebuild it"),
    ("int ps_abi_version(void) { return %d; }" % _lib.PS_ABI_VERSION, "has no ps_.*; rebuild it"), ("int other;", "rebuild it"),
])
def test_an_older_library_is_told_to_be_rebuilt(fresh, tmp_path, source, says):
    """Of another version, or of this one before an entry point was added."""
    (tmp_path / "old.c").write_text(source)
    subprocess.check_call(["gcc", "-shared", "-fPIC", str(tmp_path / "old.c"), "-o", str(tmp_path / "old.so")])
    fresh.setattr(_lib, "LIB_PATH", str(tmp_path / "old.so"))
    with pytest.raises(_lib.HipLibraryMissing, match=says):
        _lib.load()


@pytest.mark.parametrize(
    "made_for",
    [dict(), dict(abi_version=_lib.PS_ABI_VERSION - 1, built_for=build.built_for()), dict(abi_version=_lib.PS_ABI_VERSION, built_for="Python 3.9, torch 2.4.0")],
)
def test_a_binding_made_for_something_else_is_not_called(fresh, made_for):
    """It calls ps_adam_update by its address, through the signature it was compiled with."""
    other = types.ModuleType("patrickstar_amd._binding")
    other.__file__ = "_binding.so"
    other.adam_update = lambda *a: pytest.fail("called")
    other.__dict__.update(made_for)
    fresh.setitem(sys.modules, "patrickstar_amd._binding", other)
    fresh.setattr(ps, "_binding", other, raising=False)
    with pytest.warns(RuntimeWarning, match="was built for ABI version"):
        lib = _lib.load()
    assert lib.adam_update(*range(13)) is None


def test_the_binding_of_this_build_is_used(fresh):
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        lib = _lib.load()
    assert lib.adam_update.func is ps._binding.adam_update


def test_a_tree_with_the_library_alone_is_not_built(monkeypatch, tmp_path):
    assert build.is_built()
    monkeypatch.setattr(build, "BINDING_PATH", str(tmp_path / "_binding.so"))
    assert not build.is_built()


@pytest.mark.parametrize("fails", ["g++", "hipcc"])
def test_a_build_that_fails_leaves_both_files_as_they_were(monkeypatch, tmp_path, fails):
    for name in ("LIB_PATH", "BINDING_PATH"):
        path = tmp_path / os.path.basename(getattr(build, name))
        path.write_text("old")
        monkeypatch.setattr(build, name, str(path))

    def compiler(cmd):
        if fails in os.path.basename(cmd[0]):
            raise subprocess.CalledProcessError(1, cmd)
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("new")

    monkeypatch.setattr(build.subprocess, "check_call", compiler)
    monkeypatch.setattr(build, "hipcc_path", lambda: "/opt/rocm/bin/hipcc")
    with pytest.raises(subprocess.CalledProcessError):
        build.build()
    assert {p.name: p.read_text() for p in tmp_path.iterdir()} == {"libps_adam.so": "old", "_binding.so": "old"}
    fails = "nothing"
    assert build.build() == build.LIB_PATH
    assert {p.name: p.read_text() for p in tmp_path.iterdir()} == {"libps_adam.so": "new", "_binding.so": "new"}
