"""The compiled operator call is a shorter way to the library, not a part of it: the package loads without it, or beside one
that was made for something else."""
import sys

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


def test_a_tree_with_the_library_alone_is_not_built(monkeypatch, tmp_path):
    assert build.is_built()
    monkeypatch.setattr(build, "BINDING_PATH", str(tmp_path / "_binding.so"))
    assert not build.is_built()
