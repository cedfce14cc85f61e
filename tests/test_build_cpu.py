"""The host launch module is bound to the torch and the Python that it was built for."""

import pytest

from iris_amd import _native, build


def test_the_module_names_what_it_was_built_for():
    assert build.host_built_for() == build.host_abi()


def test_another_torch_rebuilds_and_does_not_load(monkeypatch):
    monkeypatch.setattr(build, "_stale", lambda target, deps: False)  # (sources as they were)
    assert not build.host_stale()
    monkeypatch.setattr(build, "host_abi", lambda: "cpython-399, torch 9.9")
    monkeypatch.setattr(_native, "_host", None)
    assert build.host_stale()
    with pytest.raises(RuntimeError, match="built for .*this is cpython-399, torch 9.9"):
        _native.host()
