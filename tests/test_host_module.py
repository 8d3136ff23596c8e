"""Which file of the launches' host side an environment loads, and what happens where none can be compiled."""
import os
import sysconfig

import pytest
import torch

from longbow_quarrel_amd import build
from longbow_quarrel_amd.kernels import hip


@pytest.fixture
def elsewhere(tmp_path, monkeypatch):
    """An empty folder in the place of those where built files lie."""
    monkeypatch.setattr(build, "lib_dirs", lambda: [str(tmp_path)])
    return tmp_path


def test_a_module_of_another_environment_is_not_taken(elsewhere, monkeypatch):
    names = {build.host_name()}
    (elsewhere / build.host_name()).write_bytes(b"")
    assert build.find_host() == str(elsewhere / build.host_name())
    for where, name, value in ((torch, "__version__", "9.9.9"), (torch._C, "_GLIBCXX_USE_CXX11_ABI", not torch._C._GLIBCXX_USE_CXX11_ABI),
                               (build, "HOST_FLAGS", build.HOST_FLAGS + ["-g"]),
                               (sysconfig, "get_config_var", lambda name: "cpython-399-other")):
        with monkeypatch.context() as m:
            m.setattr(where, name, value)
            assert build.find_host() is None
            names.add(build.host_name())
    assert len(names) == 5 and build.find_host() is not None


def test_only_the_module_is_built_again(elsewhere, monkeypatch):
    monkeypatch.setattr(build, "_hipcc", lambda: pytest.fail("the kernels were compiled"))
    path = build.ensure_host()
    assert path == str(elsewhere / build.host_name()) == build.find_host() and os.path.getsize(path) > 0
    written = os.path.getmtime(path)
    assert build.ensure_host() == path and os.path.getmtime(path) == written
    assert build.find_built() is None


@pytest.mark.parametrize("compiler", ["/nowhere/c++", "false"])
def test_without_a_compiler_the_checks_are_made_in_python(elsewhere, monkeypatch, compiler):
    monkeypatch.setenv("CXX", compiler)
    with pytest.raises(build.BuildError):
        build.ensure_host()
    monkeypatch.setattr(hip, "_HOST", None)
    monkeypatch.setattr(hip, "load_library", lambda: None)
    host = hip.load_host()
    assert [getattr(host, name)(1, 2) for name in ("linear", "linear_swiglu", "rmsnorm", "attention", "rope_store_pieces")] == [0] * 5
    assert os.listdir(elsewhere) == []
