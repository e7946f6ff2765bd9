"""When and with what the Python module is compiled: by the one compiler that the libraries need, and again for another
interpreter or torch."""
import os
import sysconfig

import pytest

from socket_amd import build


@pytest.fixture()
def compiled(monkeypatch, tmp_path):
    """Calls of the compiler, in a folder of their own."""
    calls = []

    def run(cmd):
        calls.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()

    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "HOST_PATH", str(tmp_path / "_host.so"))
    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "_stale", lambda src, out: not os.path.exists(out))
    return calls


def test_the_module_needs_no_other_compiler(compiled):
    assert os.path.exists(build.build_host())
    assert [c[0] for c in compiled] == [build._hipcc()]


def test_another_interpreter_or_torch_makes_it_again(compiled, monkeypatch):
    import torch

    build.build_host(only_changed=True)
    build.build_host(only_changed=True)
    assert len(compiled) == 1
    monkeypatch.setattr(torch, "__version__", torch.__version__ + "x")
    build.build_host(only_changed=True)
    build.build_host(only_changed=True)
    assert len(compiled) == 2
    monkeypatch.setattr(build.sys, "version", "another")
    build.build_host(only_changed=True)
    assert len(compiled) == 3


def test_missing_headers_are_named(compiled, monkeypatch, tmp_path):
    monkeypatch.setattr(sysconfig, "get_paths", lambda *a: {"include": str(tmp_path)})
    with pytest.raises(RuntimeError, match="Python.h"):
        build.build_host()
    assert not compiled
