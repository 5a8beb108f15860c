"""The native front of the basket queries is no prerequisite of anything: the
build goes on without it, and queries.py answers through its Python checks
where it is absent."""
import os
import shutil
import subprocess
import types

import pytest

import __graft_entry__ as entry
from vecgeom_amd import queries as Q


@pytest.fixture
def csrc_copy(tmp_path, monkeypatch):
    """A tree with the front's Makefile and source alone."""
    d = tmp_path / "vecgeom_amd"
    (d / "csrc").mkdir(parents=True)
    here = os.path.join(entry.ROOT, "vecgeom_amd")
    shutil.copy(os.path.join(here, "Makefile"), d)
    shutil.copy(os.path.join(here, "csrc", "py_queries.cpp"), d / "csrc")
    monkeypatch.setattr(entry, "ROOT", str(tmp_path))
    return d


def test_library_target_needs_no_front(csrc_copy):
    r = subprocess.run(["make", "-n", "-C", str(csrc_copy), "OBJ=", "HDR="], capture_output=True, text=True)
    assert r.returncode == 0 and "libvecgeom_amd.so" in r.stdout and "_vgq" not in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("break_it", ["headers", "compiler", "torch"])
def test_build_goes_on_without_the_front(csrc_copy, monkeypatch, capfd, break_it):
    if break_it == "headers":  # a torch without its C++ side
        found = types.SimpleNamespace(origin=str(csrc_copy / "__init__.py"))
        monkeypatch.setattr(entry.importlib.util, "find_spec", lambda name: found)
    elif break_it == "compiler":
        monkeypatch.setenv("CXX", "/nonexistent/c++")
    else:
        monkeypatch.setattr(entry.importlib.util, "find_spec", lambda name: None)
    assert entry.build_front() is False
    assert "native front" in capfd.readouterr().out
    assert not os.path.exists(csrc_copy / "lib" / "_vgq.so")


def test_front_follows_the_interpreter_not_the_path(csrc_copy, monkeypatch, tmp_path):
    """A PATH whose python3 has no torch changes nothing: the folders named
    are those of the interpreter that builds."""
    stub = tmp_path / "bin"
    stub.mkdir()
    (stub / "python3").write_text("#!/bin/sh\nexit 1\n")
    (stub / "python3").chmod(0o755)
    monkeypatch.setenv("PATH", f"{stub}:{os.environ['PATH']}")
    compiler = tmp_path / "cxx"
    compiler.write_text('#!/bin/sh\necho "$@" > ' + str(tmp_path / "args") + "\n")
    compiler.chmod(0o755)
    monkeypatch.setenv("CXX", str(compiler))
    assert entry.build_front() is True
    args = (tmp_path / "args").read_text().split()
    import torch
    assert f"-I{os.path.dirname(torch.__file__)}/include" in args
    assert f"-I{entry.sysconfig.get_paths()['include']}" in args


@pytest.mark.parametrize("content", [None, b"not a library"])
def test_queries_without_the_front(monkeypatch, tmp_path, content):
    path = tmp_path / "_vgq.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(Q, "_FRONT_PATH", str(path))
    monkeypatch.setattr(Q, "_front", None)

    class Geometry:
        handle = None
    with pytest.warns(RuntimeWarning, match="native front"):
        assert Q._native("vg_contains", Q._POINTS, Geometry, 0, ()) is None
    assert Q._front is False
    with pytest.raises(ValueError):  # the Python checks answer, and say why not
        Q.contains(Geometry, 0, ())
