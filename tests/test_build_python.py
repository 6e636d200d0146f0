"""The extension module is built for the interpreter that asks for the build, where it has what the source needs; the library and the tools are built in any case."""
import os
import subprocess
import sys
import sysconfig

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def would_build(tmp_path, version=None):
    """What `make all` would run, for this interpreter or one that says it is of `version`."""
    python = tmp_path / "python"
    pretend = f"import sysconfig; sys.version_info = {version}; " if version else ""
    python.write_text(f"#!/bin/sh\nexec {sys.executable} -c \"import sys; {pretend}exec(sys.argv[1])\" \"$2\"\n")
    python.chmod(0o755)
    out = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "smat_amd", "csrc"), "all", f"PYTHON={python}"], check=True, capture_output=True, text=True).stdout
    assert "libsmat_amd.so" in out and "hgemm" in out
    return out


@pytest.mark.parametrize("version", [(3, 6, 9), (3, 8, 20)])
def test_no_extension_module_for_an_interpreter_without_its_calls(tmp_path, version):
    assert "/_call" not in would_build(tmp_path, version)


def test_extension_module_of_this_interpreter(tmp_path):
    if not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")):
        pytest.skip("no Python.h")
    assert "/_call" + sysconfig.get_config_var("EXT_SUFFIX") in would_build(tmp_path)


def test_source_uses_no_later_calls():
    """Public since 3.9: vectorcall and its methods.  Py_NewRef came with 3.10."""
    with open(os.path.join(ROOT, "smat_amd", "csrc", "python", "call.cpp")) as f:
        assert "Py_NewRef" not in f.read()


def test_build_asks_for_the_interpreter_that_runs_it(monkeypatch):
    import __graft_entry__ as entry
    calls = []
    monkeypatch.setattr(entry.subprocess, "run", lambda cmd, **kw: calls.append(cmd))
    entry.build()
    assert any("csrc" in " ".join(c) and f"PYTHON={sys.executable}" in c for c in calls if "clean" not in c)
