"""The native wrappers' module where it cannot serve: another torch build, a
file that does not load, a machine without a C++ compiler.  The kernels' own
library and the Python path do not depend on it."""

from __future__ import annotations

import subprocess
import sys

import pytest
import torch

from conftest import ROOT

from starter_amd import build
from starter_amd.kernels import _lib
from starter_amd.kernels.rmsnorm import rms_norm


def test_a_file_that_does_not_load_leaves_calls_to_the_wrappers(tmp_path, monkeypatch):
    broken = tmp_path / _lib.HOST_CALLS.name
    broken.write_bytes(b"not a library")
    monkeypatch.setattr(_lib, "HOST_CALLS", broken)
    monkeypatch.setattr(_lib, "_host", None)
    with pytest.warns(RuntimeWarning, match="does not load"):
        with pytest.raises(ValueError, match="BF16"):  # the wrapper's own refusal of CPU tensors
            rms_norm(torch.ones(2, 8), torch.ones(8), 1e-6)
    assert isinstance(_lib.host(), _lib._NoHostCalls)  # and no second warning


@pytest.mark.parametrize("attribute", [None, "__version__", "git_version"])
def test_only_the_torch_it_was_built_for_loads_it(attribute):
    """In a process of its own: a module of this kind is initialised once per process."""
    code = f"""
import sys, warnings
sys.path.insert(0, {str(ROOT)!r})
import torch.version
if {attribute!r}:
    setattr(torch.version, {attribute!r}, "another")
from starter_amd.kernels import _lib
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    native = not isinstance(_lib.host(), _lib._NoHostCalls)
print(native, any("built for torch" in str(w.message) for w in seen))
"""
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, check=True)
    assert out.stdout.split()[-2:] == (["False", "True"] if attribute else ["True", "False"])


@pytest.mark.parametrize("broken", ["compiler", "torch", None])
def test_the_library_is_linked_without_it(broken, tmp_path, monkeypatch, capsys):
    """Commands are recorded, not run: each leaves its output file."""
    def run(cmd, verbose):
        if broken == "compiler" and cmd[0] == "g++":
            raise FileNotFoundError("g++")
        (tmp_path / cmd[cmd.index("-o") + 1]).write_text("")

    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "_cxx", lambda: "g++")
    monkeypatch.setattr(build, "hipcc", lambda: "/opt/rocm/bin/hipcc")
    if broken == "torch":
        monkeypatch.setattr(build.importlib.util, "find_spec", lambda name: None)
    for name, file in (("LIBRARY", "lib.so"), ("PHASES_LIBRARY", "phases.so"), ("HOST_CALLS", "host.so")):
        monkeypatch.setattr(build, name, tmp_path / file)
    monkeypatch.setattr(build, "OBJ_DIR", tmp_path / "objects")
    (tmp_path / "host.so").write_text("an older build's")
    assert build.build() == tmp_path / "lib.so"
    assert (tmp_path / "lib.so").exists() and (tmp_path / "phases.so").exists()
    assert (tmp_path / "host.so").exists() == (broken is None)
    assert ("is not built" in capsys.readouterr().err) == (broken is not None)
