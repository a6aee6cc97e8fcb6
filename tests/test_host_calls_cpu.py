"""The native wrappers' module where it cannot serve: another torch build, or a
file that does not load.  The kernels' own library and the Python path do not
depend on it."""

from __future__ import annotations

import subprocess
import sys

import pytest
import torch

from conftest import ROOT

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
