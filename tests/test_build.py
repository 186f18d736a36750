"""Building and loading the native host path beside the library (CPU only): a
host module that cannot be built or imported is reported and costs nothing else."""

import os
import shutil
import sys
import warnings

import pytest

import sparda
from sparda import _lib
from sparda import build as B


@pytest.mark.skipif(shutil.which(B.HIPCC) is None and not os.path.exists(B.HIPCC), reason="hipcc not available")
def test_the_library_is_linked_without_the_host_module(monkeypatch, tmp_path):
    def no_compiler():
        raise FileNotFoundError("g++")

    src = tmp_path / "one.hip"
    src.write_text('extern "C" int one() { return 1; }\n')
    stale = tmp_path / "_host.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(B, "sources", lambda: [str(src)])
    monkeypatch.setattr(B, "OBJ_DIR", str(tmp_path))
    monkeypatch.setattr(B, "LIB_PATH", str(tmp_path / "lib.so"))
    monkeypatch.setattr(B, "HOST_PATH", str(stale))
    monkeypatch.setattr(B, "_build_host", no_compiler)
    with pytest.warns(RuntimeWarning, match="not built.*g\\+\\+"):
        assert B.build() == str(tmp_path / "lib.so")
    assert os.path.exists(tmp_path / "lib.so") and not stale.exists()


def test_a_host_module_that_does_not_import_is_reported(monkeypatch, tmp_path):
    there = tmp_path / "_host.so"
    monkeypatch.setattr(_lib, "HOST_PATH", str(there))
    monkeypatch.setitem(sys.modules, "sparda._host", None)
    monkeypatch.delattr(sparda, "_host", raising=False)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert isinstance(_lib.load_host(), _lib._NoHost)  # never built
    there.write_bytes(b"")
    with pytest.warns(RuntimeWarning, match="cannot be imported"):
        assert isinstance(_lib.load_host(), _lib._NoHost)
