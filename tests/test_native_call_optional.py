"""Launchers are called by ctypes where ``csrc/host/ome_call.cpp`` was not built or does not load."""
import sysconfig

import pytest

from ome_amd import build
from ome_amd.ops import _native as N


def test_a_module_that_does_not_load_leaves_ctypes(monkeypatch, tmp_path, caplog):
    """A truncated copy, or one of another Python (its name tells them apart): the import of the operators does not fail."""
    assert sysconfig.get_config_var("SOABI") in N.lib_path(N.CALLER).name
    monkeypatch.setattr(N, "lib_path", lambda name: tmp_path / f"lib{name}.so")
    assert N._load_caller() is None and not caplog.records
    N.lib_path(N.CALLER).write_bytes(b"\x7fELF cut off")
    assert N._load_caller() is None
    assert ["does not load" in r.getMessage() for r in caplog.records] == [True]


@pytest.mark.parametrize("lacks", ["machine", "compiler", "headers"])
def test_a_build_does_without_it(monkeypatch, tmp_path, lacks):
    if lacks == "machine":
        monkeypatch.setattr(build.platform, "machine", lambda: "aarch64")
    elif lacks == "compiler":
        monkeypatch.setattr(build.shutil, "which", lambda name: None)
    else:
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build(verbose=False, only=("ome_call",)) == []
