"""A library of another version, or one without the newest entry points, is refused with the
remedy, not with a missing symbol."""
from __future__ import annotations

import subprocess

import pytest

from winnow_amd import _lib


@pytest.mark.parametrize("source,says", [
    ("int wn_abi_version(void) { return %d; }" % (_lib.ABI_VERSION - 1), f"has ABI {_lib.ABI_VERSION - 1}"),
    ("int wn_abi_version(void) { return %d; }" % _lib.ABI_VERSION, "lacks .*wn_append_split"),
    ("int other(void) { return 0; }", "has ABI None"),
])
def test_an_older_library(tmp_path, monkeypatch, source, says):
    (tmp_path / "old.c").write_text(source)
    path = tmp_path / "old.so"
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "old.c"), "-o", str(path)], check=True)
    monkeypatch.setattr(_lib, "LIB_PATH", path)
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.raises(_lib.HipLibraryMissing, match=says + ".*rebuild it"):
        _lib.lib()
    assert _lib._lib is None
