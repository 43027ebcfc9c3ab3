"""What a build needs: the library ROCm alone, the operators for Python torch and g++ as well."""
import shutil
import sys

import pytest

from guffin_amd import build


@pytest.mark.parametrize("missing", ["g++", "torch"])
def test_the_library_s_build_does_without(monkeypatch, tmp_path, missing, capsys):
    """It succeeds and says what is not there; operators of an older build, which another library may not fit, are gone."""
    stale = tmp_path / "_operators.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(build, "OPERATORS", str(stale))
    monkeypatch.setattr(build, "_library", lambda verbose: "the library")
    if missing == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)
    else:
        which = shutil.which
        monkeypatch.setattr(shutil, "which", lambda name, *a, **k: None if name == "g++" else which(name, *a, **k))
    assert build.build() == "the library" and not stale.exists()
    assert "no " + missing in capsys.readouterr().err
