"""The kernel library builds where its optional extension cannot."""
import subprocess

import pytest

from infurnace_amd import build


@pytest.mark.parametrize("failure", ["no compiler", "error"])
def test_library_builds_without_the_extension(monkeypatch, tmp_path, capsys, failure):
    """No g++, or headers it does not accept: the library is linked, a stale extension goes, and stderr says so."""
    for name in ("LIB_PATH", "FAST_PATH", "BUILD_DIR"):
        monkeypatch.setattr(build, name, str(tmp_path / name))
    (tmp_path / "FAST_PATH").write_text("stale")
    monkeypatch.setattr(build, "sources", lambda: [])

    def run(cmd, **kw):
        if cmd[0] == "g++":
            if failure == "no compiler":
                raise FileNotFoundError(cmd[0])
            return subprocess.CompletedProcess(cmd, 1, "", "no such header")
        if "-o" in cmd:
            open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", "")
    monkeypatch.setattr(build.subprocess, "run", run)
    assert build.build() == str(tmp_path / "LIB_PATH")
    assert (tmp_path / "LIB_PATH").exists() and not (tmp_path / "FAST_PATH").exists()
    assert "fast_call" in capsys.readouterr().err
