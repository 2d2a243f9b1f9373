"""build() compiles the library whatever state tests/cpp is in: absent, of a
revision without the targets asked for, or not writable."""
import os
import subprocess

import pytest

import __graft_entry__ as entry

OLD_MAKEFILE = "all:\n\t@true\n"                       # no metal_ops target
BLOCKED_MAKEFILE = "metal_ops all:\n\tmkdir _bin\n"    # its output folder cannot be made


@pytest.mark.parametrize("makefile", [None, OLD_MAKEFILE, BLOCKED_MAKEFILE],
                         ids=["no-tests", "other-revision", "not-writable"])
def test_build_does_not_hang_on_test_binaries(tmp_path, monkeypatch, capfd, makefile):
    """The library's own makes are recorded instead of run (their result is the
    in-tree build), everything under tests/ runs for real in a scratch tree."""
    run, library = subprocess.run, []

    def fake(cmd, **kw):
        where = cmd[cmd.index("-C") + 1]
        if os.path.join(str(tmp_path), "tests") in where:
            return run(cmd, **kw)
        library.append(os.path.relpath(where, tmp_path))
        return subprocess.CompletedProcess(cmd, 0)

    if makefile is not None:
        cpp = tmp_path / "tests" / "cpp"
        cpp.mkdir(parents=True)
        (cpp / "Makefile").write_text(makefile)
        (cpp / "_bin").write_text("in the way")
    monkeypatch.setattr(entry, "ROOT", str(tmp_path))
    monkeypatch.setattr(entry, "REFERENCE", str(tmp_path / "reference"))
    monkeypatch.setattr(subprocess, "run", fake)
    entry.build()
    assert library == ["lite_ssm_amd/csrc", "oracle"]
    assert "test binaries" in capfd.readouterr().err
