"""build() makes the reference's binaries only where its sources are: a folder of
that name with nothing in it is no reason to fail."""
import os
import sys
import types

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("sources", [False, True])
def test_build_without_reference_sources(monkeypatch, tmp_path, sources):
    monkeypatch.syspath_prepend(REPO)
    import __graft_entry__ as entry

    if sources:
        (tmp_path / "cg.F90").write_text("")
    made = []
    monkeypatch.setattr(entry, "REF_SRC", str(tmp_path))
    monkeypatch.setitem(sys.modules, "build_lib", types.SimpleNamespace(build=lambda: made.append("library")))
    monkeypatch.setattr(entry.subprocess, "run", lambda cmd, **kw: made.append(cmd[cmd.index("-C") + 1]))
    entry.build()
    ref = os.path.join(REPO, "oracle", "ref")
    assert made == ["library", os.path.join(REPO, "oracle")] + ([ref, ref] if sources else [])
