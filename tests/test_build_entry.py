"""__graft_entry__.build(): the library comes first, depends on nothing under tests/, and a failure says what failed."""
import subprocess
import types

import pytest

import __graft_entry__ as entry


def _fake_make(monkeypatch, status):
    calls = []

    def run(cmd, **kw):
        calls.append((cmd, kw))
        return types.SimpleNamespace(returncode=status, stdout="the compiler's words\n")

    monkeypatch.setattr(subprocess, "run", run)
    return calls


def test_build_makes_the_library_first_and_no_test_program(monkeypatch):
    calls = _fake_make(monkeypatch, 0)
    entry.build()
    folders = [cmd[cmd.index("-C") + 1] for cmd, _ in calls]
    assert folders[0].endswith("lumen_amd/csrc") and "-B" in calls[0][0]
    assert not any("tests" in f[len(entry.ROOT):] for f in folders), folders


def test_a_failed_build_shows_what_it_printed(monkeypatch, capsys):
    calls = _fake_make(monkeypatch, 2)
    with pytest.raises(RuntimeError, match="csrc"):
        entry.build()
    assert len(calls) == 1
    assert "the compiler's words" in capsys.readouterr().err
