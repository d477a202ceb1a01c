"""The build entry point compiles the torch-side module against the torch of the
interpreter that runs it (CPU; make itself is not run)."""
import subprocess
import sys

import __graft_entry__


def test_build_passes_its_interpreter(monkeypatch):
    commands = []
    monkeypatch.setattr(subprocess, "run", lambda args, **options: commands.append(args))
    __graft_entry__.build()
    package = next(c for c in commands if str(__graft_entry__.PKG) in c)
    assert f"PYTHON={sys.executable}" in package
