"""build() compiles the package's libraries whichever tests stand beside it."""
import concurrent.futures
import subprocess
import sys

import __graft_entry__ as entry
from anvil import export_hip


class _Serial:
    """A process pool that runs its work here."""

    def __init__(self, workers):
        pass

    def __enter__(self):
        return self

    def __exit__(self, *error):
        return False

    map = staticmethod(map)


def test_build_needs_no_test_module(monkeypatch, tmp_path, capsys):
    """Without tests/product_programs.py every other library is still built: the programs, the training
    attention's kernels and the exported function."""
    built = []
    monkeypatch.setattr(concurrent.futures, "ProcessPoolExecutor", _Serial)
    monkeypatch.setattr(entry, "_compile", lambda job: built.append(job[0]) or str(tmp_path / job[0]))
    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: built.append(cmd[-1].rsplit("/", 1)[-1]))
    monkeypatch.setattr(export_hip, "export", lambda ir, out, name: built.append(name) or [])
    monkeypatch.setitem(sys.modules, "product_programs", None)        # (an import of it then fails)
    entry.build()
    assert {*entry.PROGRAMS, *entry.FUNCTIONS, *entry.GRAPHED, "attn_train_check.so", "linear_lib"} <= set(built)
    assert "built product:" not in capsys.readouterr().out
