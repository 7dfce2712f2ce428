"""The build's own decisions, with a stand-in for the compiler."""
import subprocess
import types

from turboexl3_amd import build


def test_another_torch_rebuilds_the_binding(tmp_path, monkeypatch):
    import torch

    runs = []

    def compiler(cmd, **_):
        runs.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return types.SimpleNamespace(returncode=0, stdout="", stderr="")

    monkeypatch.setattr(subprocess, "run", compiler)
    monkeypatch.setattr(build, "OBJDIR", str(tmp_path))
    build._compile_torch(False)
    build._compile_torch(False)
    assert len(runs) == 1  # the second found its object
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    build._compile_torch(False)
    assert len(runs) == 2
    build._compile_torch(False)
    assert len(runs) == 2
