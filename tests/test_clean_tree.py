"""A checkout where nothing is built: the package and everything that builds it import without a library, and the build
command reaches the compiler."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def clean_tree(tmp_path_factory):
    to = tmp_path_factory.mktemp("clean")
    skip = shutil.ignore_patterns("lib", "__pycache__")
    for part in ("turboexl3_amd", "include"):
        shutil.copytree(os.path.join(ROOT, part), to / part, ignore=skip)
    shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), to / "__graft_entry__.py")
    return to


def python(tree, *args, **env):
    return subprocess.run([sys.executable, *args], cwd=tree, capture_output=True, text=True, timeout=300,
                          env={**os.environ, "PYTHONPATH": str(tree), **env})


def test_every_module_imports_and_a_call_names_what_is_missing(clean_tree):
    got = python(clean_tree, "-c", """
import torch, turboexl3_amd
from turboexl3_amd import _lib, api, build, pack, table
assert not __import__("os").path.exists(_lib.LIB_PATH)
t, v = torch.zeros(8, 8, 64, dtype=torch.int16), torch.ones(128, dtype=torch.float16)
try:
    api.linear(torch.zeros(1, 128), t, v, v)
except RuntimeError as e:
    assert "python -m turboexl3_amd.build" in str(e), e
else:
    raise AssertionError("a call without the library went through")
""")
    assert got.returncode == 0, got.stderr


@pytest.mark.parametrize("args", [("-m", "turboexl3_amd.build"), ("-c", "import __graft_entry__ as g; g.build()")])
def test_the_build_commands_reach_the_compiler(clean_tree, args):
    # a compiler that always fails stands for the real one, which takes minutes
    got = python(clean_tree, *args, HIPCC=shutil.which("false"), PATH="")
    assert got.returncode != 0 and "hipcc failed on t3_dense.hip" in got.stderr, got.stderr
