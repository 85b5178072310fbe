"""kraken_amd.torch_embedding without the built libraries: what needs no table works, and a table says
what is missing. Runs without a GPU."""
import glob
import os
import shutil
import subprocess
import sys

import pytest

pytest.importorskip("torch")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import torch
from kraken_amd import torch_embedding as te
jt = te.JaggedTensor.from_list_tensors([torch.ones(2, 3), torch.zeros(4, 3)])
assert jt.offsets().tolist() == [0, 2, 6]
try:
    te.Embedding(4)
except RuntimeError as e:
    assert "libkraken_hip.so is missing" in str(e), e
else:
    raise AssertionError("a table without a library")
"""


def test_module_imports_without_the_built_libraries(tmp_path):
    package = tmp_path / "kraken_amd"
    package.mkdir()
    for f in glob.glob(os.path.join(ROOT, "kraken_amd", "*.py")):
        shutil.copy(f, package)
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=tmp_path, capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, PYTHONPATH=str(tmp_path)))
    assert r.returncode == 0, r.stderr
