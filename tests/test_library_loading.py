"""What a library that is missing, or was built for other operator schemas, is reported as."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

import pytest

from tests.conftest import PACKAGE, ROOT, import_package

# An operator's implementation on the GPU, reached with CPU tensors by naming its dispatch key.
_USE = f"""
import importlib
import torch
vgo = importlib.import_module("{PACKAGE}")
lib = importlib.import_module("{PACKAGE}._lib")
keys = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
calls = [lib.load, lambda: torch.ops.vgo.csr_build.default.redispatch(keys, torch.zeros(3, dtype=torch.int32), 4)]
for call in calls:
    try:
        call()
    except lib.ExtensionUnavailable as error:
        print("unavailable:", error)
    except RuntimeError as error:
        print("other:", error)
"""


def _run(tmp_path, *libraries, edit=None):
    package = tmp_path / PACKAGE
    shutil.copytree(ROOT / PACKAGE, package, ignore=shutil.ignore_patterns("*.so", "_build", "__pycache__", "csrc"))
    for library in libraries:
        shutil.copy(library, package)
    if edit is not None:
        ops = (package / "ops.py").read_text()
        assert edit[0] in ops
        (package / "ops.py").write_text(ops.replace(*edit))
    env = dict(os.environ, PYTHONPATH=str(tmp_path), HIP_VISIBLE_DEVICES="-1")
    return subprocess.run([sys.executable, "-c", _USE], cwd=tmp_path, env=env, capture_output=True, text=True,
                          timeout=300)


def _built():
    lib = import_package("_lib")
    if not (lib.LIBRARY_PATH.exists() and lib.OPS_LIBRARY_PATH.exists()):
        pytest.skip("the library is not built")
    return lib.LIBRARY_PATH, lib.OPS_LIBRARY_PATH


@pytest.mark.parametrize("present", [0, 1])
def test_a_library_that_is_not_built(tmp_path, present):
    done = _run(tmp_path, *(_built()[:present] if present else ()))
    assert done.returncode == 0, done.stderr
    lines = done.stdout.splitlines()
    assert len(lines) == 2 and all("unavailable:" in line and "is not built (run __graft_entry__.build())" in line
                                   for line in lines), done.stdout


def test_a_library_of_other_schemas(tmp_path):
    """The process that imports the package goes on (build() is one), and each use says what to do."""
    done = _run(tmp_path, *_built(), edit=("csr_build(Tensor keys, int n_buckets)", "csr_build(Tensor keys)"))
    assert done.returncode == 0, done.stderr
    assert done.stdout.startswith("unavailable: vgo torch operators were built for other operator schemas")
    assert "csr_build" in done.stdout


def test_a_built_library_loads(tmp_path):
    done = _run(tmp_path, *_built())
    assert done.returncode == 0 and "unavailable" not in done.stdout, done.stdout + done.stderr
    assert "CPU tensor" in done.stdout  # the implementation itself answers
