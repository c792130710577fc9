"""A tests folder put in the place of another without the built C++ clients gets
them when its tests are run (CPU)."""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT


def test_clients_of_a_replaced_tests_folder(tmp_path):
    if not os.path.exists(os.path.join(ROOT, "mgpu_old_amd", "lib", "noalloc.o")):
        pytest.skip("the normal build has not run (no noalloc.o)")
    ignore = shutil.ignore_patterns("__pycache__", "client", "client_asan", "asan")
    for part in ("mgpu_old_amd", "include", "tests"):
        shutil.copytree(os.path.join(ROOT, part), tmp_path / part, ignore=ignore)
    for part in ("__graft_entry__.py", "conftest.py"):
        if os.path.exists(os.path.join(ROOT, part)):
            shutil.copy(os.path.join(ROOT, part), tmp_path / part)
    run = subprocess.run([sys.executable, "-m", "pytest", "-q", "-p", "no:cacheprovider",
                          "tests/test_client_build.py"], cwd=tmp_path, capture_output=True,
                         text=True, timeout=300)
    assert run.returncode == 0, run.stdout[-3000:] + run.stderr[-3000:]
