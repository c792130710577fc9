"""The C++ test clients find the library of the tree they lie in (CPU)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("client,lib", [("client", "lib"), ("client_asan", "lib/asan")])
def test_client_uses_its_own_tree(tmp_path, client, lib):
    built = os.path.join(ROOT, "tests", "cpp", client)
    assert os.path.exists(built), f"tests/cpp/{client} not built: run __graft_entry__.build()"
    (tmp_path / "tests" / "cpp").mkdir(parents=True)
    there = tmp_path / "mgpu_old_amd" / lib
    there.mkdir(parents=True)
    shutil.copy(built, tmp_path / "tests" / "cpp" / client)
    os.symlink(os.path.join(ROOT, "mgpu_old_amd", lib, "libmgpusort.so"), there / "libmgpusort.so")
    out = subprocess.run(["ldd", str(tmp_path / "tests" / "cpp" / client)], capture_output=True,
                         text=True, check=True).stdout
    line = next(x for x in out.splitlines() if "libmgpusort.so" in x)
    found = line.split("=>")[1].split(" (")[0].strip()
    assert os.path.normpath(found) == str(there / "libmgpusort.so"), out
