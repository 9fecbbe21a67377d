"""Parts of the library that are plain C++, checked on the host
(host_units.cpp): buffers that grow, with an allocator that can fail, and the
levels of a tree's leaves."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def units(tmp_path_factory):
    exe = tmp_path_factory.mktemp("units") / "host_units"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", f"-I{ROOT / 'research_codes_amd' / 'csrc'}",
                    str(ROOT / "tests" / "host_units.cpp"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("name", ["node_buffers", "list_rooms", "leaf_levels"])
def test_host_unit(units, name):
    r = subprocess.run([str(units), name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
