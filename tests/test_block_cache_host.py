"""CPU test of the device-block cache's tables and waits, on a runtime made of
counters (tests/cpp/block_cache.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def runner(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("block_cache") / "block_cache")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", os.path.join(HERE, "cpp", "block_cache.cpp"),
                    "-o", out], check=True)
    return out


@pytest.mark.parametrize("case", ["others_go_on", "failed_wait", "full_device", "sizes"])
def test_block_cache(runner, case):
    r = subprocess.run([runner, case], stdout=subprocess.PIPE, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n")
