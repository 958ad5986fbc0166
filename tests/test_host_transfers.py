"""HostTransfers (fluxo_amd/csrc/fx_hostcopy.hpp), compiled for the host against stand-ins for the HIP
calls it makes (tests/hostcopy): the conditions a single GPU cannot give."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostcopy") / "check")
    src = os.path.join(HERE, "hostcopy")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I" + src,
                    "-I" + os.path.join(HERE, "..", "fluxo_amd", "csrc"), os.path.join(src, "check.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("check", ["other_device", "workers_where_they_repay", "sizes", "no_memory"])
def test_host_transfers(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
