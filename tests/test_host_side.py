"""What the library and its C++ mirror ask of the HIP runtime, and in which order, checked without a GPU: fake_hip_checks.cpp
stands in for the runtime and makes it fail where a check wants that."""
import re
import subprocess
from pathlib import Path

import pytest

import bitnet_hip as bh

SOURCE = Path(__file__).with_name("fake_hip_checks.cpp")
CHECKS = re.findall(r'^    \{"(\w+)", \1\},$', SOURCE.read_text(), flags=re.M)


@pytest.fixture(scope="session")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host_side") / "checks"
    lib = bh.LIB_PATH.parent
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(SOURCE), "-o", str(exe), "-rdynamic",
                    f"-L{lib}", "-lbitnet_hip", "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{lib}"], check=True)
    return exe


@pytest.mark.parametrize("name", CHECKS)
def test_host_side(program, name):
    done = subprocess.run([str(program), name], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
