"""The large host copies (fsibe_2d_amd/csrc/transfer.hpp): what arrives, from
which size in each direction they replace the runtime's, and their threads when
the process forks or ends: a forked child, which has none of them, ends
normally, and a copy that a late destructor makes still arrives.  Compiled with
g++ on stand-ins for the HIP calls, so it runs with no GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"), "-o", exe, os.path.join(HERE, "cpp", "transfer_driver.cpp")],
                   check=True)
    return exe


@pytest.mark.parametrize("case", ["sizes", "lines", "fork", "fork_inside", "late"])
def test_copies_threads_and_process_ends(driver, case):
    r = subprocess.run([driver, case], capture_output=True, text=True, timeout=60)
    print(case, r.returncode, r.stdout, r.stderr)
    assert r.returncode == 0, r.stdout + r.stderr
