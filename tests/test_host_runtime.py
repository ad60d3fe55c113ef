"""The library's host code over a stand-in for the HIP runtime (tests/standin), on the CPU: which
launches, copies, allocations and waits a call makes, where what they must be cannot be seen on a
GPU without provoking a fault or a race."""
import glob
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "tpchq01_gpu_amd", "csrc")
STANDIN = os.path.join(HERE, "standin")
HOST = ["-O1", "-fPIE", "-std=c++17", "-Wno-unused-result", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__"]
CASES = re.findall(r'^    \{"(\w+)", \w+\},$', open(os.path.join(STANDIN, "host_cases.cpp")).read(), re.M)


@pytest.fixture(scope="module")
def host_cases(tmp_path_factory):
    """The library's sources without their device code, the stand-in and the cases, as one program."""
    out = str(tmp_path_factory.mktemp("standin"))

    def compile_one(src):
        obj = os.path.join(out, os.path.basename(src) + ".o")
        if src.endswith(".hip"):
            cmd = ["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-fPIE", "-std=c++17", "-w"]
        else:
            cmd = ["g++", *HOST]
        subprocess.run([*cmd, "-c", src, "-o", obj], check=True)
        return obj

    sources = [s for s in glob.glob(os.path.join(CSRC, "q1_*.hip")) + glob.glob(os.path.join(CSRC, "q1_*.cpp"))]
    with ThreadPoolExecutor(4) as pool:
        objs = list(pool.map(compile_one, sources + glob.glob(os.path.join(STANDIN, "*.cpp"))))
    exe = os.path.join(out, "host_cases")
    # the device code's images stay undefined: nothing reads them
    subprocess.run(["g++", "-o", exe, *objs, "-Wl,--unresolved-symbols=ignore-in-object-files", "-lpthread", "-ldl"],
                   check=True)
    return exe


def test_every_case_is_listed(host_cases):
    assert sorted(CASES) == subprocess.run([host_cases], capture_output=True, text=True).stdout.split()


@pytest.mark.parametrize("name", CASES)
def test_host_code(host_cases, name):
    p = subprocess.run([host_cases, name], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
