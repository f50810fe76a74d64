"""Device memory of plans and one-call entry points, over a device made of counters (call_memory.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "seismic.jl_amd", "csrc")
SCENARIOS = ["reuse", "bounds", "given_back", "buffers_free_themselves", "growth_after_call", "call_at_the_limit",
             "host_memory", "many_devices"]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("mem") / "call_memory")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include", f"-I{CSRC}",
                    os.path.join(HERE, "call_memory.cpp"), os.path.join(CSRC, "swem_pool.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("name", SCENARIOS)
def test_scenario(program, name):
    r = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
