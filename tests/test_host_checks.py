"""Host code of the library on the CPU, with the HIP runtime's calls replaced (native/host_checks.cpp): what happens when an allocation or a
launch fails, and which calls go to which kernel."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "sparseconvnet_amd", "libscn_hip.so")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc) or not os.path.exists(LIB):
        pytest.skip("no compiler or no built library")
    out = str(tmp_path_factory.mktemp("native") / "host_checks")
    subprocess.check_call([hipcc, "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-O1", "-rdynamic", "-x", "hip",
                           os.path.join(HERE, "native", "host_checks.cpp"), "-x", "none", LIB, "-Wl,-rpath," + os.path.dirname(LIB), "-o", out])
    return out


@pytest.mark.parametrize("name", ["failed_allocation", "identity_tables", "wave_refuses", "counts_under_capture"])
def test_host_code(program, name):
    r = subprocess.run([program, name], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=60)
    assert r.returncode == 0, r.stdout.decode()
