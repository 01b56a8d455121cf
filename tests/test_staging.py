"""The library's uploads through pinned slots, on a stand-in for the HIP runtime (staging_host.cpp): what needs several
devices, or streams held at will, and so cannot be shown on the one GPU the other tests have."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ancora-cutile_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if shutil.which(hipcc) is None or shutil.which("g++") is None:
        pytest.skip("no compiler")
    d = tmp_path_factory.mktemp("staging")
    subprocess.run([hipcc, "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-fPIC", "-c",
                    os.path.join(CSRC, "runtime.hip"), "-o", str(d / "runtime.o")], check=True)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(shutil.which(hipcc))))
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"), "-I/opt/rocm/include",
                    os.path.join(HERE, "staging_host.cpp"), str(d / "runtime.o"), "-pthread",
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(d / "staging")], check=True)
    return str(d / "staging")


@pytest.mark.parametrize("case", ["two_devices", "other_streams_do_not_wait", "many_threads", "capture", "streams_that_end",
                                  "now_waits_for_no_kernel", "memory_of_another_device", "errors_of_others", "past_the_end", "streams_of_others",
                                  "released_beside_an_upload"])
def test_uploads(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
