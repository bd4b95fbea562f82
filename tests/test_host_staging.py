"""Transfers of large pageable arrays (runtime/host_staging.cpp) without a GPU: the source compiled against stand-ins for the HIP calls
it makes (host_staging_probe.cpp).  Sizes around a chunk and around the ring, several arrays in a row, a link that lags behind;
page-locked memory, events, threads that cannot be had; a transfer that fails half-way and the ones after it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("staging") / "host_staging_probe")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    os.path.join(ROOT, "tests", "host_staging_probe.cpp"), "-lpthread", "-o", out], check=True)
    return out


@pytest.mark.parametrize("case", ["sizes", "no_page_locked_memory", "no_events", "failed_transfer", "no_memory_for_threads"])
def test_staged_transfers(probe, case):
    r = subprocess.run([probe, case], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
