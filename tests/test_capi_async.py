"""What the C ABI's host code leaves behind while a call's work is queued
(table staging, device tables, order across streams), over a host stand-in of
the HIP runtime whose streams run as late as they may
(tests/capi_async_driver.cpp).  No GPU is used."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "scriptrs_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("async") / "capi_async")
    subprocess.run([HIPCC, "-O1", "-g", "-std=c++17", "-x", "hip", "--cuda-host-only", "-ffp-contract=off",
                    "-Wno-unused-command-line-argument", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(ROOT, "tests", "capi_async_driver.cpp"),
                    *(os.path.join(CSRC, s) for s in ("sfe_capi.cpp", "sfe_share.cpp", "sfe_tables.cpp")),
                    "-lpthread", "-o", exe], check=True, stderr=subprocess.DEVNULL)
    return exe


@pytest.mark.parametrize("scenario", ["turns", "streams", "grow", "mixed", "ahead", "failed", "memory"])
def test_queued_calls(driver, scenario):
    r = subprocess.run([driver, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("bad 0"), r.stdout[-3000:] + r.stderr[-3000:]
