"""The log-mel kernel's 32 x 16 real FFT, mel schedule and raw layout
(scriptrs_amd/csrc/sfe_fft.hpp, sfe_tables.cpp, sfe_internal.hpp) run on the
host by tests/rdft_host_driver.cpp, at sample rates of both mel schedules.
No GPU is used."""
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
    exe = str(tmp_path_factory.mktemp("rdft") / "rdft_host")
    # host arithmetic exactly as written: fmaf where the header fuses, no
    # other contraction
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", "-ffp-contract=off",
                    "-Wno-unused-command-line-argument", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(ROOT, "tests", "rdft_host_driver.cpp"), os.path.join(CSRC, "sfe_tables.cpp"),
                    "-o", exe], check=True, stderr=subprocess.DEVNULL)
    return exe


@pytest.mark.parametrize("rate", [3500, 8000, 16000, 22050, 24000, 44100, 107000])
def test_real_fft_and_mel_tables(driver, rate):
    r = subprocess.run([driver, str(rate)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and "bad 0" in r.stdout, r.stdout + r.stderr
