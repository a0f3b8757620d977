"""Constant rows (digital silence; filters that hold no bin at sample rates
past 24 kHz): the closed form of the reference's sequential f32 sums
(scriptrs_amd/csrc/sfe_seqsum.hpp) is the loop's result bit for bit, and takes
rows of 2^30 values in a few hundred operations
(tests/seqsum_host_driver.cpp, on the host); on the GPU, silent clips of every
form of the normalisation have the oracle's loops' statistics."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "scriptrs_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_sequential_sum_is_the_loop(tmp_path):
    exe = str(tmp_path / "seqsum")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--cuda-host-only", "-ffp-contract=off",
                    "-Wno-unused-command-line-argument", "-I", CSRC,
                    os.path.join(ROOT, "tests", "seqsum_host_driver.cpp"), "-o", exe],
                   check=True, stderr=subprocess.DEVNULL)
    # (the 2^30-value rows alone would take the loop 20,000 x 1 s)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("bad 0"), r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("frames", [[2], [63, 1024, 1500, 2048], [2049, 12, 9001], [40_000],
                                    [500 + (37 * i) % 1400 for i in range(120)]])
def test_silent_clips_against_the_oracle(extractor, frames):
    """Few items (8 waves), 120 ragged ones (4 waves) and long ones (segments).
    One ulp of the row's sum moves x - mean by a whole ulp of the sum over T:
    at least 2^-12 of x - mean at these lengths, so sums that differ do not
    pass.  The bar, 2 ulps, leaves the device's square root one."""
    import oracle
    import torch
    off = np.concatenate([[0], np.cumsum([(t - 1) * 160 + 3 for t in frames])])
    out, fo = extractor.extract_batch(torch.zeros(int(off[-1]), device="cuda"), off)
    got = out.cpu().numpy()
    for i, t in enumerate(frames):
        want = oracle.extract(np.zeros(int(off[i + 1] - off[i]), np.float32))
        np.testing.assert_allclose(got[128 * fo[i]:128 * fo[i + 1]].reshape(128, t), want.reshape(128, t),
                                   rtol=2.0**-22, atol=0, err_msg=str(t))
