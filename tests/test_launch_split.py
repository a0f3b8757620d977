"""Calls of more workgroups than one launch holds (2^32 threads): the split
into launches on the host (tests/launch_split_driver.cpp), and on the GPU
batches of more clips than one normalisation launch takes in its 8-wave and
4-wave forms, which such a launch left unwritten without an error.  The driver also pins the
rule that picks the form.  Short clips of one length take the 4-wave form, which
is up to a quarter faster there (300 clips of 0.5 s 16 against 21 us)."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "scriptrs_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_launches_cover_every_workgroup(tmp_path):
    exe = str(tmp_path / "split")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-x", "hip", "--cuda-host-only", "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "launch_split_driver.cpp"),
                    "-o", exe], check=True, stderr=subprocess.DEVNULL)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "bad 0", r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("n,sizes", [((1 << 20) + 5, [163]), ((1 << 21) + 5, [3, 500, 10, 90, 161])])
def test_more_clips_than_one_launch_holds(extractor, n, sizes):
    """Clips of one length (8 workgroups of 512 threads each) and of 1 to 4
    frames (256): past 2^32 threads the features are those of the same clips in
    smaller calls.  (Compared as bits: clips of one frame are NaN.)"""
    import torch
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of free GPU memory")
    off = np.zeros(n + 1, np.int64)
    np.cumsum(np.resize(sizes, n), out=off[1:])
    x = torch.randn(int(off[-1]), device="cuda", generator=torch.Generator(device="cuda").manual_seed(20))
    fo = off * 0
    np.cumsum(np.diff(off) // 160 + 1, out=fo[1:])
    out = torch.full((int(fo[-1]) * 128,), 1e30, device="cuda")
    extractor.extract_batch(x, off, out=out)
    step = 500_000
    for i in range(0, n, step):
        o, f = off[i:i + step + 1], fo[i:i + step + 1]
        got, _ = extractor.extract_batch(x[int(o[0]):int(o[-1])], o - o[0])
        assert torch.equal(got.view(torch.int32), out[128 * int(f[0]):128 * int(f[-1])].view(torch.int32)), i


@pytest.mark.gpu
def test_long_item_among_more_clips_than_one_launch_holds(extractor):
    """The same with a clip past 2048 frames in front, whose segments come
    first in the launch."""
    import torch
    n, size = (1 << 21) + 5, 161
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of free GPU memory")
    lens = np.full(n, size)
    lens[7] = 160 * 3000
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    x = torch.randn(int(off[-1]), device="cuda", generator=torch.Generator(device="cuda").manual_seed(21))
    out, fo = extractor.extract_batch(x, off)
    for i, j in ((0, 100), (n // 2, n // 2 + 1000), (n - 1000, n)):
        o = off[i:j + 1]
        got, _ = extractor.extract_batch(x[int(o[0]):int(o[-1])], o - o[0])
        assert torch.equal(got, out[128 * int(fo[i]):128 * int(fo[j])]), i
