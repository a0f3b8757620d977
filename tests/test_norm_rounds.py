"""Frames shared by tasks whose starts agree modulo the hop but not modulo 4
hops (a quad of the raw log-mel): the planner shares them, the
normalisation's addressing finds every frame of such tasks across the quads of
the shared region (tests/rounds_host_driver.cpp, on the host, short and long
tasks, both workgroup forms), and on the GPU the features are bitwise those of
tasks that share nothing."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "scriptrs_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HOP = 160


def _windows(step, length, end):
    """Windows of `length` samples every `step` hops."""
    return [(s, length) for s in range(0, end, step * HOP)]


def _cases():
    rng = np.random.default_rng(19)
    cases = [
        _windows(101, 240_000, 3_200_000),       # 15 s windows every 1.01 s: all four shifts
        _windows(502, 240_000, 4_800_000),       # every 5.02 s: shifts 0 and 2
        _windows(303, 3000 * HOP + 17, 4_800_000),  # long items, segments that start and end anywhere
        [(s, 2049 * HOP + d) for s, d in zip(range(0, 400_000, 7 * HOP), range(-10 * HOP, 10_000, 53))],
    ]
    for _ in range(4):  # random starts on the hop, lengths at segment and chunk edges
        st = rng.integers(0, 5_000, 25) * HOP
        ln = rng.choice([33, 64, 127, 128, 512, 513, 1024, 2047, 2048, 2049, 2560, 2561, 4099, 33_000], 25) * HOP
        cases.append([(int(s), int(v + d)) for s, v, d in zip(st, ln, rng.integers(-170, 170, 25))])
    # and some off the hop among them
    cases.append([(s + (i % 3) * 5, v) for i, (s, v) in enumerate(cases[0])])
    return cases


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_addresses_of_shared_frames(tmp_path):
    exe = str(tmp_path / "rounds")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-x", "hip", "--cuda-host-only", "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "rounds_host_driver.cpp"),
                    os.path.join(CSRC, "sfe_share.cpp"), "-o", exe], check=True, stderr=subprocess.DEVNULL)
    cases = _cases()
    lines = []
    for c in cases:
        lines.append(str(len(c)))
        lines += [f"{s} {v}" for s, v in c]
    r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("bad 0"), r.stdout[-3000:] + r.stderr[-3000:]
    res = [ln.split() for ln in r.stdout.splitlines() if ln.startswith("case")]
    assert len(res) == len(cases)
    # one shared run: the union's quads, then at most 4 of each task's own
    with_, own, shifted = (int(res[0][i]) for i in (3, 4, 6))
    union = (cases[0][-1][0] + 240_000) / HOP / 4
    assert with_ <= union + 4 * len(cases[0]) < own / 8 and shifted >= 14, res[0]
    assert all(int(x[6]) > 0 for x in res[:-1]), res


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("case", range(9))
def test_shared_equals_own_on_the_gpu(extractor, case, dtype):
    import torch
    from scriptrs_amd import ChunkTask, synth
    spans = [(s, v) for s, v in _cases()[case] if v > HOP]
    rec = synth.speech_like(max(s + v for s, v in spans), 5)
    dev = torch.from_numpy(rec).cuda()
    tasks = [ChunkTask(s, s + v, s, 0) for s, v in spans]
    longest = max(v for _, v in spans) // HOP + 4
    bits = torch.int32 if dtype == "f32" else torch.int16
    try:
        extractor.set_frame_sharing(False)
        own, _ = extractor.extract_chunks(dev, tasks, dtype=dtype)
        own_pad, ff = extractor.extract_chunks_encoder_input(dev, tasks, target_frames=longest, dtype=dtype)
        extractor.set_frame_sharing(True)
        out, _ = extractor.extract_chunks(dev, tasks, dtype=dtype)
        pad, ff2 = extractor.extract_chunks_encoder_input(dev, tasks, target_frames=longest, dtype=dtype)
    finally:
        extractor.set_frame_sharing(True)
    assert torch.equal(out.view(bits), own.view(bits))
    assert np.array_equal(ff, ff2) and torch.equal(pad.view(bits), own_pad.view(bits))
