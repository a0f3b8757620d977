"""Every workgroup form and register class of the normalisation that a batch of
short items can take (csrc/sfe_internal.hpp, norm_wide): each clip's features
are bitwise those of the same clip in a small call of the other form, and a few
are the oracle's."""
import numpy as np
import pytest

import np_reference as R
from parity import assert_parity

pytestmark = pytest.mark.gpu


def _batch(frames, seed):
    import torch
    lens = np.array([160 * (t - 1) + (7 * i) % 160 for i, t in enumerate(frames)], np.int64)
    lens = np.maximum(lens, 1)
    off = np.concatenate([[0], np.cumsum(lens)])
    g = torch.Generator(device="cuda").manual_seed(seed)
    return 0.3 * torch.randn(int(off[-1]), device="cuda", generator=g), off


def _ragged(longest):
    """130 clips (more than 3 workgroups per CU on 256), their mean well below
    7/8 of the longest: the 4-wave form, in the class that holds `longest`
    (512, 1024, 1536 or 2048 frames)."""
    return [longest, 1, 2, 63, 64, 65] + [longest // 3 + (41 * i) % (longest // 2) for i in range(124)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("frames", [
    pytest.param(_ragged(256), id="ragged-256"),
    pytest.param(_ragged(512), id="ragged-512"),
    pytest.param(_ragged(513), id="ragged-513"),
    pytest.param(_ragged(1024), id="ragged-1024"),
    pytest.param(_ragged(1025), id="ragged-1025"),
    pytest.param(_ragged(1536), id="ragged-1536"),
    pytest.param(_ragged(1537), id="ragged-1537"),
    pytest.param(_ragged(2048), id="ragged-2048"),
    pytest.param([51] * 130, id="uniform-51"),      # 4 waves
    pytest.param([256] * 40, id="uniform-256"),     # 4 waves
    pytest.param([449] * 130, id="uniform-449"),    # 8 waves
    pytest.param([448] * 130, id="uniform-448"),    # 4 waves
])
def test_forms_and_classes_agree(extractor, frames, dtype):
    import oracle
    import torch
    x, off = _batch(frames, len(frames) + frames[0])
    bits = torch.int32 if dtype == "f32" else torch.int16
    out, fo = extractor.extract_batch(x, off, dtype=dtype)
    longest = max(frames)
    # small calls of up to 20 clips: 8 waves, as one of their clips is past 512
    # frames (appended where the batch has none)
    extra = x.new_zeros(160 * 600) if longest <= 512 else x.new_zeros(0)
    for i in range(0, len(frames), 20):
        o = off[i:i + 21] - off[i]
        part = torch.cat([x[int(off[i]):int(off[i] + o[-1])], extra])
        o2 = np.append(o, o[-1] + extra.numel()) if extra.numel() else o
        got, f = extractor.extract_batch(part, o2, dtype=dtype)
        n = 128 * int(f[len(o) - 1])
        assert torch.equal(got[:n].view(bits), out[128 * int(fo[i]):128 * int(fo[i]) + n].view(bits)), i
    for i in (0, len(frames) // 2, len(frames) - 1) if dtype == "f32" else ():
        c = x[int(off[i]):int(off[i + 1])].cpu().numpy()
        got = out[128 * int(fo[i]):128 * int(fo[i + 1])].cpu().numpy().reshape(128, -1)
        assert_parity(got, oracle.extract(c), R.extract(c), R.f32_noise_envelope(c), what=f"clip {i}")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("seconds", [1, 2, 5, 5.1])
def test_short_shifted_windows(extractor, seconds, dtype):
    """Short windows every 0.51 s share frames at all four shifts, in the 4-wave
    form."""
    import torch
    from scriptrs_amd import ChunkTask, synth
    n = int(16000 * seconds)
    rec = torch.from_numpy(synth.speech_like(16000 * 70, 3)).cuda()
    tasks = [ChunkTask(s, s + n, s, 0) for s in range(0, rec.numel() - n, 51 * 160)]
    bits = torch.int32 if dtype == "f32" else torch.int16
    try:
        extractor.set_frame_sharing(False)
        own, _ = extractor.extract_chunks(rec, tasks, dtype=dtype)
        extractor.set_frame_sharing(True)
        got, _ = extractor.extract_chunks(rec, tasks, dtype=dtype)
    finally:
        extractor.set_frame_sharing(True)
    assert torch.equal(got.view(bits), own.view(bits))
