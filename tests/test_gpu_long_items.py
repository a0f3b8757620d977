"""Normalisation of items longer than a workgroup holds in registers (2048
frames), which goes in segments of 512 frames: item lengths at the edges of
the register budget, of segments and of the segment size itself (past 32768
frames a segment is 1024), alone and mixed with short items, against the
oracle; the padded layout, shared frames and digital silence."""
import numpy as np
import pytest

import np_reference as R
from parity import assert_parity

pytestmark = pytest.mark.gpu

HOP = 160


def _clips(frames, seed):
    from scriptrs_amd.synth import sinusoids
    return [sinusoids((t - 1) * HOP + 7 * i % HOP, seed + i) for i, t in enumerate(frames)]


@pytest.mark.parametrize("frames", [[2048], [2049], [2047, 2050, 17, 2559], [2560, 2561, 100, 2563, 4097],
                                    [32768], [32769, 600]])
def test_lengths_at_segment_edges(extractor, frames):
    import oracle
    import torch
    clips = _clips(frames, 50)
    off = np.concatenate([[0], np.cumsum([c.size for c in clips])])
    dev = torch.from_numpy(np.concatenate(clips)).cuda()
    out, fo = extractor.extract_batch(dev, off)
    got = out.cpu().numpy()
    for i, c in enumerate(clips):
        assert fo[i + 1] - fo[i] == frames[i]
        g = got[128 * fo[i]:128 * fo[i + 1]].reshape(128, frames[i])
        if frames[i] <= 8192:
            assert_parity(g.T, oracle.extract(c).T, R.extract(c).T, R.f32_noise_envelope(c).T,
                          what=f"{frames[i]} frames")
        else:
            # The oracle's sequential f32 sums over T values carry up to T u
            # |x| (T = 32768: 2e-3 |x|), past the flat bar, which float64 does
            # not: the bar of assert_parity against float64 alone.
            want, env = R.extract(c), R.f32_noise_envelope(c)
            assert np.all(np.abs(g - want) <= 1e-4 + 1e-3 * np.abs(want) + env), f"{frames[i]} frames"
        # a clip's features do not depend on the others of its call
        alone, _ = extractor.extract_batch(dev[off[i]:off[i + 1]].contiguous(), [0, c.size])
        assert np.array_equal(alone.cpu().numpy(), g.reshape(-1)), frames[i]


def test_long_items_shared_padded_and_silent(extractor):
    import oracle
    import torch
    from scriptrs_amd.long_form import ChunkTask
    x = _clips([9000], 70)[0]
    x[: 3000 * HOP] = 0.0
    dev = torch.from_numpy(x).cuda()
    # overlapping tasks on the sharing grid and off it, and one all silent
    spans = [(0, 2600 * HOP), (640 * 700, 640 * 700 + 3100 * HOP), (640 * 720, 640 * 720 + 2200 * HOP + 31),
             (HOP * 3001, HOP * 5601)]
    tasks = [ChunkTask(a, b, a, 0) for a, b in spans]
    out, fo = extractor.extract_chunks(dev, tasks)
    extractor.set_frame_sharing(False)
    own, _ = extractor.extract_chunks(dev, tasks)
    extractor.set_frame_sharing(True)
    assert torch.equal(out, own)
    pad, ff = extractor.extract_chunks_encoder_input(dev, tasks, target_frames=3500)
    noalloc, _ = extractor.extract_chunks_noalloc(dev, tasks)
    assert torch.equal(out, noalloc)
    got = out.cpu().numpy()
    for i, (a, b) in enumerate(spans):
        T = int(fo[i + 1] - fo[i])
        g = got[128 * fo[i]:128 * fo[i + 1]].reshape(128, T)
        p = pad[i].cpu().numpy()
        assert ff[i] == T and np.array_equal(p[:, :T], g) and not p[:, T:].any()
        want = oracle.extract(x[a:b])
        if not x[a:b].any():
            assert np.array_equal(g, want.reshape(128, T))  # digital silence: the reference's own rounding
        else:
            assert_parity(g.T, want.T, R.extract(x[a:b]).T, R.f32_noise_envelope(x[a:b]).T, what=f"task {i}")
