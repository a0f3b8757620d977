"""The pinned staging ring of the calls' tables on the GPU: calls with tables of
their own queued one after another without a host wait, so that the ring turns
over while uploads are in flight, grows, and is used from two streams; every
output against the same call alone on another context.  (The host's side of it
is tests/test_capi_async.py.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _calls(counts, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in counts:
        lens = rng.integers(200, 1500, n) if n > 4 else rng.integers(340_000, 400_000, n)
        out.append(np.concatenate([[0], np.cumsum(lens)]).astype(np.int64))
    return out


# (160 bytes a clip: a half of the ring holds about 8,200 clips at first)
@pytest.mark.parametrize("streams,counts", [
    (1, [3000, 7, 3100, 2900, 3, 3050, 40, 2800, 3200, 900, 3000, 2, 3150, 3010]),
    (2, [8000, 5, 8100, 30, 7900, 3, 8050, 600, 8100, 9, 7000, 8000]),
    (1, [50, 4000, 9000, 60, 12_000, 11_000, 8, 20_000, 15_000, 19_000]),
    (2, [50, 4000, 9000, 60, 12_000, 11_000, 8, 20_000, 15_000, 19_000]),
])
def test_queued_tables(streams, counts):
    import torch
    from scriptrs_amd import ParakeetFeatureExtractor
    calls = _calls(counts, len(counts) + streams)
    x = torch.randn(int(max(o[-1] for o in calls)), device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(4))
    alone = ParakeetFeatureExtractor()
    want = []
    for o in calls:
        want.append(alone.extract_batch(x, o)[0])
        torch.cuda.synchronize()
    ext = ParakeetFeatureExtractor()
    s = [torch.cuda.Stream() for _ in range(streams)]
    out = [torch.zeros_like(w) for w in want]
    torch.cuda.synchronize()
    for i, o in enumerate(calls):
        ext.extract_batch(x, o, stream=s[i % streams], out=out[i])
    torch.cuda.synchronize()
    for i in range(len(calls)):
        assert torch.equal(out[i].view(torch.int32), want[i].view(torch.int32)), i
    ext.close()
    alone.close()
