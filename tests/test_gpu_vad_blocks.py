"""VAD framing at the edges of its workgroups (4 rows each) and on both sides
of the size past which 4-byte samples are read with streaming loads: bit-exact
against the gather x(512 w - 64 + p) (zero before the recording, the last
sample past its end), which tests/test_vad_framing.py pins to the reference's
loop; and a recording of more rows than one launch holds."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "int16", "int32"])
@pytest.mark.parametrize("n", [1, 511, 512 * 3, 512 * 4, 512 * 4 + 1, 512 * 8 - 1, 31_500_000, 31_700_003])
def test_rows_at_workgroup_edges(n, dtype):
    import torch
    from scriptrs_amd import SileroVadFramer
    g = torch.Generator(device="cuda").manual_seed(n)
    if dtype == "float32":
        x = torch.randn(n, device="cuda", generator=g)
    else:
        x = torch.randint(-32768, 32768, (n,), device="cuda", generator=g, dtype=torch.int32)
        x = x.to(torch.int16) if dtype == "int16" else x * 65536 + 12345
    # the WAV reader's `value as f32 / ((1 << (bits - 1)) - 1) as f32`; at 32
    # bits the divisor rounds to 2^31, so the quotient is exact
    y = {"float32": lambda: x, "int16": lambda: (x.double() / 32767.0).float(),
         "int32": lambda: x.float() / 2147483648.0}[dtype]()
    windows = (n + 511) // 512
    want = torch.cat([y.new_zeros(64), y, y[-1:].expand(windows * 512 - n)]).unfold(0, 576, 512)
    framer = SileroVadFramer()
    got = framer.model_inputs(x)
    assert torch.equal(got, want)
    framer.close()


def test_rows_past_one_launch():
    """A launch holds fewer than 2^32 threads, 144 a row: past 29,826,160 rows a
    second one follows.  30,000,000 rows of 16-bit PCM (31 GB in, 69 GB out):
    every row is written, and those at the ends and around the limit are the
    gather."""
    import torch
    from scriptrs_amd import SileroVadFramer
    windows = 30_000_000
    n = 512 * windows - 100
    if torch.cuda.mem_get_info()[0] < 110 << 30:
        pytest.skip("needs 110 GB of free GPU memory")
    g = torch.Generator(device="cuda").manual_seed(30)
    x = torch.empty(n, dtype=torch.int16, device="cuda")
    tile = torch.randint(-32768, 32768, (99_999_989,), device="cuda", generator=g, dtype=torch.int16)
    for i in range(0, n, tile.numel()):
        x[i:i + tile.numel()] = tile[:n - i]
    out = torch.full((windows, 576), float("nan"), device="cuda")
    framer = SileroVadFramer()
    framer.model_inputs(x, out=out)
    for i in range(0, windows, 1_000_000):
        assert not torch.isnan(out[i:i + 1_000_000]).any(), i
    for w0, w1 in ((0, 1000), (29_826_000, 29_827_000), (windows - 1000, windows)):
        lo, hi = w0 * 512 - 64, min(n, w1 * 512)
        y = (x[max(lo, 0):hi].double() / 32767.0).float()
        y = torch.cat([y.new_zeros(max(-lo, 0)), y, y[-1:].expand(w1 * 512 - hi)])
        assert torch.equal(out[w0:w1], y.unfold(0, 576, 512)), w0
    framer.close()
