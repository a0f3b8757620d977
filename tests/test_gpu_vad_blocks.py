"""VAD framing at the edges of its workgroups (4 rows each) and on both sides
of the size past which 4-byte samples are read with streaming loads: bit-exact
against the gather x(512 w - 64 + p) (zero before the recording, the last
sample past its end), which tests/test_vad_framing.py pins to the reference's
loop."""
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
