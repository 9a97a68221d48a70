"""The quantisers write the padding rows of head-major code buffers themselves:
every byte of rows [S, pitch) is zero, every code below S what the same call
leaves in a cleared buffer, for pitches and lengths that are not whole words."""

import pytest
import torch

from conftest import cpu_randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s,pitch", [(1, 256), (64, 64), (97, 100), (1000, 1024), (1023, 1280), (320, 512)])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mode", ["channel", "mx_qk", "block", "mx_v"])
def test_padding_rows_are_zeroed(gpu, mode, d, s, pitch):
    from low_bit_fake_quant import _lib as L
    from low_bit_fake_quant._ops import RowSource, channel_amax, rowtile
    b, h = 2, 3
    if mode in ("block", "mx_v") and s % 64:
        pytest.skip("the block quantisers take whole blocks")
    src = RowSource(cpu_randn(b, s, h, d, seed=s + d).to(gpu))
    transposed = mode in ("channel", "mx_v")
    shape = (b, h, d, pitch) if transposed else (b, h, pitch, d)
    out = []
    for fill in (0, 0xAB):
        codes = torch.full(shape, fill, dtype=torch.uint8, device=gpu)
        scale = torch.zeros((b, h, pitch, d), dtype=torch.float32, device=gpu)
        kw = dict(codes=codes, codes_layout=L.LAYOUT_BHDS if transposed else L.LAYOUT_BHSD, codes_spitch=pitch,
                  scale=scale, scale_strides=(h * pitch * d, d, pitch * d, 1))
        if mode == "channel":
            rowtile(src, R=64, quant_mode=L.Q_CHANNEL, amax_table=channel_amax(src), **kw)
        elif mode == "mx_qk":
            rowtile(src, R=64, quant_mode=L.Q_MX_QK, mx_block=32, **kw)
        else:
            rowtile(src, R=64, quant_mode=L.Q_FP8_BLOCK if mode == "block" else L.Q_MX_V, **kw)
        out.append(codes if transposed else codes.transpose(2, 3))
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
    assert not out[1][..., s:].any() and (s < 64 or out[1][..., :s].any())
