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


@pytest.mark.parametrize("mode,pair", [("channel", False), ("mx_v", False), ("mx_qk", False), ("mx_qk", True),
                                       ("block", False), ("block", True)])   # the pair entry takes the Q / K modes
def test_rows_not_given_are_left_alone(gpu, mode, pair):
    """A head-major buffer filled in pieces, each call writing its own rows only:
    the codes of one call over all rows, and every byte past them (the padding
    rows and the space behind the buffer) as it was."""
    from low_bit_fake_quant import _lib as L, _ops
    b, s, h, d, pitch, slack = 2, 320, 3, 64, 512, 4096
    x = cpu_randn(b, s, h, d, seed=8).to(gpu)
    transposed = mode in ("channel", "mx_v")
    qm = dict(channel=L.Q_CHANNEL, mx_qk=L.Q_MX_QK, block=L.Q_FP8_BLOCK, mx_v=L.Q_MX_V)[mode]
    table = _ops.channel_amax(_ops.RowSource(x)) if mode == "channel" else None

    def buffer():
        flat = torch.full((b * h * pitch * d + slack,), 0xAB, dtype=torch.uint8, device=gpu)
        codes = flat[:b * h * pitch * d].view((b, h, d, pitch) if transposed else (b, h, pitch, d))
        return flat, codes

    def fill(codes, s0, s1):
        piece = codes[..., s0:] if transposed else codes[:, :, s0:]
        scale = torch.empty((b, h, pitch, d), dtype=torch.float32, device=gpu)
        p = _ops.rowtile_params(_ops.RowSource(x[:, s0:s1].contiguous()), R=64, quant_mode=qm, codes=piece,
                                codes_layout=L.LAYOUT_BHDS if transposed else L.LAYOUT_BHSD, codes_spitch=pitch,
                                scale=scale, scale_strides=(h * pitch * d, d, pitch * d, 1), amax_table=table,
                                zero_pad=False)
        lib, st = L.load(), L.stream_handle(gpu)
        if pair:
            L.check(lib.lbfq_rowtile_pair(p, None, None, 0, 0, st), "lbfq_rowtile_pair")
        else:
            L.check(lib.lbfq_rowtile(p, st), "lbfq_rowtile")
        torch.cuda.synchronize()  # piece x is a temporary

    (whole, w), (pieces, c) = buffer(), buffer()
    fill(w, 0, s)
    for s0, s1 in ((0, 64), (64, 256), (256, 320)):
        fill(c, s0, s1)
    assert torch.equal(pieces, whole)
    rows = c if transposed else c.transpose(2, 3)
    assert bool((rows[..., s:] == 0xAB).all()) and bool((pieces[-slack:] == 0xAB).all())
    assert bool((rows[..., :s] != 0xAB).any())
