"""Q and K quantised by one call, with the channel maxima's table set beside
them: the bytes of the separate calls, where both share a launch and where the
second follows on its own, over the last tile's edges."""

import pytest
import torch

from conftest import cpu_randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp8_block", "mxfp8"])
@pytest.mark.parametrize("sub", ["none", "both", "second"])
@pytest.mark.parametrize("dtype,dtype2,hadamard", [(torch.bfloat16, torch.bfloat16, False),
                                                   (torch.float16, torch.float16, True),
                                                   (torch.float32, torch.bfloat16, False)])
def test_same_bytes_as_two_calls(gpu, mode, sub, dtype, dtype2, hadamard):
    from low_bit_fake_quant import _lib as L, _ops
    b, s, h, d, P = 2, 192, 3, 64, 256
    srcs = [_ops.RowSource(x=cpu_randn(b, s, h, d, seed=i, dtype=t).to(gpu)) for i, t in enumerate((dtype, dtype2))]
    mean = cpu_randn(b, h, d, seed=5, dtype=torch.float32).to(gpu)
    for i, src in enumerate(srcs):
        if sub == "both" or (sub == "second" and i == 1):
            src.sub_mode, src.sub = L.SUB_COLVEC, mean

    def params(src):
        codes = torch.full((b, h, P, d), 0x55, dtype=torch.uint8, device=gpu)
        kw = dict(codes=codes, codes_layout=L.LAYOUT_BHSD, codes_spitch=P, hadamard=hadamard, had_scale=d ** -0.5)
        if mode == "fp8_block":
            scale = torch.zeros((b, h, s // 64), dtype=torch.float32, device=gpu)
            kw.update(R=64, quant_mode=L.Q_FP8_BLOCK, scale=scale, scale_strides=(h * (s // 64), 1, s // 64, 0))
        else:
            scale = torch.zeros((b, h, P, d // 32), dtype=torch.uint8, device=gpu)
            kw.update(R=64, quant_mode=L.Q_MX_QK, scale=scale, scale_strides=(h * P * 2, 2, P * 2, 1), mx_block=32,
                      scale_e8m0=True)
        return codes, scale, kw

    want = []
    for src in srcs:
        codes, scale, kw = params(src)
        _ops.rowtile(src, **kw)
        want += [codes, scale]
    for n in (1, 2):
        table = torch.zeros(b * h * d + 1, dtype=torch.int32, device=gpu)
        sets = [params(src) for src in srcs[:n]]
        ps = [_ops.rowtile_params(src, **kw) for src, (_, _, kw) in zip(srcs, sets)] + [None]
        _ops.rowtile_pair(ps[0], ps[1], gpu, table[:-1])
        for got, ref in zip([t for c, sc, _ in sets for t in (c, sc)], want):
            assert torch.equal(got, ref)
        assert bool((table[:-1] == _ops.AMAX_FLOOR_BITS).all()) and int(table[-1]) == 0


def test_other_modes_are_refused(gpu):
    from low_bit_fake_quant import _lib as L, _ops
    src = _ops.RowSource(x=torch.ones(1, 64, 1, 64, device=gpu))
    table = torch.zeros(64, dtype=torch.int32, device=gpu)
    p = _ops.rowtile_params(src, R=64, quant_mode=L.Q_CHANNEL_AMAX, amax_table=table)
    with pytest.raises(Exception, match="FP8_BLOCK and MX_QK"):
        _ops.rowtile_pair(p, None, src.x.device)
