"""Path A at the sizes where its kernels change over: a single tile, few queries
(each query's keys split over a workgroup's waves, some of them without tiles),
and the first size past that; groups whose correction rows are staged (>= 32
queries) and not.  Checked as tests/test_gpu_sdpa.py: against a float64 replay
on the kernel's own operands."""

import pytest
import torch

import parity
from conftest import cpu_randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,s,d,group", [(1, 64, 64, 0), (1, 65, 128, 0), (3, 300, 64, 0), (2, 1000, 128, 0),
                                         (1, 64, 64, 64), (2, 320, 128, 16), (1, 520, 64, 40), (2, 1024, 128, 256),
                                         (9, 960, 64, 0), (9, 960, 64, 48), (9, 960, 64, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_float64(gpu, h, s, d, group, dtype):
    from low_bit_fake_quant import QuantConfig
    from low_bit_fake_quant import attention as A
    kw = dict(qk_quant="mxfp8", v_quant="fp8_channel", q_kmeans_k=None, p_requant=False)
    cfg = QuantConfig(smoothing="full" if group else "off", q_smooth_block_size=group or 256, **kw)
    q, k, v = (cpu_randn(1, s, h, d, seed=70 + i + s, dtype=dtype).to(gpu) for i in range(3))
    sm = d ** -0.5
    ops = A.sdpa_operands(A._lazy_preprocess(q, k * 1.5, v, cfg), cfg, sm, dtype)
    out = A.launch_sdpa(ops, sm, dtype)
    torch.cuda.synchronize()
    st = parity.sdpa_replay(ops, out, sm)
    assert st["excess"] <= 1.0, st
    assert st["frac_equal"] >= 0.97, st


@pytest.mark.parametrize("tiles", [(1,), (7, 12), (1, 9), (0,), (0, 1, 2, 3, 4, 5, 6, 7)])
@pytest.mark.parametrize("d", [64, 128])
def test_a_wave_whose_products_all_overflow(gpu, d, tiles):
    """Keys whose products with Q overflow to -inf weigh nothing, also where
    they are the first (and only) keys that one of the row's waves sees."""
    from low_bit_fake_quant import QuantConfig
    from low_bit_fake_quant import attention as A
    s, h = 812, 2   # 13 tiles of 64 keys, wave w takes tiles w and w + 8
    cfg = QuantConfig(qk_quant="mxfp8", v_quant="fp8_channel", q_kmeans_k=None, p_requant=False, smoothing="off")
    q, k, v = (cpu_randn(1, s, h, d, seed=30 + i).to(gpu) for i in range(3))
    sm = d ** -0.5
    ops = A.sdpa_operands(A._lazy_preprocess(q, k, v, cfg), cfg, sm, torch.bfloat16)
    ops.q[..., 0], ops.k[..., 0] = 1e4, 0.0
    keep = torch.ones(s, dtype=torch.bool)
    for t in tiles:
        ops.k[:, :, 64 * t:64 * t + 64, 0] = -1e37
        keep[64 * t:64 * t + 64] = False
    out = A.launch_sdpa(ops, sm, torch.bfloat16)
    torch.cuda.synchronize()
    qd, kd = ops.q[:, :, :s].cpu().double(), ops.k[:, :, :s].cpu().double()[:, :, keep]
    vd = ops.v_t[..., :s].cpu().double().transpose(-1, -2)[:, :, keep]
    want = (torch.softmax(qd @ kd.transpose(-1, -2) * sm, -1) @ vd).permute(0, 2, 1, 3)
    # the output's rounding to bf16; fp32 scores, weights and sums are within 2^-14 of max|v|
    bound = want.abs() * 2.0 ** -8 + float(vd.abs().max()) * 2.0 ** -14
    assert bool(((out.cpu().double() - want).abs() <= bound).all())
