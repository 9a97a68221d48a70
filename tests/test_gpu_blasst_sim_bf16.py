"""The simulator's matrix-core kernels (bf16 matmul operands) at the edges of
their work split: one key block, a workgroup whose second query tile lies past
S, every input dtype, both head sizes, and operands that share one tensor."""

import pytest
import torch

from conftest import cpu_randn
from oracle import blasst_sim as osim

pytestmark = pytest.mark.gpu


def _close(a, b):
    """As tests/test_gpu_blasst_sim.py: a P weight may cross a bf16 or E4M3
    rounding boundary (one step is 2^-8 of the weight at most)."""
    a, b = a.double().flatten(), b.double().flatten()
    assert float(a @ b / (a.norm() * b.norm())) >= 0.99999
    assert float((a - b).abs().max()) <= 2e-3 * float(b.abs().max())


@pytest.mark.parametrize("s,h,d,dtype", [(128, 3, 64, torch.bfloat16), (128, 1, 128, torch.float32),
                                         (256, 2, 128, torch.float16), (384, 5, 64, torch.float32),
                                         (640, 1, 128, torch.bfloat16)])
def test_rungs_match_oracle(gpu, s, h, d, dtype):
    from low_bit_fake_quant import blasst_skip as bs
    q, k, v = (cpu_randn(1, s, h, d, seed=90 + i, dtype=torch.float32) for i in range(3))
    k[:, :128] *= 6.0          # the first block dominates: later ones can be skipped
    q, k, v = (t.to(dtype) for t in (q, k, v))
    ths = [0.05, 2.0]
    res = bs.simulate_workload(q.to(gpu), k.to(gpu), v.to(gpu), skip_thresholds=ths)
    ref = osim.simulate(q, k, v, skip_thresholds=ths, mm_dtype=torch.bfloat16)
    for lv in ("bf16_ref", "fp8_qkv", "fp8_static_p"):
        _close(res.outputs[lv][0].cpu(), ref[lv])
    for th in ths:
        _close(res.skip_outputs[th][0].cpu(), ref["skip"][th])
        dg = res.skip_diagnostics[th]
        assert dg.skip_rate == ref["skip_rate"][th] and dg.force_keep_count == ref["force"][th]
        assert abs(dg.dropped_mass_max - float(ref["dropped"][th].max())) < 1e-4
    for name in ("q", "k", "v"):
        st, so = res.quant_stats[name], ref["stats"][name]
        assert st.saturation_rate == so["saturation_rate"] and st.underflow_zero_rate == so["underflow_zero_rate"]
        assert abs(st.roundtrip_rmse - so["roundtrip_rmse"]) <= 1e-6 * so["roundtrip_rmse"] + 1e-12
    sp, op = res.quant_stats["p"], ref["stats"]["p"]
    assert abs(sp.underflow_zero_rate - op["underflow_zero_rate"]) < 1e-4
    assert abs(sp.roundtrip_rmse - op["roundtrip_rmse"]) <= 1e-3 * op["roundtrip_rmse"]


def test_one_tensor_as_all_three(gpu):
    from low_bit_fake_quant import blasst_skip as bs
    x = cpu_randn(1, 256, 2, 64, seed=4)
    xg = x.to(gpu)
    one = bs.simulate_workload(xg, xg, xg, skip_thresholds=[0.05])
    three = bs.simulate_workload(xg, xg.clone(), xg.clone(), skip_thresholds=[0.05])
    for lv in one.outputs:
        assert torch.equal(one.outputs[lv], three.outputs[lv])
    _close(one.outputs["bf16_ref"][0].cpu(), osim.simulate(x, x, x)["bf16_ref"])


@pytest.mark.parametrize("dtype", [torch.float64, torch.int32])
def test_reference_rung_takes_any_dtype_that_casts(gpu, dtype):
    """The bf16 reference rung rounds its operands to bf16 whatever they are;
    the quantising rungs take the float dtypes of the kernels only."""
    from low_bit_fake_quant import blasst_skip as bs
    q, k, v = ((3 * cpu_randn(1, 256, 2, 64, seed=i, dtype=torch.float64)).to(dtype).to(gpu) for i in range(3))
    res = bs.simulate_workload(q, k, v, skip_thresholds=[], levels=[bs.LEVEL_REFERENCE])
    want = bs.simulate_workload(*(t.to(torch.bfloat16) for t in (q, k, v)), skip_thresholds=[],
                                levels=[bs.LEVEL_REFERENCE])
    assert torch.equal(res.outputs[bs.LEVEL_REFERENCE], want.outputs[bs.LEVEL_REFERENCE])
    with pytest.raises(TypeError, match="unsupported dtype"):
        bs.simulate_workload(q, k, v, skip_thresholds=[], levels=[bs.LEVEL_FP8_QKV])


@pytest.mark.parametrize("mode,lv", [(1, "fp8_qkv"), (2, "fp8_static_p")])
@pytest.mark.parametrize("d", [64, 128])
def test_large_scores_keep_their_differences(gpu, d, mode, lv):
    """Scores that are exact integers around 13000: the weights depend on their
    differences, which are exact, so a rung is within fp32 exponentials and sums
    of 64 bits (rounding each scaled score would put 2^-24 * 13000 / sqrt(d) =
    1e-4 on each weight, and a thousandth of them on another E4M3 code)."""
    from low_bit_fake_quant import blasst_skip as bs
    s, h = 128, 16   # one block: its maximum is the final one
    g = torch.Generator().manual_seed(d + mode)
    q, k = (torch.randint(-2, 3, (s, h, d), generator=g).float() for _ in range(2))
    q[..., 0], k[..., 0] = 64.0, 200.0
    v = torch.randn(s, h, d, generator=g).to(torch.bfloat16)
    sim = bs._SimBf16(s, h, d, d ** -0.5, gpu)
    qg, kg, vg = (sim.operand(t.to(torch.bfloat16).to(gpu), quantise=False, transposed=tr)[0]
                  for t, tr in ((q, False), (k, False), (v, True)))
    fm = sim.scan(qg, kg)[0]
    out = sim.attend(qg, kg, vg, fm, mode)[0].cpu().double().permute(1, 0, 2)
    qd, kd, vd = (t.double().permute(1, 0, 2) for t in (q, k, v))
    u = qd @ kd.transpose(1, 2)
    top = u.amax(-1, keepdim=True)
    sm = float(torch.tensor(d ** -0.5, dtype=torch.float32))   # the scale the kernels are given
    p = torch.exp((u - top) * sm)
    w = (p * 256.0).float().to(torch.float8_e4m3fn).double() / 256.0 if mode == 2 else p
    want = w.to(torch.bfloat16).double() @ vd / p.sum(-1, keepdim=True)
    # fp32 sums and quotients stay within 2^-20; the few weights within 2^-22 of a rounding boundary may fall on
    # the other side of it (of 2^18 weights about one, by 2^-4 of a single weight)
    assert float((out - want).norm() / want.norm()) <= 2e-5


def test_fp32_entries_with_bf16_rounding(gpu):
    """The C entries of the fp32 kernels round their operands (mm_bf16) and P
    (round_p_bf16) to bf16 where asked: the rungs of the matrix-core entries."""
    from low_bit_fake_quant import _lib as L
    from low_bit_fake_quant import blasst_skip as bs
    s, h, d = 384, 2, 64
    xs = [cpu_randn(s, h, d, seed=60 + i).to(gpu) for i in range(3)]
    lib, st = L.load(), L.stream_handle(gpu)

    def quantised(x):
        deq, mm = (torch.empty(s, h, d, device=gpu) for _ in range(2))
        scale, ws = torch.empty(h, device=gpu), torch.empty(h, dtype=torch.int32, device=gpu)
        counts, sq = torch.zeros(2, dtype=torch.int64, device=gpu), torch.zeros(1, dtype=torch.float64, device=gpu)
        L.check(lib.lbfq_head_fp8_quant(x.data_ptr(), L.DTYPE_CODE[x.dtype], s, h, d, deq.data_ptr(), mm.data_ptr(), 1,
                                        scale.data_ptr(), ws.data_ptr(), counts.data_ptr(), sq.data_ptr(), st), "quant")
        assert torch.equal(mm, deq.to(torch.bfloat16).float())
        return mm

    fp32, mfma = bs._Sim(s, h, d, d ** -0.5, gpu), bs._SimBf16(s, h, d, d ** -0.5, gpu)
    a = [quantised(x) for x in xs]
    b = [mfma.operand(x, quantise=True, transposed=i == 2)[0] for i, x in enumerate(xs)]
    assert torch.equal(a[0].permute(1, 0, 2), b[0].float()) and torch.equal(a[2].permute(1, 2, 0), b[2].float())
    fm = fp32.scan(a[0], a[1])[0]
    for mode in (0, 1, 2):
        out = torch.empty(s, h, d, device=gpu)
        p = L.BlasstAttendParams()
        p.S, p.H, p.D = s, h, d
        p.q, p.k, p.v = (t.data_ptr() for t in a)
        p.sm_scale, p.mode, p.round_p_bf16, p.final_max, p.out = d ** -0.5, mode, 1, fm.data_ptr(), out.data_ptr()
        L.check(lib.lbfq_blasst_attend(p, st), "attend")
        plain = fp32.attend(*a, fm, mode)[0]
        want = mfma.attend(*b, mfma.scan(b[0], b[1])[0], mode)[0]
        _close(out.cpu(), want.cpu())
        # rounded, unlike P in fp32 (in the static rung the online weights' codes are bf16 values but for the rescale)
        assert mode == 2 or float((out - want).norm()) < 0.2 * float((plain - want).norm())
