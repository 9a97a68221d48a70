"""The k-means assignment kernel (approximate distances on the matrix cores,
settled by the specification's FMA chain where they are close) and its update,
bit for bit against the oracle's scalar C restatement."""

import pytest
import torch

from oracle import kmeans as okm

pytestmark = pytest.mark.gpu


def _check(x, gpu, k, iters=3, seed=3):
    from low_bit_fake_quant import kmeans_reorder_tokens
    r = kmeans_reorder_tokens(x.to(gpu), n_clusters=k, max_iters=iters, seed=seed)
    ref = okm.kmeans_reorder_tokens(x, n_clusters=k, max_iters=iters, seed=seed)
    assert torch.equal(r.labels.cpu(), ref["labels"])
    assert torch.equal(r.order.cpu(), ref["order"])
    assert torch.equal(r.inverse_order.cpu(), ref["inverse_order"])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("s,k", [(64, 64), (65, 33), (255, 32), (257, 31), (1025, 1), (1300, 64)])
def test_tile_edges(gpu, s, k, d, dtype):
    """Cluster counts on both sides of a 32-row tile, lengths on both sides of
    a 32-token wave, a 256-token slab and a 1024-token chunk."""
    g = torch.Generator().manual_seed(s + k + d)
    _check((torch.randn(2, s, 3, d, generator=g) + torch.randn(1, 1, 3, d, generator=g)).to(dtype), gpu, k)


@pytest.mark.parametrize("kind", ["all_equal", "duplicates", "zeros", "two_scales", "tiny", "huge", "non_finite"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_undecided_tokens(gpu, kind, dtype):
    """Inputs whose distances tie, nearly tie, underflow, overflow or are not
    numbers: every token takes the label of the first smallest fp32 distance."""
    g = torch.Generator().manual_seed(9)
    x = torch.randn(1, 700, 2, 128, generator=g)
    if kind == "all_equal":
        x = x[:, :1].expand(-1, 700, -1, -1).clone()
    elif kind == "duplicates":
        x = x[:, torch.randint(0, 20, (700,), generator=g)]
    elif kind == "zeros":
        x = torch.zeros_like(x)
    elif kind == "two_scales":   # a common offset far above the spread: distances agree to their last bits
        x = x * 2.0 ** -6 + 64.0
    elif kind == "tiny":
        x = x * 1e-30
    elif kind == "huge":
        x = x * 1e19
    else:
        x[0, 3, 0, 5], x[0, 70, 0, 0], x[0, 400, 1, 127] = float("nan"), float("inf"), -float("inf")
    _check(x.to(dtype), gpu, 40)


@pytest.mark.parametrize("kind", ["clustered", "drifting", "outlier_scale", "signed_zeros"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rounds_that_reuse_the_last(gpu, kind, dtype):
    """Later rounds read only the tokens whose label may change and update
    exact chunks by their moved tokens (fp32 and wide-range chunks are summed
    anew): every round count gives the labels of the full rounds, from few moves
    a round to most of a chunk, over chunk and slab edges."""
    g = torch.Generator().manual_seed(21)
    s, h, d, k = 2309, 2, 128, 32
    if kind == "drifting":   # one slow blob: centroids keep moving, few tokens are certain
        x = torch.randn(1, s, h, d, generator=g)
        x[..., 0] = torch.linspace(-20, 20, s)[None, :, None]
    else:
        cent = 3 * torch.randn(h, k, d, generator=g)
        pick = torch.randint(0, k, (s, h), generator=g)
        x = (torch.stack([cent[i][pick[:, i]] for i in range(h)], 1) + torch.randn(s, h, d, generator=g))[None]
    if kind == "outlier_scale":   # chunk 0's values span more than fp64 holds exactly
        x[0, 100, :, 3], x[0, 200, :, 4] = 2.0 ** 14, 2.0 ** -24
        x[0, 300, 1, 5] = 1e-30
    elif kind == "signed_zeros":
        x = torch.where(torch.rand(x.shape, generator=g) < 0.7, -0.0 * x, x)
    for iters in (2, 3, 12):
        _check(x.to(dtype), gpu, k, iters=iters, seed=iters)


@pytest.mark.parametrize("pad", ["zeros", "last_row"])
@pytest.mark.parametrize("s,k,dtype", [(272, 32, torch.bfloat16), (372, 64, torch.bfloat16), (300, 40, torch.float32)])
def test_repeated_centroids(gpu, s, k, dtype, pad):
    """A padded sequence starts with many centroids that are one and the same
    row; the first of them moves off with its cluster's other tokens, and the
    pad tokens go to the next repeat."""
    g = torch.Generator().manual_seed(s)
    x = torch.randn(2, 512, 3, 64, generator=g)
    x[:, :s // 2] *= 0.1   # tokens that share the pad rows' cluster at first
    x[:, s - 1] *= 0.1
    x[:, s:] = 0.0 if pad == "zeros" else x[:, s - 1:s]
    for iters in (1, 2, 3, 10):
        _check(x.to(dtype), gpu, k, iters=iters, seed=iters)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_many_rounds_of_small_steps(gpu, dtype):
    """Centroids that start far out, jump to the tokens in one round and then
    creep for hundreds: steps below the last bit of their path so far still
    move the bounds."""
    g = torch.Generator().manual_seed(2)
    s, h, d, k, seed = 3000, 2, 64, 16, 9
    x = 1e-3 * torch.randn(1, s, h, d, generator=g)
    x[..., 0] = (torch.rand(1, s, h, generator=g) - 0.5)
    for i in range(h):   # the initial centroids: far tokens in random directions
        for j in range(k):
            far = torch.randn(d, generator=g)
            x[0, j * (s // k) + okm.mix(seed, i, k, j) % (s // k), i] = 2000.0 * far / far.norm()
    for iters in (3, 400):
        _check(x.to(dtype), gpu, k, iters=iters, seed=seed)


@pytest.mark.parametrize("k,repeats", [(1, 0), (30, 0), (31, 0), (62, 0), (63, 0), (32, 1), (40, 1), (64, 2), (31, 5)])
@pytest.mark.parametrize("norm2", [0.9e38, 2.2e38, 3.0e38])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_centroid_norms_near_the_top_of_fp32(gpu, k, repeats, norm2, dtype):
    """Finite centroids whose squared norms lie on both sides of what the rows
    that must never win (padding to a whole 32-row tile, repeats) start from,
    and tokens short enough that no distance overflows: the label is still the
    first smallest distance's, never a padding row or a repeat."""
    s, h, d, seed = 20 * k + 7, 2, 128, 5
    g = torch.Generator().manual_seed(k + repeats)
    x = 0.02 * torch.randn(1, s, h, d, generator=g)
    x[:, ::5] = 0.0
    stride = s // k
    for i in range(h):   # the rows of the initial centroids
        c = torch.randn(k, d, generator=g, dtype=torch.float64)
        c *= (norm2 * (0.97 + 0.06 * torch.rand(k, 1, generator=g, dtype=torch.float64))).sqrt() / c.norm(dim=1, keepdim=True)
        c[k - repeats:] = c[0]
        for j in range(k):
            x[0, j * stride + okm.mix(seed, i, k, j) % stride, i] = c[j].float()
    for iters in (1, 2, 4):
        _check(x.to(dtype), gpu, k, iters=iters, seed=seed)


@pytest.mark.parametrize("s,h", [(60 << 16, 2), (1024, 8192)])
def test_noalloc_without_room_for_the_carried_state(gpu, s, h):
    """A problem that fits the built-in scratch only without the state carried
    between rounds (long slices, and many of one chunk) still runs there, with
    the same labels."""
    from low_bit_fake_quant import _lib as L
    lib = L.load()
    b, d, k = 1, 64, 8
    need = int(lib.lbfq_kmeans_workspace_bytes(b, s, h, d, k))
    assert need > int(lib.lbfq_kmeans_noalloc_max_workspace_bytes())
    x = torch.randn(b, s, h, d, device=gpu, dtype=torch.bfloat16)
    st = L.stream_handle(gpu)
    outs = [[torch.full((b * h, s), -1, dtype=torch.int32, device=gpu) for _ in range(3)] for _ in range(2)]
    L.check(lib.lbfq_kmeans_noalloc(x.data_ptr(), L.DTYPE_CODE[x.dtype], b, s, h, d, k, 4, 0,
                                    *(t.data_ptr() for t in outs[0]), st), "lbfq_kmeans_noalloc")
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    L.check(lib.lbfq_kmeans(x.data_ptr(), L.DTYPE_CODE[x.dtype], b, s, h, d, k, 4, 0, ws.data_ptr(),
                            *(t.data_ptr() for t in outs[1]), st), "lbfq_kmeans")
    torch.cuda.synchronize()
    for got, want in zip(*outs):
        assert torch.equal(got, want)


@pytest.mark.parametrize("spread", [0, 4, 12])
@pytest.mark.parametrize("carry", [False, True])
def test_mfma_error_that_the_gap_allows_for(gpu, carry, spread):
    """The assignment's gap counts 2^-20 of the magnitudes added for each
    v_mfma_f32_32x32x16_bf16.  One such instruction, its accumulator zero or
    (carry) one product of an earlier one, through the simulator's score scan
    at scale 1: every key of a head is the same, so a row's maximum is its
    score.  Operands of one magnitude up to ones over 2^24 (products 2^48)."""
    from low_bit_fake_quant.blasst_skip import _SimBf16
    s, h, d = 128, 256, 64
    g = torch.Generator().manual_seed(spread + 100 * carry)

    def values(*shape):
        mag = torch.exp2(spread * (2 * torch.rand(*shape, generator=g) - 1))
        return (torch.randn(*shape, generator=g) * mag).to(torch.bfloat16)

    q, k = torch.zeros(h, s, d, dtype=torch.bfloat16), torch.zeros(h, 1, d, dtype=torch.bfloat16)
    q[..., 16:32], k[..., 16:32] = values(h, s, 16), values(h, 1, 16)
    if carry:   # dimensions 0-15 come first: one exact product stands in the accumulator
        q[..., 0], k[..., 0] = 8 * values(h, s), values(h, 1)
    sim = _SimBf16(s, h, d, 1.0, gpu)
    got = sim.scan(q.to(gpu), k.expand(h, s, d).contiguous().to(gpu))[0].cpu().double()
    prod = q.double() * k.double()
    worst = float(((got - prod.sum(-1)).abs() / prod.abs().sum(-1).clamp_min(1e-300)).max())
    print(f"largest MFMA error / magnitudes, spread 2^{spread}, carry {carry}: {worst * 2 ** 20:.3f} * 2^-20")
    assert worst <= 2.0 ** -20
