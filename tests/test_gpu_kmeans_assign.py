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
