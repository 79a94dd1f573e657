"""Forward of long windows on large grids, on whole key tiles (head dimension 64) and half a tile at a time (256): agreement
with float64 and with a small grid, and the running maximum is that of a whole tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("D", [64, 256])
# windows of at least 1024 keys after both have been limited to T (the long-window form).  Lengths of 129 (one row past a
# workgroup) and 1100 end in the first half of a 64-key tile, 511 in the second.
@pytest.mark.parametrize("B,H,T,C,R", [(513, 1, 129, 33, 31), (513, 1, 129, 1000, 1000), (257, 1, 511, 33, 31), (16, 8, 1100, 1100, 0)])
def test_forward_halves(B, H, T, C, R, D, dtype, eps):
    from streaming_attention import streaming_attention

    assert min(C, T) * (min(R, T) + 1) >= 1024 and B * H * -(-T // 128) > 1024
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(5)
    q, k, v = (torch.randn(B, H, T, D, generator=g, device=dev).to(dtype) for _ in range(3))
    lens = torch.randint(1, T + 1, (B,), generator=g, device=dev, dtype=torch.int32)
    lens[:3] = torch.tensor([T, T - 31, 32], device=dev)
    out, lse = streaming_attention(q, k, v, lens, C, R, return_lse=True)
    for b in [*range(6), B - 1]:
        L = int(lens[b])
        chunk = torch.arange(L, device=dev) // C
        mask = (chunk[None] <= chunk[:, None]) & (chunk[None] >= chunk[:, None] - R)
        s = (q[b, :, :L].double() @ k[b, :, :L].double().mT / D ** 0.5).masked_fill(~mask, float("-inf"))
        want = s.softmax(-1) @ v[b, :, :L].double()
        # one rounding of the result and one of each probability
        assert ((out[b, :, :L].double() - want).norm() / want.norm()).item() <= 2 * eps
        assert (lse[b, :, :L].double() - s.logsumexp(-1) * 1.4426950408889634).abs().max() <= 1e-4
        assert not out[b, :, L:].any()
    few, few_lse = streaming_attention(q[:2], k[:2], v[:2], lens[:2], C, R, return_lse=True)
    assert (few.double() - out[:2].double()).abs().max() <= 4 * eps * max(1.0, v[:2].abs().max().item())
    assert (few_lse - lse[:2]).abs().max() <= 1e-4


@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])   # 11 and 8 significand bits
@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T,C,R", [(1100, 1100, 0), (1100, 64, 3), (64, 64, 0)])
def test_largest_weight_of_the_first_tile_is_exact(T, C, R, D, dtype, eps):
    """A tile's largest score is subtracted before the probabilities are rounded to the element type, so its own is exactly one
    there, also where it stands in the second half of the tile; a maximum of the first half would be within the limit up to
    which it is kept (8 in the exponent of two), and the weight would be rounded."""
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    B, H = 8, 16
    g = torch.Generator(device=dev).manual_seed(6)
    q, k = (torch.zeros(B, H, T, D, device=dev) for _ in range(2))
    v = torch.randn(B, H, T, D, generator=g, device=dev).to(dtype)
    q[..., 0] = 1
    s = torch.rand(B, H, T, generator=g, device=dev) * 2
    top = 40
    s[:, :, top] = 2.1 + 3 * torch.rand(B, H, generator=g, device=dev)
    k[..., 0] = s * D ** 0.5
    q, k = q.to(dtype), k.to(dtype)
    v[..., 0] = 0
    v[:, :, top, 0] = 1
    n = min(T, C * (R + 1))   # the queries whose window begins with that tile
    out = streaming_attention(q, k, v, None, C, R)[:, :, :n, 0].double()
    chunk = torch.arange(T, device=dev) // C
    seen = ((chunk[None] <= chunk[:n, None]) & (chunk[None] >= chunk[:n, None] - R)).double()
    e = (k[..., 0].double() * D ** -0.5).exp()
    want = e[:, :, top, None] / (e[:, :, None] * seen).sum(-1)
    assert ((out - want).abs() / want).max().item() <= eps * (1 + 2.0 ** -6)   # one rounding, the result's own
