"""Head dimension 64, forward on grids large enough to go through key tiles in halves: the form that small grids run must agree."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
# windows of at least 1024 keys after both have been limited to T: shorter ones take whole tiles.  Lengths of 129 (one row past a
# workgroup) and 1100 end in the first half of a 64-key tile, 511 in the second.
@pytest.mark.parametrize("B,H,T,C,R", [(513, 1, 129, 33, 31), (513, 1, 129, 1000, 1000), (257, 1, 511, 33, 31), (16, 8, 1100, 1100, 0)])
def test_forward_halves(B, H, T, C, R, dtype, eps):
    from streaming_attention import streaming_attention

    assert min(C, T) * (min(R, T) + 1) >= 1024 and B * H * -(-T // 128) > 1024
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(5)
    q, k, v = (torch.randn(B, H, T, 64, generator=g, device=dev).to(dtype) for _ in range(3))
    lens = torch.randint(1, T + 1, (B,), generator=g, device=dev, dtype=torch.int32)
    lens[:3] = torch.tensor([T, T - 31, 32], device=dev)
    out, lse = streaming_attention(q, k, v, lens, C, R, return_lse=True)
    for b in [*range(6), B - 1]:
        L = int(lens[b])
        chunk = torch.arange(L, device=dev) // C
        mask = (chunk[None] <= chunk[:, None]) & (chunk[None] >= chunk[:, None] - R)
        s = (q[b, :, :L].double() @ k[b, :, :L].double().mT / 8).masked_fill(~mask, float("-inf"))
        want = s.softmax(-1) @ v[b, :, :L].double()
        # one rounding of the result and one of each probability
        assert ((out[b, :, :L].double() - want).norm() / want.norm()).item() <= 2 * eps
        assert (lse[b, :, :L].double() - s.logsumexp(-1) * 1.4426950408889634).abs().max() <= 1e-4
        assert not out[b, :, L:].any()
    few, few_lse = streaming_attention(q[:2], k[:2], v[:2], lens[:2], C, R, return_lse=True)
    assert (few.double() - out[:2].double()).abs().max() <= 4 * eps * max(1.0, v[:2].abs().max().item())
    assert (few_lse - lse[:2]).abs().max() <= 1e-4
