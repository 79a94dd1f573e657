"""A sequence has the same bits alone and in a batch of any size: where the size of the grid picks the workgroups, their results
do not differ.  Batches on both sides of every such rule (up to 1024 and 128 workgroups of 128 rows, 256 of 256 rows)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def bits_alone_and_in_batches(dtype, H, T, D, C, R, batches):
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(31)
    B = max(batches)
    q, k, v, d_o = (torch.randn(B, H, T, D, generator=g, device=dev).to(dtype) for _ in range(4))
    lens = torch.randint(T // 2, T + 1, (B,), generator=g, device=dev, dtype=torch.int32)
    lens[:2] = torch.tensor([T, T // 3])

    def step(n0, n1):
        x = [t[n0:n1].clone().requires_grad_() for t in (q, k, v)]
        o, lse = streaming_attention(*x, lens[n0:n1], C, R, return_lse=True)
        return [o.detach(), lse.detach(), *torch.autograd.grad(o, x, d_o[n0:n1])]

    alone = [torch.cat(pair) for pair in zip(step(0, 1), step(1, 2))]
    for n in batches:
        for name, one, many in zip(("O", "LSE", "dQ", "dK", "dV"), alone, step(0, n)):
            assert torch.equal(one, many[:2]), (name, n, int((one != many[:2]).sum()))


@pytest.mark.parametrize("C,R", [(32, 2), (64, 1), (64, 2), (128, 0), (128, 1), (16, 2), (10, 9), (50, 3), (200, 0)])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_16_bit_short_windows(dtype, D, C, R):
    bits_alone_and_in_batches(dtype, 8, 300, D, C, R, (2, 42, 43))   # 1008 and 1032 workgroups of 128 rows


@pytest.mark.parametrize("C,R", [(64, 2), (50, 1), (10, 9), (32, 2), (128, 1), (24, 5)])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_float32(D, C, R):
    """Two, four and eight waves to a workgroup go through the tiles of a row's window in one order and form its row sum in one order."""
    bits_alone_and_in_batches(torch.float32, 8, 600, D, C, R, (2, 3, 4, 10, 11))   # 120 and 160 workgroups of 128 rows, 240 and 264 of 256


@pytest.mark.parametrize("D", [32, 64, 128])
def test_float32_long_windows(D):
    bits_alone_and_in_batches(torch.float32, 8, 1500, D, 96, 4, (2, 4, 6))   # 192 workgroups of 128 rows, 288 of 256


@pytest.mark.parametrize("C,R", [(1000, 0), (96, 30), (64, 2)])   # one chunk over everything, chunks whose windows do, and those that do not
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_float32_padded_to_another_length(D, C, R):
    """The padded length T of a batch, to which longer windows are cut, changes no bit either."""
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    B, H, L = 2, 8, 180
    g = torch.Generator(device=dev).manual_seed(32)
    q, k, v, d_o = (torch.randn(B, H, 1600, D, generator=g, device=dev) for _ in range(4))
    lens = torch.tensor([L, L - 37], dtype=torch.int32, device=dev)

    def step(T):
        x = [t[:, :, :T].clone().requires_grad_() for t in (q, k, v)]
        o, lse = streaming_attention(*x, lens, C, R, return_lse=True)
        return [t[:, :, :L] for t in (o.detach(), lse.detach(), *torch.autograd.grad(o, x, d_o[:, :, :T]))]

    short = step(L)
    for T in (191, 192, 511, 512, 1600):
        for name, a, b in zip(("O", "LSE", "dQ", "dK", "dV"), short, step(T)):
            assert torch.equal(a, b), (name, T)
