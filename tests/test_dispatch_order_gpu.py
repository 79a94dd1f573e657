"""The order in which workgroups are dispatched (short windows first from 512 workgroups on, last below; pairs that do and do not
divide over the eight XCDs) changes no bit of any result: a large grid against the same sequences one at a time.  16-bit elements;
float32, whose workgroups are of another size on a small grid, in test_batch_invariance_gpu.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D,C,R", [(torch.float16, 256, 64, 3), (torch.bfloat16, 256, 50, 2), (torch.float16, 128, 64, 1),
                                         (torch.bfloat16, 128, 70, 2), (torch.float16, 128, 256, 9), (torch.float16, 64, 100, 5)], ids=str)
@pytest.mark.parametrize("B,H", [(8, 8), (9, 7)])
def test_large_grid_equals_single_sequences(B, H, dtype, D, C, R):
    from streaming_attention import streaming_attention

    T = 1100   # nine workgroups of 128 rows a pair
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(9)
    q, k, v, d_o = (torch.randn(B, H, T, D, generator=g, device=dev).to(dtype) for _ in range(4))
    lens = torch.tensor([T, T - 1, 129, 128, 1, 0, 700, 640, 1023][:B], device=dev, dtype=torch.int32)

    def step(b0, b1):
        x = [t[b0:b1].clone().requires_grad_() for t in (q, k, v)]
        o = streaming_attention(*x, lens[b0:b1], C, R)
        return [o.detach(), *torch.autograd.grad(o, x, d_o[b0:b1])]

    many = step(0, B)
    for b in range(B):
        for name, m, one in zip(("O", "dQ", "dK", "dV"), many, step(b, b + 1)):
            assert torch.equal(m[b:b + 1], one), (name, b)
            assert not one[:, :, int(lens[b]):].any()
