"""Short windows in workgroups of two waves (64 rows, tiles of 32) at head dimensions 32 and 64: the forward and the one-launch
backward against the float64 oracle, at lengths around the tiles and workgroups, on windows that end at, inside and beyond a
block of 32 rows, and on both sides of the rules that pick the small workgroups (a large grid is what the other side takes)."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import assert_close, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,R", [(8, 3), (16, 2), (32, 1), (64, 0), (10, 9), (50, 1), (7, 0), (33, 6), (96, 0), (64, 3)])
@pytest.mark.parametrize("T,lens", [(1, [1, 1]), (33, [33, 31]), (65, [64, 65]), (161, [0, 97]), (700, [700, 385])])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_short_windows(dtype, D, T, lens, C, R):
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    B, H = 2, 3
    q, k, v, d_o = make_inputs(B, H, T, D, seed=82, dtype=dtype)
    ld = torch.tensor(lens, dtype=torch.int32)
    # [B,T,H,D]-stored q and v: strided rows through the fragment loads and the tile copies
    qd, vd = (t.to(dev).transpose(1, 2).contiguous().transpose(1, 2).requires_grad_() for t in (q, v))
    kd = k.to(dev).requires_grad_()
    o, lse = streaming_attention(qd, kd, vd, ld.to(dev), C, R, return_lse=True)
    got = torch.autograd.grad(o, (qd, kd, vd), d_o.to(dev))
    ref = sa_oracle.dense_f64(q, k, v, ld, C, R, d_out=d_o)
    for name, g in zip(("O", "dQ", "dK", "dV"), (o, *got)):
        assert_close(name, g, ref[name], dtype)
        for b, n in enumerate(lens):
            assert not g[b, :, n:].any()
    assert (lse.cpu().double() - torch.from_numpy(ref["LSE"].copy())).abs().max().item() <= 1e-4
    # the same problems inside a grid of more than 1024 workgroups of 128 rows, whose rule looks at the windows alone
    n = -(-1025 // (B * H * -(-T // 128)))
    if n * B * H * T * D < 1 << 24:
        with torch.no_grad():
            many = streaming_attention(*(t.detach().repeat(n, 1, 1, 1) for t in (qd, kd, vd)), ld.to(dev).repeat(n), C, R)
        eps = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7   # one rounding of a result apart, and one of a probability
        assert (many.float() - o.detach().float().repeat(n, 1, 1, 1)).abs().max().item() <= 2 * eps * max(1.0, float(v.abs().max()))


@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])   # 11 and 8 significand bits
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("top", [3, 31, 32, 40, 63])
def test_largest_weight_of_the_first_two_tiles_is_exact(top, D, dtype, eps):
    """The second tile that a wave sees moves the maximum by however little, so the largest weight of the first 64 keys is
    not rounded on its way into the second product."""
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    B, H, T = 2, 4, 64
    g = torch.Generator(device=dev).manual_seed(7)
    q, k = (torch.zeros(B, H, T, D, device=dev) for _ in range(2))
    q[..., 0] = 1
    s = torch.rand(B, H, T, generator=g, device=dev) * 2
    s[:, :, top] = 2.1 + 3 * torch.rand(B, H, generator=g, device=dev)
    k[..., 0] = s * D ** 0.5
    q, k = q.to(dtype), k.to(dtype)
    v = torch.zeros(B, H, T, D, device=dev, dtype=dtype)
    v[:, :, top, 0] = 1
    out = streaming_attention(q, k, v, None, 64, 0)[..., 0].double()
    e = (k[..., 0].double() * D ** -0.5).exp()
    want = (e[:, :, top] / e.sum(-1))[..., None]
    assert ((out - want).abs() / want).max().item() <= eps * (1 + 2.0 ** -6)   # one rounding, the result's own
