"""float32 kernels that form their products from two float16 parts of scaled rows, and the rule that picks them: rows of very different
magnitude side by side, those that a query or key does not see included, at the edges of tiles, workgroups and windows."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu


# both sides of the rule (192 keys at D=64, 512 at D=32; every window at 128), B*H*ceil(T/256) on both sides of 256 at 128,
# grids of two- and four-wave workgroups, remainders of a row and of a tile
@pytest.mark.parametrize("B,H,T,D,C,R", [(1, 2, 300, 64, 64, 2), (1, 2, 300, 64, 191, 0), (2, 16, 641, 64, 96, 1), (1, 1, 2, 64, 192, 0),
                                         (1, 2, 700, 32, 256, 1), (1, 2, 700, 32, 511, 0), (3, 16, 545, 32, 128, 3),
                                         (1, 2, 300, 128, 10, 9), (8, 32, 97, 128, 32, 1), (1, 3, 513, 128, 1000, 0), (1, 1, 1, 128, 1, 0)])
@pytest.mark.parametrize("spread", [0, 12])   # rows of V and dO times powers of two up to this, either way
def test_rows_of_different_magnitude(B, H, T, D, C, R, spread):
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    q, k, v, d_o = (t.to(dev) for t in make_inputs(B, H, T, D, seed=81))
    g = torch.Generator().manual_seed(82)
    v, d_o = (t * torch.exp2(torch.randint(-spread, spread + 1, (B, H, T, 1), generator=g).float()).to(dev) for t in (v, d_o))
    lens = torch.tensor([T - (b * 37) % max(T // 2, 1) for b in range(B)], dtype=torch.int32, device=dev)
    qd, kd, vd = (t.clone().requires_grad_() for t in (q, k, v))
    out, lse = streaming_attention(qd, kd, vd, lens, C, R, return_lse=True)
    out.backward(d_o)
    want_lse = sa_oracle.windowed(q, k, v, lens, C, R, dtype=torch.float64)[1]
    assert ((lse.detach().double() - want_lse).abs() <= 32 * 2.0 ** -24 * want_lse.abs().clamp_min(1.0)).all()
    scale = D ** -0.5
    for b in range(B):
        L = int(lens[b])
        Q, K, V, G = (t[b, :, :L].double() for t in (q, k, v, d_o))
        chunk = torch.arange(L, device=dev) // C
        seen = (chunk[None] <= chunk[:, None]) & (chunk[None] >= chunk[:, None] - R)
        s = (Q @ K.transpose(1, 2).contiguous() * scale).masked_fill(~seen, -float("inf"))
        p = torch.softmax(s, -1)
        o = p @ V
        dp, delta = G @ V.transpose(1, 2).contiguous(), (o * G).sum(-1, keepdim=True)
        ds = p * (dp - delta)
        pt, dst = p.transpose(1, 2).contiguous(), ds.transpose(1, 2).contiguous()
        # An element of a result is a sum; the sizes of its terms, with the largest element of each row for all of the row's.
        # dS is known as well as the products that it is the difference of.
        top = lambda x: x.abs().amax(-1, keepdim=True)
        size = p * (G.norm(dim=-1, keepdim=True) * V.norm(dim=-1)[:, None] + (o * G).abs().sum(-1, keepdim=True))
        size_t = size.transpose(1, 2).contiguous()
        # 32 roundings of 2^-24 of those sizes: chains of fewer than 1024 terms, as a sum of n is off by about sqrt(n) roundings
        for name, got, want, terms in (("O", out, o, p @ top(V)), ("dQ", qd.grad, ds @ K * scale, size @ top(K) * scale),
                                       ("dK", kd.grad, dst @ Q * scale, size_t @ top(Q) * scale), ("dV", vd.grad, pt @ G, pt @ top(G))):
            err = (got[b, :, :L].detach().double() - want).abs()
            assert (err <= 32 * 2.0 ** -24 * terms).all(), f"{name}: {(err / terms).max().item() * 2 ** 24:.1f} roundings"
            assert not got[b, :, L:].any(), name
