"""float32: rows, channels and single elements of very different magnitude side by side, those that a query or key does not see included,
at the edges of tiles, workgroups and windows."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu


# short and long windows, B*H*ceil(T/256) on both sides of 256 at D=128, grids of two- and four-wave workgroups, remainders of a row and of a tile
SIZES = [(1, 2, 300, 64, 64, 2), (1, 2, 300, 64, 191, 0), (2, 16, 641, 64, 96, 1), (1, 1, 2, 64, 192, 0), (1, 2, 700, 32, 256, 1),
         (1, 2, 700, 32, 511, 0), (3, 16, 545, 32, 128, 3), (1, 2, 300, 16, 40, 2), (3, 16, 545, 16, 128, 3), (1, 2, 300, 128, 10, 9),
         (8, 33, 97, 128, 32, 1), (1, 3, 513, 128, 1000, 0), (1, 1, 1, 128, 1, 0), (1, 2, 130, 256, 40, 1)]


def ragged(B, T, dev):
    return torch.tensor([T - (b * 37) % max(T // 2, 1) for b in range(B)], dtype=torch.int32, device=dev)


def run(q, k, v, lens, C, R, d_o):
    from streaming_attention import streaming_attention

    q, k, v = (t.clone().requires_grad_() for t in (q, k, v))
    out, lse = streaming_attention(q, k, v, lens, C, R, return_lse=True)
    return [out.detach(), *torch.autograd.grad(out, (q, k, v), d_o), lse.detach()]


@pytest.mark.parametrize("B,H,T,D,C,R", SIZES)
@pytest.mark.parametrize("span", [20, 40])
def test_powers_of_two_on_channels_change_no_bit(B, H, T, D, C, R, span):
    """Channels of K and V times powers of two, those of Q and dO divided by them: every product of a score or of dP is what it was, and
    every sum over keys or queries is in units of one power.  Float32 arithmetic gives the same significands; so does whatever holds
    all 24 bits of an element next to others that are 2^(2 * span) times as large."""
    dev = torch.device("cuda:0")
    q, k, v, d_o = (t.to(dev) for t in make_inputs(B, H, T, D, seed=84))
    lens = ragged(B, T, dev)
    g = torch.Generator().manual_seed(85)
    fk, fv = (torch.exp2(torch.randint(-span, span + 1, (D,), generator=g).float()).to(dev) for _ in range(2))
    plain = run(q, k, v, lens, C, R, d_o)
    scaled = run(q / fk, k * fk, v * fv, lens, C, R, d_o / fv)
    for name, x, y, f in zip(("O", "dQ", "dK", "dV", "LSE"), plain, scaled, (fv, fk, 1 / fk, 1 / fv, 1.0)):
        assert torch.equal(x * f, y), f"{name}: {((x * f - y).double().norm() / (x * f).double().norm()).item():.2e}"


@pytest.mark.parametrize("B,H,T,D,C,R", SIZES)
@pytest.mark.parametrize("spread", [0, 12])   # rows of V and dO times powers of two up to this, either way
def test_rows_of_different_magnitude(B, H, T, D, C, R, spread):
    dev = torch.device("cuda:0")
    q, k, v, d_o = (t.to(dev) for t in make_inputs(B, H, T, D, seed=81))
    g = torch.Generator().manual_seed(82)
    v, d_o = (t * torch.exp2(torch.randint(-spread, spread + 1, (B, H, T, 1), generator=g).float()).to(dev) for t in (v, d_o))
    lens = ragged(B, T, dev)
    out, dq, dk, dv, lse = run(q, k, v, lens, C, R, d_o)
    want_lse = sa_oracle.windowed(q, k, v, lens, C, R, dtype=torch.float64)[1]
    assert ((lse.double() - want_lse).abs() <= 32 * 2.0 ** -24 * want_lse.abs().clamp_min(1.0)).all()
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
        # An element of a result is a sum; the sizes of its terms.  dS is known as well as the products that it is the difference of.
        size = p * (G.abs() @ V.abs().transpose(1, 2).contiguous() + (o * G).abs().sum(-1, keepdim=True))
        size_t = size.transpose(1, 2).contiguous()
        # 32 roundings of 2^-24 of those sizes: chains of fewer than 1024 terms, as a sum of n is off by about sqrt(n) roundings
        for name, got, want, terms in (("O", out, o, p @ V.abs()), ("dQ", dq, ds @ K * scale, size @ K.abs() * scale),
                                       ("dK", dk, dst @ Q * scale, size_t @ Q.abs() * scale), ("dV", dv, pt @ G, pt @ G.abs())):
            err = (got[b, :, :L].double() - want).abs()
            assert (err <= 32 * 2.0 ** -24 * terms).all(), f"{name}: {(err / terms).max().item() * 2 ** 24:.1f} roundings"
            assert not got[b, :, L:].any(), name
