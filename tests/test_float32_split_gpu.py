"""float32 kernels that form their products from bfloat16 parts (head dimensions 16 to 128): float32 accuracy at the edges of
the 32-row tiles and of the 128- and 256-row workgroups, on ordinary, very large and very small magnitudes."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu


# (B*H, T): two rows; tile and workgroup edges; B*H*ceil(T/256) below and from 256 on (the two forward shapes at D=128)
@pytest.mark.parametrize("B,H,T,C,R", [(1, 1, 2, 4, 1), (2, 3, 129, 32, 2), (2, 2, 257, 1000, 0), (1, 2, 415, 100, 1),
                                      (8, 16, 260, 48, 2), (8, 32, 96, 10, 3)])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("gain", [1.0, 1e15, 1e-15])
def test_float32_accuracy(B, H, T, C, R, D, gain):
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    q, k, v, d_o = (t.to(dev) for t in make_inputs(B, H, T, D, seed=71))
    # scores and dP keep their size; the tensors cover thirty decades (bfloat16 has float32's exponents)
    q, k, v, d_o = q * gain, k / gain, v * gain, d_o / gain
    lens = torch.tensor([T - (b * 37) % max(T // 2, 1) for b in range(B)], dtype=torch.int32, device=dev)
    qd, kd, vd = (t.clone().requires_grad_() for t in (q, k, v))
    out, lse = streaming_attention(qd, kd, vd, lens, C, R, return_lse=True)
    out.backward(d_o)
    want = sa_oracle.windowed(q, k, v, lens, C, R, d_out=d_o, dtype=torch.float64)
    # float32 rounds to 2^-24; a sum of n terms in any order is off by about sqrt(n) roundings, and the longest chain here
    # (scores over D, sums over a window of up to 415 keys, delta over D) has fewer than 1024 terms in all: 32 roundings
    bound = 32 * 2.0 ** -24
    for name, got, ref in zip(("O", "LSE", "dQ", "dK", "dV"), (out, lse, qd.grad, kd.grad, vd.grad), want):
        got = got.detach().double()
        assert torch.isfinite(got).all(), name
        rel = ((got - ref).norm() / ref.norm()).item()
        assert rel <= bound, f"{name}: relative error {rel:.2e}"
    for b in range(B):
        assert not out[b, :, int(lens[b]):].any() and not qd.grad[b, :, int(lens[b]):].any()


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("B,H", [(1, 2), (8, 32)])   # both forward shapes at D=128
def test_float32_range_ends(B, H, D):
    """Infinities and finite values beyond bfloat16's largest give what float32 arithmetic gives, not NaN.  Chunks are
    whole tiles, so that no masked key or query shares a tile with the planted values."""
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    T, C, R = 128, 32, 1
    q, k, v, d_o = (t.to(dev) for t in make_inputs(B, H, T, D, seed=72))
    lowest, inf = torch.finfo(torch.float32).min, float("inf")
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, :, 5, 0] = lowest             # score far below all others: the key has no weight
    k[:, :, 70, 0] = -inf              # score -inf: no weight either, but 0 * inf in dQ
    v[:, :, 33, 1], v[:, :, 34, 2] = inf, -inf
    v[:, :, 100, 3] = lowest / 2 ** 10
    v[:, :, 5, 4] = -lowest            # 0 * finite
    qd, kd, vd = (t.clone().requires_grad_() for t in (q, k, v))
    out = streaming_attention(qd, kd, vd, None, C, R)
    want = sa_oracle.windowed(q, k, v, None, C, R, dtype=torch.float64)[0]
    got = out.detach().double()
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and not torch.isnan(got).any()
    assert torch.equal(got[torch.isinf(want)].sign(), want[torch.isinf(want)].sign())
    fin = torch.isfinite(want)
    # 32 roundings as above, relative to the largest term of the sum (position 100 dwarfs the others in element 3)
    for d in range(D):
        scale = want[..., d][fin[..., d]].abs().max()
        assert ((got - want)[..., d][fin[..., d]].abs() <= 32 * 2.0 ** -24 * max(scale, 8.0)).all(), d

    # an infinite dO reaches dV of every key its query sees, and no other element of dV
    kd.data[:, :, 70, 0] = 0.0
    vd.data.copy_(torch.where(torch.isinf(v), torch.zeros_like(v), v))
    d_o[:, :, 40, 6] = inf
    out = streaming_attention(qd, kd, vd, None, C, R)
    dv = torch.autograd.grad(out, vd, d_o)[0]
    bad = ~torch.isfinite(dv)
    expect = torch.zeros_like(bad)
    expect[:, :, :64, 6] = True
    expect[:, :, 5, 6] = False         # its weight is zero: 0 * inf
    assert torch.equal(torch.isinf(dv), expect) and torch.isnan(dv[:, :, 5, 6]).all()
    assert torch.equal(bad.sum(), expect.sum() + B * H)


# magnitudes whose bfloat16 parts fall below or above bfloat16's range: tiny and huge operands that balance each other, and tiny
# values or upstream gradients by themselves (dS is tiny then too)
@pytest.mark.parametrize("B,H,T,C,R", [(2, 2, 129, 32, 2), (1, 2, 415, 100, 1), (8, 32, 260, 48, 2)])   # 64, 128 and 256 rows
@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("gq,gv,gd", [(1e33, 1e-33, 1e33), (1e36, 1e-36, 1e36), (1e-36, 1e36, 1e-36), (1.0, 1.0, 1e-36),
                                      (1.0, 1e-36, 1.0), (1.0, 1e18, 1e-36)])
def test_float32_accuracy_at_the_ends_of_the_range(B, H, T, D, C, R, gq, gv, gd):
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    q, k, v, d_o = (t.to(dev) for t in make_inputs(B, H, T, D, seed=73))
    q, k, v, d_o = q * gq, k / gq, v * gv, d_o * gd
    lens = torch.tensor([T - (b * 37) % (T // 2) for b in range(B)], dtype=torch.int32, device=dev)
    qd, kd, vd = (t.clone().requires_grad_() for t in (q, k, v))
    out, lse = streaming_attention(qd, kd, vd, lens, C, R, return_lse=True)
    out.backward(d_o)
    want = sa_oracle.windowed(q, k, v, lens, C, R, d_out=d_o, dtype=torch.float64)
    for name, got, ref in zip(("O", "LSE", "dQ", "dK", "dV"), (out, lse, qd.grad, kd.grad, vd.grad), want):
        rel = ((got.detach().double() - ref).norm() / ref.norm()).item()
        assert rel <= 32 * 2.0 ** -24, f"{name}: relative error {rel:.2e}"   # as in test_float32_accuracy


@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B", [1, 8, 33])   # 64-row workgroups up to head dimension 64, 128-row ones, more than one round of them
@pytest.mark.parametrize("dp", [float("inf"), 2.0 ** 128 * (1 - 2.0 ** -10)])   # the latter rounds to an infinite bfloat16
def test_float32_ds_at_the_end_of_the_range(B, D, dp):
    """An infinite dS gives signed infinities (NaN against a zero), a finite one that rounds to an infinite bfloat16 finite
    gradients, as float32 arithmetic does."""
    dev = torch.device("cuda:0")
    H, T, C, q0, j0 = 4, 128, 32, 37, 50   # one key tile per chunk; query 37 and key 50 share one
    g = torch.Generator().manual_seed(3)
    q, k, v, o, d_o = (torch.zeros(B, H, T, D, device=dev) for _ in range(5))
    q[..., 0] = (torch.rand(B, H, T, generator=g) + 0.5).to(dev) * 2.0 ** -10   # scores are zero: q and k are orthogonal
    k[..., 1:] = torch.randn(B, H, T, D - 1, generator=g).to(dev) * 2.0 ** -10
    v[:, :, j0, 0], d_o[:, :, q0, 0] = 2.0 ** 100, dp * 2.0 ** -100 if dp < float("inf") else 2.0 ** 30
    lse = torch.zeros(B, H, T, device=dev)   # every probability is one
    dq, dk, dv = torch.ops.alexdremov_streaming_attention.backward(q, k, v, None, o, lse, d_o, C, 0, 1.0, False, False, "ieee")
    ds = torch.tensor(dp)
    want_q, want_k = ds * k[:, :, j0].cpu(), ds * q[:, :, q0].cpu()
    torch.testing.assert_close(dq[:, :, q0].cpu(), want_q, rtol=2.0 ** -20, atol=0, equal_nan=True)
    torch.testing.assert_close(dk[:, :, j0].cpu(), want_k, rtol=2.0 ** -20, atol=0, equal_nan=True)
    rest_q, rest_k = dq.clone(), dk.clone()
    rest_q[:, :, q0], rest_k[:, :, j0] = 0.0, 0.0
    assert not rest_q.any() and not rest_k.any()
    assert torch.equal(dv[:, :, 32:64, 0], d_o[:, :, q0, :1].expand(B, H, 32)) and not dv[:, :, :32].any()
