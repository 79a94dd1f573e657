"""Head dimension 256 at the edges of its 32-row tiles and 128-row workgroups: lengths around them, windows of one tile and of many,
padded rows, q, k and v with strides of their own."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("T,C,R", [(1, 4, 0), (31, 8, 1), (33, 32, 0), (64, 64, 0), (97, 1000, 0), (129, 16, 2), (257, 10, 30),
                                  (383, 96, 2), (700, 33, 3)])
@pytest.mark.parametrize("packed", [False, True])
def test_wide_heads(T, C, R, dtype, eps, packed):
    from streaming_attention import streaming_attention

    dev = torch.device("cuda:0")
    B, H, D = 3, 2, 256
    q, k, v, d_o = (t.to(dtype).to(dev) for t in make_inputs(B, H, T, D, seed=81))
    if packed:
        q, k, v = torch.stack((q, k, v), 2).permute(0, 3, 2, 1, 4).contiguous().permute(2, 0, 3, 1, 4).unbind(0)
    lens = torch.tensor([T, max(T - 33, 1), T // 2], dtype=torch.int32, device=dev)
    qd, kd, vd = (t.detach().requires_grad_() for t in (q, k, v))
    out, lse = streaming_attention(qd, kd, vd, lens, C, R, return_lse=True)
    dq, dk, dv = torch.autograd.grad(out, (qd, kd, vd), d_o)
    want = sa_oracle.windowed(q, k, v, lens, C, R, d_out=d_o, dtype=torch.float64)
    # one rounding each of the result, of P or dS, and of O inside delta; P and dS enter sums whose terms' errors are
    # independent: three roundings of relative size eps, twice over for terms that cancel in dS
    for name, got, ref in zip(("O", "dQ", "dK", "dV"), (out.detach(), dq, dk, dv), (want[0], *want[2:])):
        got = got.double()
        assert torch.isfinite(got).all(), name
        rel = ((got - ref).norm() / ref.norm().clamp_min(1e-30)).item()
        assert ref.norm() == 0 or rel <= 6 * eps or (got - ref).abs().max() <= 6 * eps, f"{name}: relative error {rel:.2e}"
    assert (lse.double() - want[1]).abs().max() <= 1e-4
    for b in range(B):
        for t in (out, dq, dk, dv):
            assert not t[b, :, int(lens[b]):].any()
