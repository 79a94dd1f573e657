"""Head dimension 16, 16-bit elements: every form that the windows pick (workgroups of two and four waves, the backward in one launch and
in two, long windows) against the float64 oracle at lengths around tiles and workgroups, and the same values in slices that 32-bit
byte offsets do not reach, which run the first kernels."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import assert_close, assert_close_lse, make_inputs

pytestmark = pytest.mark.gpu


def run(q, k, v, d_o, lens, C, R, scale=None):
    from streaming_attention import streaming_attention

    o, lse = streaming_attention(q, k, v, lens, C, R, sm_scale=scale, return_lse=True)
    return [o, *torch.autograd.grad(o, (q, k, v), d_o), lse]


# forward in two waves below chunks of 128 and up to 512 keys, the backward in one launch up to 256 rows in reach (in two waves below chunks
# of 128), long windows from 1024 keys on (both chunk and back limited to T)
WINDOWS = [(7, 0), (8, 3), (10, 9), (32, 2), (64, 1), (33, 6), (128, 0), (128, 1), (130, 4), (700, 1)]


@pytest.mark.parametrize("C,R", WINDOWS)
@pytest.mark.parametrize("T,lens", [(1, [1, 1]), (31, [31, 2]), (33, [33, 32]), (65, [64, 65]), (129, [128, 129]), (161, [0, 97]), (700, [700, 385])])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_against_the_oracle(dtype, T, lens, C, R):
    dev = torch.device("cuda:0")
    q, k, v, d_o = make_inputs(2, 3, T, 16, seed=61, dtype=dtype)
    ld = torch.tensor(lens, dtype=torch.int32)
    # q, k and v read in place from one [B, T, 3, H, D] projection
    packed = torch.stack((q, k, v), 2).permute(0, 3, 2, 1, 4).contiguous().to(dev)   # [B, T, 3, H, D]
    qd, kd, vd = (packed[:, :, i].transpose(1, 2).requires_grad_() for i in range(3))
    got = run(qd, kd, vd, d_o.to(dev), ld.to(dev), C, R)
    ref = sa_oracle.dense_f64(q, k, v, ld, C, R, d_out=d_o)
    for name, g in zip(("O", "dQ", "dK", "dV"), got):
        assert_close(name, g, ref[name], dtype)
        for b, n in enumerate(lens):
            assert not g[b, :, n:].any()
    assert_close_lse(got[4], ref["LSE"].copy(), dtype)


@pytest.mark.parametrize("scale", [-0.3, 0.0, 0.25])
@pytest.mark.parametrize("C,R", [(16, 2), (64, 5), (128, 1)])
@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)], ids=str)
def test_slices_beyond_32_bit_offsets(dtype, eps, C, R, scale):
    """The tile kernels and the first kernels differ by the order of their sums and by the probabilities' reference, so by a rounding of
    each probability and dS (eps each) and one of the result: relative in the 2-norm, as the roundings of a row are independent."""
    dev = torch.device("cuda:0")
    T, H = 140, 2
    stride = -(-(1 << 31) // (T + 1024) // 64) * 64 + 64   # elements: (T + 1024) rows are more than 4 GiB
    q, k, v, d_o = (t.to(dev) for t in make_inputs(1, H, T, 16, seed=62, dtype=dtype))
    room = torch.empty(T * stride, dtype=dtype, device=dev)
    far = []
    for i, t in enumerate((q, k, v)):
        view = room.as_strided((1, H, T, 16), (48 * H, 48, stride, 1), 16 * i)
        view.copy_(t)
        far.append(view.requires_grad_())
    lens = torch.tensor([133], dtype=torch.int32, device=dev)
    near = [t.clone().requires_grad_() for t in (q, k, v)]
    a, b = (run(*x, d_o, lens, C, R, scale) for x in (near, far))
    ref = sa_oracle.dense_f64(q.cpu(), k.cpu(), v.cpu(), lens.cpu(), C, R, sm_scale=scale, d_out=d_o.cpu())
    for name, x, y in zip(("O", "dQ", "dK", "dV"), a, b):
        assert_close(name, x, ref[name], dtype)
        assert_close(name, y, ref[name], dtype)
        assert (x.double() - y.double()).norm() <= 3 * eps * y.double().norm()
    assert (a[4] - b[4]).abs().max().item() <= 1e-5   # float32 sums of up to 140 terms, 2^-24 each
