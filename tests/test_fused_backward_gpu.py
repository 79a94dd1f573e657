"""The one-launch backward for short windows: against the float64 oracle and against the two launches it replaces (pinned
variants), at lengths around its 64-row tiles and 128-row workgroups and at windows on both sides of the rule that picks it."""
import pytest
import torch

from oracle import sa_oracle
from tests.helpers import assert_close, make_inputs

pytestmark = pytest.mark.gpu


# query rows that a workgroup walks: up to 320 are chosen at D=64, up to 256 at D=32, 384 run the two launches.  Chunks of 112 and
# 256 end more than a tile beyond a workgroup's rows, whose own key rows are then read from memory again.
@pytest.mark.parametrize("C,R,rows", [(128, 0, 128), (32, 2, 192), (64, 2, 256), (256, 0, 256), (10, 9, 320), (112, 0, 320),
                                      (100, 0, 384), (50, 2, 384)])
@pytest.mark.parametrize("T,lens", [(1, [1, 1]), (64, [64, 3]), (129, [129, 128]), (193, [0, 65]), (700, [700, 385])])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_one_launch_backward(dtype, D, T, lens, C, R, rows):
    from streaming_attention import _lib

    lib = _lib.load()
    assert lib.sa_launch_choice(D, C, R, 3) == (rows <= (320 if D == 64 else 256))
    dev = torch.device("cuda:0")
    B, H = 2, 3
    q, k, v, d_o = make_inputs(B, H, T, D, seed=81, dtype=dtype)
    ld = torch.tensor(lens, dtype=torch.int32)
    # [B,T,H,D]-stored q and dO: strided rows through the tile copies and the row sums
    qd, gd = (t.to(dev).transpose(1, 2).contiguous().transpose(1, 2) for t in (q, d_o))
    kd, vd, le = k.to(dev), v.to(dev), ld.to(dev)
    fwd = torch.ops.alexdremov_streaming_attention.forward
    bwd = torch.ops.alexdremov_streaming_attention.backward
    o, lse = fwd(qd, kd, vd, le, C, R, D ** -0.5, False, True, False, "ieee")
    got = bwd(qd, kd, vd, le, o, lse, gd, C, R, D ** -0.5, False, False, "ieee")
    ref = sa_oracle.dense_f64(q, k, v, ld, C, R, d_out=d_o)
    for name, g in zip(("dQ", "dK", "dV"), got):
        assert_close(name, g, ref[name], dtype)
        for b, n in enumerate(lens):
            assert not g[b, :, n:].any()
    try:
        assert lib.sa_tune_override(1, 0) == 0      # pinned variants run as launches of their own
        two = bwd(qd, kd, vd, le, o, lse, gd, C, R, D ** -0.5, False, False, "ieee")
    finally:
        lib.sa_tune_override(1, -1)
    # same products in the same order; only delta is summed in another order, one float32 rounding before dS is rounded
    eps = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    for name, g, w in zip(("dQ", "dK", "dV"), got, two):
        assert (g.float() - w.float()).abs().max().item() <= 4 * eps * max(w.float().abs().max().item(), 1.0), name
