"""Dense ragged batches, and chunks whose windows reach over all of T, whose workgroups are dispatched by the lengths of their sequences: every sequence has the bits that it has alone
(where there is nothing to order), with lengths that are equal, none, beyond T and negative, up to the most batch entries and (batch entry,
head) pairs that are ordered."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.float16, 16), (torch.bfloat16, 32), (torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 256),
                                     (torch.float32, 16), (torch.float32, 64), (torch.float32, 128)], ids=str)
@pytest.mark.parametrize("C,R", [(None, None), (250, 6)])   # None: self_attention
@pytest.mark.parametrize("B,H,T", [(2, 28, 769), (9, 8, 1100), (32, 16, 768), (17, 8, 1281)])
def test_each_sequence_as_if_alone(B, H, T, dtype, D, C, R):
    from self_attention import self_attention
    from streaming_attention import streaming_attention

    def run(q, k, v, lens):   # O, and the LSE of a streaming call
        if C is None:
            return (self_attention(q, k, v, lens),)
        return streaming_attention(q, k, v, lens, C, R, return_lse=True)

    dev = torch.device("cuda:0")
    assert B * H % 8 == 0 and B * H <= 512 and B * H * -(-T // 256) > 256 or B == 2
    g = torch.Generator(device=dev).manual_seed(B + T)
    q, k, v = (torch.randn(B, H, T, D, generator=g, device=dev).to(dtype) for _ in range(3))
    r = torch.Generator().manual_seed(B)
    lens = torch.randint(1, T + 1, (B,), generator=r, dtype=torch.int32)
    lens[0], lens[-1] = T, T + 7
    if B > 4:
        lens[1], lens[2], lens[4] = 0, -3, lens[3]
    outs = run(q, k, v, torch.stack((lens, lens * 0 + 5), 1).to(dev)[:, 0])   # (every other element)
    for b in range(B):
        n = min(max(int(lens[b]), 0), T)
        for out, one in zip(outs, run(q[b:b + 1], k[b:b + 1], v[b:b + 1], lens[b:b + 1].to(dev))):
            assert torch.equal(out[b:b + 1], one), b
            assert not out[b, :, n:].any() and (n == 0 or out[b, :, :n].any())
