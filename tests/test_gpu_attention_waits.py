"""dQ of a launch whose workgroups start in turns: a wavefront that leaves its loop has its last loads landed before the others read them."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,B,H,T", [(128, 5, 8, 1920), (64, 5, 8, 1920)])
def test_repeated_attention_gradients_are_the_same(D, B, H, T):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(D)
    # (the heads of one buffer, a row of all of them 6 KB or 3 KB: the loads' usual way)
    qkv = torch.randn(B, T, 3, H, D, generator=g, device=dev).bfloat16()
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    go = torch.randn(B, T, H, D, generator=g, device=dev).bfloat16()
    scale = D ** -0.5
    o, lse = ops.attn_fwd(q, k, v, scale)
    want = [t.clone() for t in ops.attn_bwd(q, k, v, o, go, lse, scale)]
    for _ in range(40):
        for got, w in zip(ops.attn_bwd(q, k, v, o, go, lse, scale), want):
            assert torch.equal(got, w)
