"""Causal attention over more heads than one tail of the program order holds:
the order decides only when a block runs, so every batch's outputs are those
of its own launch, bit for bit."""
import pytest
import torch

from tests.conftest import announce
from warpir_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bsz,heads,hkv,seq,d", [(16, 9, 9, 2048, 64), (12, 11, 11, 2048, 128), (9, 16, 4, 2112, 128),
                                                 (3, 7, 7, 192, 64)])
def test_causal_order_does_not_change_any_head(gpu, bsz, heads, hkv, seq, d):
    announce(f"causal order B{bsz} H{heads}/{hkv} S{seq} D{d}")
    gen = torch.Generator(device="cuda").manual_seed(7)

    def normal(h):
        return torch.randn(bsz, h, seq, d, generator=gen, device="cuda", dtype=torch.bfloat16)

    q, k, v, do = normal(heads), normal(hkv), normal(hkv), normal(heads)
    o, lse = api.attention_forward(q, k, v, causal=True)
    grads = api.attention_backward(q, k, v, o, lse, do, causal=True)
    for i in range(bsz):
        s = slice(i, i + 1)
        o1, lse1 = api.attention_forward(q[s], k[s], v[s], causal=True)
        g1 = api.attention_backward(q[s], k[s], v[s], o1, lse1, do[s], causal=True)
        for whole, one in zip((o, lse, *grads), (o1, lse1, *g1)):
            assert torch.equal(whole[s], one)
