"""The tiled attention kernels at sizes where api would take the split ones:
every tile edge of the forward and the backward against the oracle, with the
route asserted."""
import pytest
import torch

from oracle.torch_ref import attention_bwd_ref, attention_ref, rel_err, seeded_normal
from tests.conftest import announce
from warpir_amd import api, kernels

TOL = 1e-2
pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 64), (1, 1, 128), (2, 3, 192), (1, 2, 320), (2, 1, 704), (1, 2, 1088)]


@pytest.fixture(autouse=True)
def launched(monkeypatch):
    """Names of the generated kernels launched; the split routes are closed."""
    log, real = [], kernels.handle

    def handle(name):
        log.append(name)
        return real(name)

    monkeypatch.setattr(kernels, "handle", handle)
    monkeypatch.setattr(api, "_split_bwd_fits", lambda *a: False)
    monkeypatch.setattr(api, "_split_kv_fits", lambda *a: False)
    for name in ("_attention_split_kv", "_attention_bwd_split"):
        monkeypatch.setattr(api, name, None)
    for name in ("_forward_plans", "_backward_plans"):
        monkeypatch.setattr(api, name, api.Plans(name))
    return log


def _inputs(b, h, s, d, packed, seed=0):
    if packed:
        q, k, v = seeded_normal((b, s, 3, h, d), seed).permute(2, 0, 3, 1, 4)
        base = torch.stack([q, k, v]).permute(1, 3, 0, 2, 4).contiguous().cuda()
        return (q, k, v), tuple(base.permute(2, 0, 3, 1, 4))
    host = tuple(seeded_normal((b, h, s, d), seed + i) for i in range(3))
    return host, tuple(x.cuda() for x in host)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("b,h,s", SHAPES)
def test_tiled_attention_matches_the_oracle(gpu, launched, b, h, s, d, causal, packed):
    announce(f"tiled attention B{b} H{h} S{s} D{d} causal={causal} packed={packed}")
    (q, k, v), dev = _inputs(b, h, s, d, packed)
    do = seeded_normal((b, h, s, d), 9)
    ref, ref_lse = attention_ref(q, k, v, causal=causal)
    grads_ref = attention_bwd_ref(q, k, v, do, causal=causal)
    for _ in range(2):   # the calls and their plans
        o, lse = api.attention_forward(*dev, causal=causal)
        grads = api.attention_backward(*dev, o, lse, do.cuda(), causal=causal)
        assert rel_err(o.cpu(), ref) <= TOL
        assert float((lse.cpu() - ref_lse).abs().max()) <= 1e-3 * float(ref_lse.abs().max()) + 1e-3
        for got, want in zip(grads, grads_ref):
            assert rel_err(got.cpu().float(), want) <= TOL
    sfx = f"d{d}" + "_causal" * causal
    forward = "mha_d128_w4" if (d, causal) == (128, False) else f"mha_{sfx}"
    assert forward in launched and {f"mha_bwd_dq_prep_{sfx}", f"mha_bwd_dkdv_{sfx}"} <= set(launched)


@pytest.mark.parametrize("d,causal", [(64, False), (64, True), (128, True), (128, False)])
@pytest.mark.parametrize("b,h,s", SHAPES)
def test_tiled_forward_variants_match_the_oracle(gpu, b, h, s, d, causal):
    """By name, at every edge (mha_d128: 256-row blocks)."""
    (q, k, v), dev = _inputs(b, h, s, d, False, seed=20)
    o, lse = api.attention_forward(*dev, causal=causal, variant=f"mha_d{d}" + "_causal" * causal)
    ref, ref_lse = attention_ref(q, k, v, causal=causal)
    assert rel_err(o.cpu(), ref) <= TOL
    assert float((lse.cpu() - ref_lse).abs().max()) <= 1e-3 * float(ref_lse.abs().max()) + 1e-3
