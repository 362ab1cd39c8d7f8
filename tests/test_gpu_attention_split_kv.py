"""The split-key attention forward (launches that leave CUs idle) against the
fp32 oracle and the tiled kernel, at the edges of its tiles and of its range."""
import math

import pytest
import torch

from oracle.torch_ref import attention_ref, rel_err, seeded_normal
from tests.conftest import announce
from warpir_amd import api, kernels

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def taken(monkeypatch):
    """Counts the launches that take the split-key kernel."""
    count, real = [], api._attention_split_kv
    monkeypatch.setattr(api, "_attention_split_kv", lambda *a: count.append(1) or real(*a))
    for name in ("_forward_plans",):
        monkeypatch.setattr(api, name, api.Plans(name))
    return count


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bsz,heads,hkv,seq", [(1, 1, 1, 64), (2, 3, 1, 128), (1, 6, 3, 192), (1, 5, 5, 320),
                                               (1, 8, 8, 1024), (1, 1, 1, 4160)])
def test_split_kv_matches_the_oracle(gpu, taken, bsz, heads, hkv, seq, d, causal):
    announce(f"split-kv B{bsz} H{heads}/{hkv} S{seq} D{d} causal={causal}")
    q = seeded_normal((bsz, heads, seq, d), 0)
    k, v = (seeded_normal((bsz, hkv, seq, d), s) for s in (1, 2))
    ref, ref_lse = attention_ref(q, *(x.repeat_interleave(heads // hkv, 1) for x in (k, v)), scale=1 / math.sqrt(d),
                                 causal=causal)
    for _ in range(2):   # the call and its plan
        big = torch.full((bsz, heads, seq + 64, d), -7.0, dtype=torch.bfloat16, device="cuda")
        out = big[:, :, :seq]
        o, lse = api.attention_forward(q.cuda(), k.cuda(), v.cuda(), causal=causal, out=out)
        # as the tiled forward's bar: probabilities and O rounded to bf16
        assert rel_err(o.cpu(), ref) <= 1e-2 and (lse.cpu() - ref_lse).abs().max() <= 1e-4
        assert bool((big[:, :, seq:] == -7.0).all())
    assert len(taken) == 1


@pytest.mark.parametrize("d", [64, 128])
def test_split_kv_reads_packed_views(gpu, taken, d):
    qkv = seeded_normal((2, 192, 3, 2, d), 5).cuda().permute(2, 0, 3, 1, 4)
    o, lse = api.attention_forward(*qkv, causal=True)
    o2, lse2 = api.attention_forward(*(x.contiguous() for x in qkv), causal=True)
    assert taken and torch.equal(o, o2) and torch.equal(lse, lse2)


@pytest.mark.parametrize("causal", [False, True])
def test_split_kv_special_scores(gpu, taken, causal):
    """A wave whose own tiles score -inf in a row adds nothing to it; NaN and
    +inf keys make NaN of the rows that see them, and of no others."""
    q, k, v = (seeded_normal((1, 1, 256, 64), s) for s in (0, 1, 2))
    q = q.abs()
    k[0, 0, 64:128] = float("-inf")          # one wave's whole tile
    o, lse = api.attention_forward(q.cuda(), k.cuda(), v.cuda(), causal=causal)
    keep = torch.cat([torch.arange(64), torch.arange(128, 256)])
    rows = torch.arange(64) if causal else torch.arange(256)
    ref, _ = attention_ref(q, k[:, :, keep], v[:, :, keep], scale=0.125)
    if causal:
        ref, _ = attention_ref(q[:, :, :64], k[:, :, :64], v[:, :, :64], scale=0.125, causal=True)
    assert bool(o.isfinite().all()) and bool(lse.isfinite().all())
    assert rel_err(o.cpu()[:, :, rows], ref) <= 1e-2
    for bad in (float("nan"), float("inf")):
        k2 = seeded_normal((1, 1, 256, 64), 1)
        k2[0, 0, 200] = bad
        o, lse = (x.cpu() for x in api.attention_forward(q.cuda(), k2.cuda(), v.cuda(), causal=causal))
        seen = torch.arange(256) >= 200 if causal else torch.ones(256, dtype=torch.bool)
        assert bool(o[0, 0, seen].isnan().all()) and bool(o[0, 0, ~seen].isfinite().all())
        tiled = kernels.handle("mha_d64_causal" if causal else "mha_d64")
        o3, l3 = torch.empty_like(o, device="cuda"), torch.empty_like(lse, device="cuda")
        tiled(Q=q.cuda(), K=k2.cuda(), V=v.cuda(), N=256, O=o3, L=l3)
        assert torch.equal(o.isnan(), o3.cpu().isnan()) and torch.equal(lse.isnan(), l3.cpu().isnan())


def test_split_kv_is_left_at_its_limits(gpu, taken):
    for bsz, seq, causal, want in ((8, 1024, False, 1), (9, 1024, False, 0), (16, 1024, True, 1), (17, 1024, True, 0)):
        taken.clear()
        q = torch.zeros(bsz, 1, seq, 64, dtype=torch.bfloat16, device="cuda")
        api.attention_forward(q, torch.zeros_like(q), torch.zeros_like(q), causal=causal)
        assert len(taken) == want
    with pytest.raises(ValueError, match="multiple of the KV tile"):
        api.attention_forward(*(torch.zeros(1, 1, 96, 64, dtype=torch.bfloat16, device="cuda") for _ in range(3)))


def test_few_256_row_blocks_take_128_row_blocks(gpu, taken):
    q, k, v = (seeded_normal((3, 8, 704, 128), s).cuda() for s in range(3))
    o, lse = api.attention_forward(q, k, v)
    o2, lse2 = api.attention_forward(q, k, v, variant="mha_d128_w4")
    assert not taken and torch.equal(o, o2) and torch.equal(lse, lse2)
    q, k, v = (seeded_normal((6, 8, 896, 128), s).cuda() for s in range(3))   # 336 of them: 256-row blocks
    o, lse = api.attention_forward(q, k, v)
    o2, lse2 = api.attention_forward(q, k, v, variant="mha_d128")
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
