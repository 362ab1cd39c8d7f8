"""The split attention backward (launches that leave CUs idle) against the
autograd oracle and the tiled kernels, at the edges of its tiles and range."""
import pytest
import torch

from oracle.torch_ref import attention_bwd_ref, rel_err, seeded_normal
from tests.conftest import announce
from warpir_amd import api

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def taken(monkeypatch):
    """Counts the backward passes that take the split kernels."""
    count, real = [], api._attention_bwd_split
    monkeypatch.setattr(api, "_attention_bwd_split", lambda *a: count.append(1) or real(*a))
    monkeypatch.setattr(api, "_backward_plans", api.Plans("attention_backward"))
    return count


def _inputs(bsz, heads, seq, d, causal):
    q, k, v, do = (seeded_normal((bsz, heads, seq, d), s) for s in range(4))
    dev = [x.cuda() for x in (q, k, v, do)]
    o, lse = api.attention_forward(*dev[:3], causal=causal)
    return (q, k, v, do), (*dev[:3], o, lse, dev[3])


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bsz,heads,seq", [(1, 1, 64), (2, 3, 128), (1, 5, 192), (1, 2, 320), (1, 8, 1024)])
def test_split_backward_matches_autograd(gpu, taken, bsz, heads, seq, d, causal):
    announce(f"split backward B{bsz} H{heads} S{seq} D{d} causal={causal}")
    host, dev = _inputs(bsz, heads, seq, d, causal)
    ref = attention_bwd_ref(*host, causal=causal)
    big = torch.full((3, bsz, heads, seq + 64, d), -7.0, dtype=torch.bfloat16, device="cuda")
    dvec = torch.empty(bsz, heads, seq, device="cuda")
    for _ in range(2):   # the call and its plan
        big[:, :, :, :seq] = 0
        got = api.attention_backward(*dev, *(x[:, :, :seq] for x in big), dvec, causal=causal)
        for x, y in zip(got, ref):   # the tiled kernels' bar
            assert rel_err(x.cpu().float(), y) <= 1e-2
        assert bool((big[:, :, :, seq:] == -7.0).all())
        want = (dev[5].float() * dev[3].float()).sum(-1)
        assert torch.allclose(dvec, want, rtol=1e-4, atol=1e-4)
    assert len(taken) == 1


@pytest.mark.parametrize("causal", [False, True])
def test_split_backward_reads_packed_views_as_the_tiled_kernels_do(gpu, taken, causal):
    q, k, v = seeded_normal((2, 192, 3, 2, 64), 5).cuda().permute(2, 0, 3, 1, 4)
    do = seeded_normal((2, 192, 2, 64), 6).cuda().transpose(1, 2)
    o, lse = api.attention_forward(q, k, v, causal=causal)
    got = api.attention_backward(q, k, v, o, lse, do, causal=causal)
    assert taken
    dense = api.attention_backward(*(x.contiguous() for x in (q, k, v, o)), lse, do.contiguous(), causal=causal)
    assert all(torch.equal(x, y) for x, y in zip(got, dense))
    # a workspace (read by grouped heads only) keeps the tiled kernels
    tiled = api.attention_backward(q, k, v, o, lse, do, causal=causal, workspace=torch.empty(1, device="cuda"))
    for x, y in zip(got, tiled):   # the same products summed in another order: one bf16 rounding
        assert rel_err(x.cpu().float(), y.cpu().float()) <= 2.0 ** -7


def test_split_backward_is_left_at_its_limits(gpu, taken):
    for bsz, heads, hkv, seq, want in ((16, 1, 1, 1024, 1), (17, 1, 1, 1024, 0), (1, 4, 2, 128, 0)):
        taken.clear()
        q = torch.zeros(bsz, heads, seq, 64, dtype=torch.bfloat16, device="cuda")
        k = torch.zeros(bsz, hkv, seq, 64, dtype=torch.bfloat16, device="cuda")
        o, lse = api.attention_forward(q, k, k.clone())
        api.attention_backward(q, k, k.clone(), o, lse, q.clone())
        assert len(taken) == want


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["k", "v", "q", "do"])
def test_split_backward_special_values(gpu, taken, monkeypatch, where, bad, d, causal):
    """A row of NaN or infinities spoils every gradient that depends on it, and
    no element that the tiled kernels keep finite."""
    announce(f"split backward {where} {bad} D{d} causal={causal}")
    host = dict(zip(("q", "k", "v", "do"), (seeded_normal((1, 2, 256, d), s) for s in range(4))))
    host[where][0, 1, 200] = bad
    q, k, v, do = (host[x].cuda() for x in ("q", "k", "v", "do"))
    o, lse = api.attention_forward(q, k, v, causal=causal)
    got = api.attention_backward(q, k, v, o, lse, do, causal=causal)
    assert taken
    monkeypatch.setattr(api, "_split_bwd_fits", lambda *a: False)
    monkeypatch.setattr(api, "_backward_plans", api.Plans("attention_backward"))
    tiled = api.attention_backward(q, k, v, o, lse, do, causal=causal)
    assert len(taken) == 1
    exact = attention_bwd_ref(*(host[x] for x in ("q", "k", "v", "do")), causal=causal)
    # the query rows whose O, LSE or dP see the bad row, and the keys that those rows see
    i = torch.arange(256)
    rows = (i >= 200 if causal else i >= 0) if where in ("k", "v") else i == 200
    keys = i <= (255 if where in ("k", "v") else 200) if causal else i >= 0
    spoiled = rows, keys, keys & (where != "v")
    for g, t, e, bad_rows in zip(got, tiled, exact, spoiled):
        g, t = g.cpu().float(), t.cpu().float()
        assert not bool(g[0, 1, bad_rows].isfinite().any())
        assert int((t.isfinite() & ~g.isfinite()).sum()) == 0
        assert bool(g[0, 0].isfinite().all())   # the other head
        # (where the fp32 reference is finite: its 0 * NaN of masked scores is NaN, theirs often not formed)
        both = g.isfinite() & e.isfinite()
        assert rel_err(g[both], e[both]) <= 1e-2


@pytest.mark.parametrize("bsz,heads,seq,causal", [(32, 8, 64, True), (16, 8, 128, False), (8, 8, 256, True)])
def test_many_short_heads_keep_the_tiled_kernels(gpu, taken, monkeypatch, bsz, heads, seq, causal):
    """512 programs of a few tiles: two rounds of the split kernels are slower."""
    split, real = [], api._attention_split_kv
    monkeypatch.setattr(api, "_attention_split_kv", lambda *a: split.append(1) or real(*a))
    monkeypatch.setattr(api, "_forward_plans", api.Plans("attention_forward"))
    host, dev = _inputs(bsz, heads, seq, 64, causal)
    got = api.attention_backward(*dev, causal=causal)
    assert not taken and not split
    for x, y in zip(got, attention_bwd_ref(*host, causal=causal)):
        assert rel_err(x.cpu().float(), y) <= 1e-2
