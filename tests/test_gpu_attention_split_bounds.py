"""Destinations that do not have the result's shape, and the split attention
kernels: elements that do not fit are dropped, as by every tiled kernel.  The
destinations are views inside larger allocations filled with a marker."""
import pytest
import torch

from oracle.torch_ref import attention_bwd_ref, attention_ref, rel_err, seeded_normal
from tests.conftest import announce
from warpir_amd import api, kernels
from warpir_amd.plans import NO_RECORDING

pytestmark = pytest.mark.gpu

B, H, S = 2, 3, 128
MARK = -7.0


@pytest.fixture(autouse=True)
def fresh(monkeypatch):
    for name in ("_forward_plans", "_backward_plans"):
        monkeypatch.setattr(api, name, api.Plans(name))


def _view(shape, full, dtype=torch.bfloat16):
    """(allocation of twice *full*, its view of *shape* somewhere in the middle)"""
    big = torch.full((2 * full.numel() + 4096,), MARK, dtype=dtype, device="cuda")
    n = torch.Size(shape).numel()
    return big, big[full.numel() // 2 // 8 * 8:][:n].view(shape)


def _untouched(big, view):
    inside = torch.zeros_like(big, dtype=torch.bool)
    lo = (view.data_ptr() - big.data_ptr()) // big.element_size()
    inside.as_strided(view.shape, view.stride(), lo).fill_(True)
    return bool((big[~inside] == MARK).all())


def _inputs(d):
    q, k, v, do = (seeded_normal((B, H, S, d), s) for s in range(4))
    return (q, k, v, do), [x.cuda() for x in (q, k, v, do)]


SHAPES = [lambda d: (1, H, S, d), lambda d: (B, 1, S, d), lambda d: (B, H, S - 40, d), lambda d: (B, H, S, d - 24),
          lambda d: (H, S, d), lambda d: (B, H, S, d)]


def _fits(small, whole):
    """The part of *whole* that a destination like *small* keeps."""
    shape = (1,) * (whole.dim() - small.dim()) + tuple(small.shape)
    return whole[tuple(slice(0, n) for n in shape)].reshape(small.shape)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("shape", SHAPES)
def test_forward_drops_what_does_not_fit(gpu, d, causal, shape):
    announce(f"split bounds forward D{d} causal={causal} out {shape(d)}")
    host, (q, k, v, _) = _inputs(d)
    ref, ref_lse = attention_ref(*host[:3], scale=d ** -0.5, causal=causal)
    lse_shape = shape(d)[:-1] if len(shape(d)) == 4 else (B * H, S)   # (the latter: batch 0 is what fits)
    big, out = _view(shape(d), ref)
    lbig, lse = _view(lse_shape, ref_lse, torch.float32)
    handle = kernels.handle({(64, False): "mha_d64", (64, True): "mha_d64_causal", (128, False): "mha_d128",
                             (128, True): "mha_d128_causal"}[d, causal])

    def split():   # the split kernel itself, which no route gives such destinations
        args = dict(Q=q, K=k, V=v, N=S, O=out, L=lse)
        api._attention_split_kv(handle.pack(args), args, q.shape, 1, causal, NO_RECORDING)

    for launch in (lambda: api.attention_forward(q, k, v, causal=causal, out=out, lse=lse),) * 2 + (split,):
        big.fill_(MARK), lbig.fill_(MARK)
        launch()
        assert rel_err(out.cpu(), _fits(out, ref)) <= 1e-2
        if lse_shape == (B * H, S):
            # (a tiled launch's grid covers the B * H rows: past the H heads of Q it sees zeros)
            assert float((lse.cpu()[:H] - ref_lse[0]).abs().max()) <= 1e-4
            assert launch is not split or bool((lse[H:] == MARK).all())
        else:
            assert float((lse.cpu() - _fits(lse, ref_lse)).abs().max()) <= 1e-4
        assert _untouched(big, out) and _untouched(lbig, lse)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("shape", SHAPES)
def test_backward_drops_what_does_not_fit(gpu, d, causal, shape):
    announce(f"split bounds backward D{d} causal={causal} gradients {shape(d)}")
    host, (q, k, v, do) = _inputs(d)
    ref = attention_bwd_ref(*host, causal=causal)
    o, lse = api.attention_forward(q, k, v, causal=causal)
    bigs, grads = zip(*(_view(shape(d), x) for x in ref))
    dvec, lse2 = torch.empty_like(lse), torch.empty_like(lse)
    sfx = f"d{d}" + "_causal" * causal
    launches = [(kernels.handle(f"mha_bwd_dq_prep_{sfx}"),
                 dict(Q=q, K=k, V=v, dO=do, O=o, L=lse, N=S, dQ=grads[0], Dv=dvec, L2=lse2), None),
                (kernels.handle(f"mha_bwd_dkdv_{sfx}"),
                 dict(Q=q, K=k, V=v, dO=do, L2=lse2, Dv=dvec, N=S, dK=grads[1], dV=grads[2]), None)]

    def split():
        api._attention_bwd_split(launches, causal, NO_RECORDING, dvec)

    for launch in (lambda: api.attention_backward(q, k, v, o, lse, do, *grads, causal=causal),) * 2 + (split,):
        for big in bigs:
            big.fill_(MARK)
        launch()
        for big, got, want in zip(bigs, grads, ref):
            assert rel_err(got.cpu().float(), _fits(got, want)) <= 1e-2
            assert _untouched(big, got)


@pytest.mark.parametrize("pad", [8, 4, 1])
@pytest.mark.parametrize("d", [64, 128])
def test_destinations_whose_heads_are_not_16_byte_aligned(gpu, d, pad):
    host, (q, k, v, do) = _inputs(d)
    ref, _ = attention_ref(*host[:3], scale=d ** -0.5)
    step = S * d + pad
    bigs = [torch.full((B * H * step + 64,), MARK, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    out, *grads = (x.as_strided((B, H, S, d), (H * step, step, d, 1)) for x in bigs)
    for _ in range(2):
        o, lse = api.attention_forward(q, k, v, out=out)
        api.attention_backward(q, k, v, o.contiguous(), lse, do, *grads)
        for big, got, want in zip(bigs, (out, *grads), (ref, *attention_bwd_ref(*host))):
            assert rel_err(got.cpu().float(), want) <= 1e-2 and _untouched(big, got)
