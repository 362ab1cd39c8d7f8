"""GEMM kernels at ragged extents (the clamped body): the operands are views
of larger tensors filled with NaN, and C of one filled with a marker, so a
lane that read or stored past an edge would show."""
from __future__ import annotations

import pytest
import torch

from oracle.torch_ref import gemm_ref, rel_err, seeded_normal
from warpir_amd import api, kernels

pytestmark = pytest.mark.gpu

# fp32 accumulation, one bf16 rounding of C: at most 2^-8 of the largest value (rel_err's scale)
TOL = 2.0 ** -8

EDGE_VARIANTS = ["gemm_256_k64", "gemm_256x128", "gemm_128x256_k64", "gemm_128_k64", "gemm_128_k64_s3",
                 "gemm_128x64_k64", "gemm_64x128_k64", "gemm_64_k64", "gemm_128x32_k64"]


def _inside(t, rows, cols, fill):
    """*t* as the top left corner of a larger tensor (row pitch a multiple of 8)."""
    big = torch.full((t.shape[0] + rows, t.shape[1] + cols), fill, dtype=t.dtype, device="cuda")
    big[:t.shape[0], :t.shape[1]] = t
    return big, big[:t.shape[0], :t.shape[1]]


@pytest.mark.parametrize("variant", EDGE_VARIANTS)
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (255, 248, 128), (257, 264, 136), (256, 256, 56), (256, 256, 72),
                                   (384, 520, 192), (31, 8, 1032), (513, 1032, 264)])
def test_ragged_gemm_reads_and_stores_only_its_tensors(gpu, variant, m, n, k):
    a, b = seeded_normal((m, k), 0), seeded_normal((k, n), 1)
    nan = float("nan")
    _, av = _inside(a.cuda(), 40, 64, nan)
    _, bv = _inside(b.cuda(), 72, 264, nan)
    big, c = _inside(torch.zeros(m, n, dtype=torch.bfloat16, device="cuda"), 264, 264, -7.0)
    kernels.handle(variant)(A=av, B=bv, N=k, C_global=c)
    torch.cuda.synchronize()
    assert rel_err(c.cpu(), gemm_ref(a, b)) <= TOL
    big[:m, :n] = -7.0
    assert bool((big == -7.0).all())


@pytest.mark.parametrize("variant", EDGE_VARIANTS)
def test_ragged_gemm_keeps_infinities_in_their_row_and_column(gpu, variant):
    """Clamped lanes read the last row of A and the last columns of B again,
    and the reduction's cut tile reads zeros: an infinity there must not
    reach any other element of C."""
    m, n, k = 300, 264, 136
    a, b = seeded_normal((m, k), 2), seeded_normal((k, n), 3)
    a[m - 1, 5] = float("inf")
    b[k - 1, n - 1] = float("inf")
    c = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    kernels.handle(variant)(A=a.cuda(), B=b.cuda(), N=k, C_global=c)
    c = c.cpu().float()
    assert not bool(c[m - 1].isfinite().any()) and not bool(c[:, n - 1].isfinite().any())
    assert bool(c[:m - 1, :n - 1].isfinite().all())
    assert rel_err(c[:m - 1, :n - 1], gemm_ref(a[:m - 1], b[:, :n - 1])) <= TOL


@pytest.mark.parametrize("variant", EDGE_VARIANTS)
@pytest.mark.parametrize("rows,cols", [(28, 0), (0, 24), (300, 264), (-5, 0), (0, -8)])
def test_destination_of_another_shape_has_zeros_past_the_product(gpu, variant, rows, cols):
    """Clamped lanes feed only results past the end of A or B: where C goes on
    there, its elements are zero, and a smaller C drops what does not fit."""
    m, n, k = 100, 136, 264
    a, b = seeded_normal((m, k), 6), seeded_normal((k, n), 7)
    c = torch.full((m + rows, n + cols), -7.0, dtype=torch.bfloat16, device="cuda")
    kernels.handle(variant)(A=a.cuda(), B=b.cuda(), N=k, C_global=c)
    want = torch.zeros(m + max(rows, 0), n + max(cols, 0))
    want[:m, :n] = gemm_ref(a, b)
    want = want[:m + rows, :n + cols]
    assert rel_err(c.cpu(), want) <= TOL
    assert bool((c.cpu()[m:] == 0).all()) and bool((c.cpu()[:, n:] == 0).all())


@pytest.mark.parametrize("variant", ["gemm_64_k64", "gemm_64x128_k64"])
@pytest.mark.parametrize("m,n,k", [(64, 128, 64), (128, 128, 256), (192, 256, 320), (1024, 1024, 1024)])
def test_small_tiles_match_the_256_tile_bit_for_bit(gpu, variant, m, n, k):
    """Every tiled variant adds the same MFMA products in the same k order."""
    a, b = seeded_normal((m, k), 4).cuda(), seeded_normal((k, n), 5).cuda()
    c, ref = (torch.empty(m, n, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    kernels.handle(variant)(A=a, B=b, N=k, C_global=c)
    kernels.handle("gemm_256_k64")(A=a, B=b, N=k, C_global=ref)
    assert torch.equal(c, ref)


@pytest.mark.parametrize("m,n,k", [(200, 1024, 8192), (333, 264, 4096), (16, 8192, 6336)])
def test_split_k_by_estimate(gpu, monkeypatch, m, n, k):
    """Products that no fixed rule sends to split-K (M > 128, fewer than four
    slices), on the first call and by its plan."""
    assert api.gemm_variant(m, n, k) == api.SPLITK_GEMM_VARIANT
    split, real = [], api.gemm_split_k
    monkeypatch.setattr(api, "gemm_split_k", lambda *a, **kw: split.append(1) or real(*a, **kw))
    monkeypatch.setattr(api, "_gemm_plans", api.Plans("gemm"))
    for seed in (0, 2):
        a, b = seeded_normal((m, k), seed), seeded_normal((k, n), seed + 1)
        big, c = _inside(torch.zeros(m, n, dtype=torch.bfloat16, device="cuda"), 8, 0, -7.0)   # rows after the last
        api.gemm(a.cuda(), b.cuda(), out=c)
        assert rel_err(c.cpu(), gemm_ref(a, b)) <= TOL and bool((big[m:] == -7.0).all())
    assert len(split) == 1
