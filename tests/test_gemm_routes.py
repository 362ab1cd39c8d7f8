"""api.gemm's choice of a kernel, on the CPU: kernels and split-K replaced by
recorders."""
import pytest
import torch

from warpir_amd import api, kernels


def _bf16(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


@pytest.fixture
def taken(monkeypatch):
    log = []

    class Handle:
        def __init__(self, name):
            self.name = name

        def __call__(self, **kw):
            log.append(self.name)

    monkeypatch.setattr(kernels, "handle", Handle)
    monkeypatch.setattr(api, "gemm_split_k", lambda a, b, out=None, workspace=None: log.append("split-K") or out)
    return log


# (m, n, k) that split-K takes by estimate: long K with M > 128, and with M <= 128 but fewer than four slices
SPLIT = [(200, 1024, 8192), (16, 8192, 6336)]


@pytest.mark.parametrize("m,n,k", SPLIT)
def test_destinations_of_another_shape_keep_the_tiled_kernels(taken, m, n, k):
    assert api.gemm_variant(m, n, k) == api.SPLITK_GEMM_VARIANT
    a, b = _bf16(m, k), _bf16(k, n)
    api.gemm(a, b, out=_bf16(m, n))
    for shape in ((m - 8, n), (m + 8, n), (m, n + 64), (1, m, n)):
        api.gemm(a, b, out=_bf16(*shape))
    assert taken == ["split-K", *[api._gemm_route(m, n, k)[1]] * 4]


def test_short_m_of_long_k_still_refuses_them():
    """Where M <= 128 has four slices every dense call went to split-K, which
    refuses a destination of another shape, and so it does where the estimate
    now prefers a tiled kernel."""
    refused = 0
    for m, n, k in ((64, 8192, 8192), (64, 1024, 512), (8, 256, 1024), (128, 512, 256)):
        assert api.splitk_count(m, n, k) >= 4
        refused += api.gemm_variant(m, n, k) != api.SPLITK_GEMM_VARIANT
        with pytest.raises(ValueError, match="out must be"):
            api.gemm(_bf16(m, k), _bf16(k, n), out=_bf16(m + 8, n))
    assert refused


@pytest.mark.parametrize("m,n,k", SPLIT)
def test_a_workspace_that_split_k_does_not_take_keeps_the_tiled_kernels(taken, m, n, k):
    """A call with a workspace allocates no partials of its own."""
    assert not (m <= 128 and api.splitk_count(m, n, k) >= 4)
    api.gemm(_bf16(m, k), _bf16(k, n), out=_bf16(m, n), workspace=torch.zeros(8))
    assert taken == [api._gemm_route(m, n, k)[1]]


def test_a_workspace_asks_for_split_k(taken):
    assert api.gemm_variant(64, 1024, 512) != api.SPLITK_GEMM_VARIANT
    api.gemm(_bf16(64, 512), _bf16(512, 1024), workspace=torch.zeros(8 * 64 * 1024))
    assert taken == ["split-K"]


@pytest.mark.parametrize("m,n,k", [(128, 16384, 8192), (128, 16384, 16384), (64, 8192, 8192), (200, 1024, 8192)])
def test_operands_that_split_k_does_not_take_get_the_fastest_tile(m, n, k):
    """Strided operands of a product that split-K would take go to the tiled
    variant with the smallest estimate, for short M too."""
    route, fallback = api._gemm_route(m, n, k)
    assert route == api.SPLITK_GEMM_VARIANT
    est = {v: api._tiled_estimate(c, m, n, k) for v, c in api._TILE_COST.items()}
    assert est[fallback] == min(est.values())


@pytest.mark.parametrize("m,n,k,variant", [
    (64, 8192, 104, "gemm_64_k64"), (128, 8192, 512, "gemm_64_k64"), (256, 8192, 512, "gemm_128x64_k64"), (2048, 2048, 2048, "gemm_128_k64_s3"),
    (64, 8192, 8192, "gemm_128_splitk_k64_b7")])
def test_routes_of_products_that_the_call_accepts(taken, m, n, k, variant):
    """The call takes the kernel of ``gemm_variant`` with its own K."""
    want = api.gemm_variant(m, n, k)
    assert variant in (None, want)
    api.gemm(_bf16(m, k), _bf16(k, n))
    assert taken == ["split-K" if want == api.SPLITK_GEMM_VARIANT else want]
