"""Tensors without memory (fake tensors, as tracing makes them) are refused
before any launch: a kernel would follow their null pointers.  The checks are
host code, so this runs on the CPU with fake GPU tensors."""
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from warpir_amd import api, kernels

pytestmark = pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor")


@pytest.fixture(autouse=True)
def never_launched(monkeypatch):
    """Whatever gets past the checks stops before the native library."""
    from warpir_amd import runtime

    def library():
        raise AssertionError("a launch was reached")

    def current_stream(device=None):
        raise AssertionError("a launch was reached")

    monkeypatch.setattr(runtime, "library", library)
    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(runtime.KernelHandle, "load", lambda self: library())
    for name in ("_gemm_plans", "_forward_plans", "_backward_plans"):   # no plan module either
        monkeypatch.setattr(api, name, _NoPlans())


class _NoPlans(api.Plans):
    def __init__(self):
        super().__init__("none")

    def run(self, flags, *tensors):
        return None


def _fake(*shape, dtype=torch.bfloat16):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        with FakeTensorMode():
            return torch.empty(*shape, dtype=dtype, device="cuda")


@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (300, 520, 264)])
def test_gemm(m, n, k):
    with pytest.raises(ValueError, match="no memory"):
        api.gemm(_fake(m, k), _fake(k, n), out=_fake(m, n))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,hkv,seq", [(2, 2, 128), (4, 2, 128), (64, 64, 2048)])
def test_attention(heads, hkv, seq, causal, d):
    q, o, do = (_fake(1, heads, seq, d) for _ in range(3))
    k, v = (_fake(1, hkv, seq, d) for _ in range(2))
    lse = _fake(1, heads, seq, dtype=torch.float32)
    with pytest.raises(ValueError, match="no memory"):
        api.attention_forward(q, k, v, causal=causal, out=o, lse=lse)
    with pytest.raises(ValueError, match="no memory"):
        api.attention_backward(q, k, v, o, lse, do, _fake(1, heads, seq, d), _fake(1, hkv, seq, d), _fake(1, hkv, seq, d),
                               _fake(1, heads, seq, dtype=torch.float32), causal=causal,
                               workspace=_fake(2 * heads * seq * d, dtype=torch.float32))


def test_grouped_reduction_stays_on_the_operands_gpu():
    with pytest.raises(ValueError, match="memory of the operands' GPU"):
        api._group_reduce(_fake(1, 4, 128, 64, dtype=torch.float32), torch.zeros(1, 2, 128, 64, dtype=torch.bfloat16), 2)
    with pytest.raises(ValueError, match="memory of the operands' GPU"):
        api._group_reduce(_fake(1, 4, 128, 64, dtype=torch.float32), _fake(1, 2, 128, 64), 2)


def test_a_kernel_handle():
    with pytest.raises(ValueError, match="no memory"):
        kernels.handle("gemm_64_k64").pack(dict(A=_fake(64, 64), B=_fake(64, 64), N=64, C_global=_fake(64, 64)))


@pytest.mark.parametrize("missing", range(4))
def test_split_k_null_pointers_are_refused_by_the_library(monkeypatch, missing):
    """gemm_split_k leaves them to its C entry (which has returned before it
    looks at the kernels)."""
    monkeypatch.undo()
    from warpir_amd.runtime import library

    lib, ptrs = library(), [16, 16, 16, 16]
    ptrs[missing] = 0
    a, b, out, ws = ptrs
    assert lib.wir_gemm_splitk(16, 16, a, b, out, ws, 8 * 64 * 64, 64, 64, 512, 8, None) != 0
    assert lib.wir_gemm_splitk_fused(16, a, b, out, ws, 8 * 64 * 64, 16, 64, 64, 64, 512, 8, None) != 0
