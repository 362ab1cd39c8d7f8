"""The dQ kernel that also does the backward's preparation (Dv, LSE in log2
units): on the CPU interpreter, as text, and on the GPU against the separate
prep and dQ kernels."""
import math

import pytest
import torch

from oracle.ir_interp import run_kernel
from oracle.torch_ref import attention_bwd_ref, attention_ref, rel_err, seeded_normal
from tests.conftest import announce
from warpir_amd import kernels
from warpir_amd.ir import RowDotOp
from warpir_amd.passes.modulo_scheduler import gfx950_attention_cost_model, kernel_pass
from warpir_amd.printing import print_kernel
from warpir_amd.workloads import build_mha_bwd_dq_kernel


@pytest.mark.parametrize("pipelined", [False, True])
@pytest.mark.parametrize("s,causal,hr", [(256, False, 1), (192, True, 1), (128, True, 2)])
def test_dq_with_prep_matches_autograd(pipelined, s, causal, hr):
    q, do = (seeded_normal((1, 2, s, 64), i) for i in (0, 3))
    k, v = (seeded_normal((1, 2 // hr, s, 64), i) for i in (1, 2))
    ke, ve = (x.repeat_interleave(hr, 1) for x in (k, v))
    o, lse = attention_ref(q, ke, ve, causal=causal)
    o = o.to(torch.bfloat16)
    kernel = build_mha_bwd_dq_kernel(d=64, block_q=128, block_kv=64, wave_rows=32, causal=causal, gqa=hr > 1,
                                     prep=True)
    if pipelined:
        kernel = kernel_pass(kernel, cost_model=gfx950_attention_cost_model(128, 64, 64))
    out = {"dQ": torch.zeros_like(q), "Dv": torch.zeros(1, 2, s), "L2": torch.zeros(1, 2, s)}
    run_kernel(kernel, {"Q": q, "K": k, "V": v, "dO": do, "O": o, "L": lse, **out},
               {"N": s, **({"HR": hr} if hr > 1 else {})})
    assert rel_err(out["dQ"].float(), attention_bwd_ref(q, ke, ve, do, causal=causal)[0]) <= 1e-2
    assert torch.allclose(out["Dv"], (do.float() * o.float()).sum(-1), rtol=1e-5, atol=1e-5)
    assert torch.equal(out["L2"], lse * math.log2(math.e))


def test_row_dot_prints_and_takes_its_tiles_from_registers(capsys):
    kernel = kernels.kernel("mha_bwd_dq_prep_d64")
    assert sum(isinstance(o, RowDotOp) for o in kernel.body) == 1
    print_kernel(kernel)
    assert "row_dot(" in capsys.readouterr().out
    src = kernels.lowerer("mha_bwd_dq_prep_d64").lower(kernel)
    body = src[src.rindex('extern "C"'):]
    assert "wir::row_dot(v_d_vec, hf_do_shared, hf_o_shared);" in body
    low = kernels.lowerer("mha_bwd_dq_prep_d64")
    low.lower(kernel)
    assert low.lds_total == 24576     # O and dO take no LDS beside the K and V rings


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bsz,heads,hkv,s,d", [(1, 1, 1, 64, 64), (2, 3, 3, 192, 128), (1, 4, 2, 320, 64),
                                               (1, 2, 1, 128, 128), (2, 2, 2, 1024, 64)])
def test_dq_prep_kernel_matches_the_separate_kernels(gpu, bsz, heads, hkv, s, d, causal):
    announce(f"dq+prep B{bsz} H{heads}/{hkv} S{s} D{d} causal={causal}")
    q, do = (seeded_normal((bsz, heads, s, d), i).cuda() for i in (0, 3))
    k, v = (seeded_normal((bsz, hkv, s, d), i).cuda() for i in (1, 2))
    o = seeded_normal((bsz, heads, s, d), 4).cuda()
    lse = seeded_normal((bsz, heads, s), 5).float().cuda() + 6.0
    sfx = ("_causal" if causal else "") + ("_gqa" if hkv < heads else "")
    hr = {"HR": heads // hkv} if hkv < heads else {}
    got, ref = ([torch.full_like(q, float("nan"))] + [torch.full_like(lse, float("nan")) for _ in range(2)]
                for _ in range(2))
    kernels.handle(f"mha_bwd_dq_prep_d{d}{sfx}")(Q=q, K=k, V=v, dO=do, O=o, L=lse, N=s, dQ=got[0], Dv=got[1],
                                                 L2=got[2], **hr)
    kernels.handle(f"mha_bwd_prep_d{d}")(O=o, dO=do, L=lse, Dv=ref[1], L2=ref[2])
    kernels.handle(f"mha_bwd_dq_d{d}{sfx}")(Q=q, K=k, V=v, dO=do, L=lse, Dv=ref[1], N=s, dQ=ref[0], **hr)
    assert torch.equal(got[2], ref[2])
    # fp32 sums of d exact products in two orders: d rounding errors of the sum of magnitudes
    bound = d * 2.0 ** -24 * (do.float() * o.float()).abs().sum(-1)
    assert bool(((got[1] - ref[1]).abs() <= bound).all())
    # dQ from Dv values that differ by that much: one bf16 rounding apart
    assert rel_err(got[0].cpu(), ref[0].cpu().float()) <= 2.0 ** -8
