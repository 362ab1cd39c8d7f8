"""The clamped (WIR_EDGE) body of the buffer-form GEMM kernels on the CPU:
its run-time conditions against an interpretation of every tile load."""
from __future__ import annotations

import re

import pytest

from test_lowering import _tile_loads
from warpir_amd import api, kernels
from warpir_amd.lowering import CDNA4Lowerer, CDNA4Target

VARIANTS = ["gemm_256_k64", "gemm_128_k64", "gemm_128_k64_s3", "gemm_128x64_k64", "gemm_64x128_k64",
            "gemm_64_k64", "gemm_128x32_k64", "gemm_256x128", "gemm_128x256_k64", "gemm_128_splitk_k64_b7"]


# a ring of five slots: its loop is one copy with run-time slots
FIVE_SLOTS = "five slots"


def _kernel(name):
    if name != FIVE_SLOTS:
        return kernels.kernel(name)
    return kernels._gemm_mi355x(64, block_m=64, block_n=64, wave_m=32, wave_n=32, lds_budget=80 * 1024)


def _source(name):
    low = CDNA4Lowerer(CDNA4Target(clamp_edges=True)) if name == FIVE_SLOTS else kernels.lowerer(name)
    src = low.lower(_kernel(name))
    return src[src.rindex('extern "C" __global__'):]


def _conditions(body):
    line = next(ln for ln in body.split("\n") if "else if (" in ln and "clamped" in ln)
    cond = line[line.index("(") + 1:line.rindex(")  //")]
    return [c for c in cond.split(" && ") if "Loader<" not in c]


def _eval(expr, ext, pid, n):
    for k, v in zip(("pid_x", "pid_y", "pid_z"), pid):
        expr = expr.replace(k, str(v))
    for g, dims in ext.items():
        for k, v in zip("bdrc", dims):
            expr = expr.replace(f"globals.{g}.{k}", str(v))
    return eval(expr.replace("globals.N", str(n)).replace("/", "//"))   # noqa: S307 - integers only


@pytest.mark.parametrize("name", [*VARIANTS, FIVE_SLOTS])
def test_clamped_body_loads_only_inside_its_tensors(name):
    """Wherever a program's conditions hold, each of its unchecked tile loads
    has its origin inside the tensor in the dimensions that a program id
    indexes (lanes clamp to the last row or chunk there) and lies whole
    inside in the others; the loop's checked copy takes the tiles from
    ``wir_full`` on.  Some swept launches do leave a tensor, and are refused."""
    kernel, body = _kernel(name), _source(name)
    conds = _conditions(body)
    loop = next(o for o in kernel.body if type(o).__name__ == "ForOp")
    tk, c = loop.tile_size, kernel.outputs[0].type.sub_tile_type
    full = re.search(r"const int wir_full_i = WIR_EDGE \? (.*) : ", body)
    clamped = {"A": 2, "B": 3}   # position of the dimension a program id indexes
    refused = 0
    for n in (0, 8, tk, tk + 8, 5 * tk, 6 * tk + 8, 7 * tk):
        for ka in (n, n - 8, n + tk):
            for m, nn in ((1, 8), (c.rows, c.cols), (c.rows + 1, c.cols + 8)):
                ext = {"A": (1, 2, m, max(ka, 0)), "B": (1, 2, n, nn)}
                for pid in ((0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 2)):
                    tiles = -(-n // tk)
                    whole = tiles
                    if full:
                        text = full.group(1)
                        whole = _eval(text, ext, pid, n)
                    inside = True
                    for src, coords, unit in _tile_loads(kernel, tiles, [p + 1 for p in pid]):
                        kpos = 5 - clamped[src]
                        if full and loop.start <= coords[kpos] and coords[kpos] >= whole:
                            continue   # the checked copy
                        for pos, (x, u, e) in enumerate(zip(coords, unit, ext[src])):
                            inside &= 0 <= x * u < e if pos == clamped[src] else 0 <= x and (x + 1) * u <= e
                    holds = all(_eval(x, ext, pid, n) for x in conds)
                    assert inside or not holds, (n, ka, m, nn, pid)
                    refused += not inside
    assert refused


def test_clamped_body_is_emitted_for_plain_gemms_only():
    """Attention kernels, warp-specialised and 8-wave ping-pong GEMMs and the
    reference's SSA form keep their two bodies, also when asked."""
    for name in VARIANTS:
        assert "wir_body(wir::bool_tag<true, true>{});" in _source(name)
    for name in ("mha_d128", "mha_d64_causal", "mha_bwd_dq_d128", "gemm_256x128_ws", "gemm_256_pp", "gemm_ref_ssa"):
        target = CDNA4Target(**{**kernels.TARGETS.get(name, {}), "clamp_edges": True})
        assert "wir_body(wir::bool_tag<true, true>" not in CDNA4Lowerer(target).lower(kernels.kernel(name))


@pytest.mark.parametrize("name", VARIANTS)
def test_clamped_body_needs_results_that_end_with_the_operands(name):
    """A destination that goes on past A's rows or B's columns has zeros there,
    which clamped lanes do not give."""
    line = next(ln for ln in _source(name).split("\n") if "else if (" in ln and "clamped" in ln)
    assert "::clampable<1>(globals.A, globals.C_global.r)" in line
    assert "::clampable<2>(globals.B, globals.C_global.c)" in line


def test_only_a_loop_without_shifted_rings_has_a_checked_copy():
    """A ring that runs behind the loop loads its last tiles in drain steps,
    which have no checked copy: its reduction extent must be whole tiles."""
    assert "WIR_EDGE && v_i < " in _source("gemm_128_k64")
    assert "WIR_EDGE && v_i < " in _source(FIVE_SLOTS) and "wir_base_i" not in _source(FIVE_SLOTS)
    assert "WIR_EDGE && v_i < " not in _source("gemm_128_splitk_k64_b7")


@pytest.mark.parametrize("m,n,k,variant", [
    (256, 256, 256, "gemm_64_k64"), (1, 8, 8, "gemm_64_k64"), (0, 8, 8, None), (8, 8, 0, None),
    (512, 4096, 8192, "gemm_64x128_k64"), (2048, 2048, 2048, "gemm_128_k64_s3"),
    (1024, 8192, 8192, None), (4096, 4096, 4096, "gemm_256_k64"), (8192, 8192, 8192, "gemm_256_k64"),
    (3000, 4104, 4040, "gemm_256_k64"), (128, 8192, 8192, "gemm_128_splitk_k64_b7"),
    (16384, 16384, 8, None)])
def test_gemm_route_by_estimated_time(m, n, k, variant):
    """One tile per CU takes the tile that makes it so; the fallback for
    strided operands is always a tiled kernel, and every route is built."""
    got, tiled = api._gemm_route(m, n, k)
    assert variant in (None, got) and {got, tiled} <= set(kernels.VARIANTS)
    assert tiled != api.SPLITK_GEMM_VARIANT
    assert api.gemm_variant(m, n, k) == got
