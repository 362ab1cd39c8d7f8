"""Host entry points for the two workloads, over the generated kernels.

These play the role of the reference harness's launch wrappers
(``launch_gemm(A, B, C)``, ``tests/test_modal_gpu.py:24-50``;
``launch_attention(Q, K, V, O)``, ``tests/test_modal_attention.py:25-39``):
validate shapes, allocate nothing but the outputs and fp32 workspaces the
caller did not pass, and launch the WarpIR-generated HIP kernel through the
C ABI on the current stream.  They raise on a CPU tensor or a missing GPU; there is no
fallback implementation.
"""
from __future__ import annotations

import ctypes
import functools
import math
from typing import Optional, Tuple

from warpir_amd import kernels
from warpir_amd.plans import Plans, Recording
from warpir_amd.runtime import GL, RawKernel

# Plans of the calls below, by flags: gemm 0; attention_forward and
# attention_backward the causal bit.  A stream of calls, by the Python path -> by
# its plan: gemm 256^3 10.7 -> 4.8 us (the kernel's 3.8-4.2 and the gap between
# launches); attention_forward B1 H8 S512 D64 16.0 -> 10.1 us on the tiled kernel
# and 5.9 on the split-key one, the kernels' own time.
_gemm_plans = Plans("gemm")
_forward_plans = Plans("attention_forward")
_backward_plans = Plans("attention_backward")

GEMM_VARIANT = "gemm_256_k64"
SKINNY_GEMM_VARIANT = "gemm_64_k64"       # short M and few columns: what the estimate gives there
MID_GEMM_VARIANT = "gemm_128_k64"         # K unknown, fewer 256x256 tiles than CUs: 128x128 tiles

# Time of one product on the 256 CUs of an MI355X, in microseconds, as a
# function of its tiles T and 64-deep K steps S:
#   fixed + S * step + per_mb * (MB of A and B)
#   step = light + busy * T / 256                                T <= 256
#        = full * (T // 256), plus the same line from light to
#          full for the tiles of a last, partial round           T > 256
# A workgroup's step is slower the more CUs are busy (they share the L2s and
# the power limit), and `full` is the cost of a step where every CU has
# another tile to go to.  The constants are least-squares fits (rms 11-13% in
# log time) to device times of 83 products from 1x312x408 to 14336x12344x1320,
# ragged and aligned; the variant with the smallest estimate was within 0.6%
# (geometric mean; 10% at worst) of the fastest one measured.
#   variant: (tile M, tile N, fixed, light, busy, full, per_mb)
_TILE_COST = {
    GEMM_VARIANT: (256, 256, 11.0, 0.837, 0.508, 1.61, 0.0975),
    "gemm_256x128": (256, 128, 6.62, 0.466, 0.350, 0.950, 0.00306),
    "gemm_128x256_k64": (128, 256, 7.76, 0.444, 0.168, 0.847, 0.110),
    "gemm_128_k64_s3": (128, 128, 4.71, 0.293, 0.119, 0.542, 0.0761),
    "gemm_128x64_k64": (128, 64, 3.41, 0.223, 0.0793, 0.330, 0.0701),
    "gemm_64x128_k64": (64, 128, 3.68, 0.219, 0.0474, 0.307, 0.103),
    "gemm_64_k64": (64, 64, 3.26, 0.143, 0.0543, 0.205, 0.0739),
}
# split-K (128x128 tiles, `splits` slices) with its reduction:
#   fixed + S / splits * (light + busy * T * splits / 256) + per_mb * (MB of partials) + per_mb_ab * (MB of A and B)
_SPLITK_COST = (6.14, 0.459, 0.0407, 0.559, 0.0422)


def _tiled_estimate(cost, m: int, n: int, k: int) -> float:
    bm, bn, fixed, light, busy, full, per_mb = cost
    rounds, rest = divmod(-(-m // bm) * -(-n // bn), 256)
    if rounds == 0 or (rounds == 1 and rest == 0):
        step = light + busy * (rounds + rest / 256)
    else:
        step = full * rounds + (light + (full - light) * rest / 256 if rest else 0.0)
    return fixed + -(-k // 64) * step + per_mb * 2e-6 * k * (m + n)


def _splitk_estimate(m: int, n: int, k: int, splits: int) -> float:
    fixed, light, busy, per_mb, per_mb_ab = _SPLITK_COST
    programs = -(-m // 128) * -(-n // 128) * splits
    return (fixed + k / (64 * splits) * (light + busy * programs / 256) + per_mb * 4e-6 * splits * m * n
            + per_mb_ab * 2e-6 * k * (m + n))


def gemm_variant(m: int, n: int, k: Optional[int] = None) -> str:
    """Kernel variant for an M x N (x K) GEMM on the 256 CUs of one MI355X:
    the tiled variant, or split-K, with the smallest estimated time
    (``_TILE_COST``).  Measured against the rule it replaced (128x128 tiles
    below 256 tiles of 256x256, 128x64 for M <= 256), microseconds:
    512x4096x8192 43.0 vs 72.6, 1024x8192x8192 113.7 vs 146.1,
    2048x2048x8192 61.9 vs 79.0, 200x4096x4096 14.9 vs 20.4,
    3000x4104x4040 102 vs 129.  Without K (or with one that is no multiple of
    8, which no tile load takes) the choice goes by the tile counts alone."""
    if k is None or k % 8:
        if m <= 128:
            return "gemm_128x32_k64"
        if m <= 256:
            return "gemm_128x64_k64"
        if math.ceil(m / 256) * math.ceil(n / 256) < 256:
            return MID_GEMM_VARIANT
        return GEMM_VARIANT
    return _gemm_route(m, n, k)[0]


@functools.lru_cache(maxsize=1024)
def _gemm_route(m: int, n: int, k: int) -> Tuple[str, str]:
    """(variant, variant for operands that split-K does not take: the tile with
    the smallest estimate.  Row-strided A, us: 128x16384x8192 gemm_128x64_k64
    74.8 against gemm_64_k64's 95.3, 128x8192x8192 the other way, 67.4 and
    48.7)."""
    tiled, est = min(((v, _tiled_estimate(c, m, n, k)) for v, c in _TILE_COST.items()), key=lambda x: x[1])
    splits = splitk_count(m, n, k)
    if splits > 1 and _splitk_estimate(m, n, k, splits) < est:
        return SPLITK_GEMM_VARIANT, tiled
    return tiled, tiled


@functools.lru_cache(maxsize=1024)
def _always_split(m: int, n: int, k: int) -> bool:
    """Short M of long K: what goes to split-K without an estimate."""
    return m <= 128 and splitk_count(m, n, k) >= 4


# 128x128 tiles, 64-deep K steps; kernel_pass sizes the rings per operand:
# B (streamed from HBM) seven slots loaded six steps ahead, A (the row panel
# every program re-reads from L2) three slots, filling 160 KiB of LDS
# (measured at M=128, N=K=8192: 36.6 us against 37.8 for 128-deep steps with
# three B slots, and 41.5 for 32-deep steps with fourteen).  The slices are
# summed by the separate reduction kernel (two launches in one C call), also
# the form of wir_gemm_splitk_noalloc.
SPLITK_TWO_LAUNCH_VARIANT = "gemm_128_splitk_k64_b7"
SPLITK_GEMM_VARIANT = SPLITK_TWO_LAUNCH_VARIANT
# The same GEMM summing the slices itself (one launch: the last slice to store
# an output tile adds the partials).  Correct, but slower on MI355X: its
# device-scope release and acquire write back and invalidate an XCD's whole
# L2 per workgroup (58 against 38 microseconds at M=128, N=K=8192).
SPLITK_FUSED_VARIANT = "gemm_128_splitk_fused"
_reduce_kernel = None
# Zeroed per-tile arrival counters of the fused split-K kernels, one buffer
# per (device, stream): the kernel leaves them zero, so launches ordered on
# one stream share a buffer and launches on different streams never do.
_arrivals: dict = {}
_arrivals_lock = __import__("threading").Lock()


def _arrival_counters(device, stream: int, count: int):
    import torch

    key = (device.index, stream)
    with _arrivals_lock:
        buf = _arrivals.get(key)
        if buf is None or buf.numel() < count:
            buf = torch.zeros(max(count, 256), dtype=torch.int32, device=device)
            _arrivals[key] = buf
        return buf


_fused_variants: dict = {}


def _fused(variant: str) -> bool:
    """Whether the split-K variant sums its slices itself (a reduce_slices op)."""
    from warpir_amd.ir import ReduceSlicesOp
    if variant not in _fused_variants:
        _fused_variants[variant] = any(isinstance(op, ReduceSlicesOp) for op in kernels.handle(variant).kernel.body)
    return _fused_variants[variant]


def splitk_count(m: int, n: int, k: int, num_cus: int = 256) -> int:
    """Number of K slices for the split-K kernel: enough 128x128 tiles x
    slices to cover the CUs, with every slice a whole number of 64-deep
    K steps.  1 means no split (also for an empty product)."""
    if m <= 0 or n <= 0 or k <= 0:
        return 1
    tiles = math.ceil(m / 128) * math.ceil(n / 128)
    best = 1
    for s in range(2, 17):
        if tiles * s > num_cus:
            break
        if k % (64 * s) == 0:
            best = s
    return best


_splitk_checked: set = set()


def _splitk_functions(variant: str):
    """(GEMM, reduction) kernel functions of a split-K variant, loaded.  The
    first use of a variant checks that its launch geometry is the one the C
    ABI's split-K entry points build (128x128 tiles, 256 threads, slices on
    blockIdx.z)."""
    global _reduce_kernel
    h = kernels.handle(variant)
    if variant not in _splitk_checked:
        cfg = h.lowerer.launch_config(h.kernel, {"A": (1, 2, 256, 512), "B": (1, 2, 512, 384),
                                                 "C_global": (1, 2, 256, 384)})
        if cfg.grid != (3, 2, 2) or tuple(cfg.block) != (256, 1, 1):
            raise ValueError(f"{variant}: launch geometry {cfg} is not the split-K entry points' "
                             "(128x128 tiles, 256 threads)")
        _splitk_checked.add(variant)
    h.load()
    if _fused(variant):
        return h._function, None
    if _reduce_kernel is None:
        _reduce_kernel = RawKernel("splitk_reduce.hsaco", "wir_splitk_reduce")
    _reduce_kernel._load()
    return h._function, _reduce_kernel._function


def gemm_split_k(a, b, out=None, splits: Optional[int] = None, workspace=None, variant: Optional[str] = None):
    """``out = a @ b`` as ``splits`` K slices run side by side (``blockIdx.z``)
    plus an fp32 reduction: the form for short M and long K, where the
    output alone has too few tiles to fill the chip.  The default variant
    sums the slices with the separate reduction kernel; the fused variant
    (``SPLITK_FUSED_VARIANT``) sums them inside the GEMM kernel (one launch,
    per-tile arrival counters kept per device and stream).  ``workspace`` is an
    fp32 tensor of at least ``splits * M * N`` elements (allocated if
    omitted); ``variant`` names a split-K kernel variant (default
    ``SPLITK_GEMM_VARIANT``)."""
    import torch

    from warpir_amd.runtime import check, library

    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[0]:
        raise ValueError(f"gemm: shapes {tuple(a.shape)} @ {tuple(b.shape)} do not chain")
    m, k = a.shape
    n = b.shape[1]
    if k == 0:
        raise ValueError("gemm_split_k: K must be positive (api.gemm takes K = 0)")
    splits = splits or splitk_count(m, n, k)
    if k % (64 * splits) or n % 8 or not a.is_contiguous() or not b.is_contiguous():
        raise ValueError(f"gemm_split_k: K={k} must split into {splits} multiples of 64, N % 8 == 0, "
                         "contiguous operands")
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise TypeError("gemm_split_k: a and b must be bf16")
    if out is None:
        out = torch.empty(m, n, dtype=torch.bfloat16, device=a.device)
    # the reduction writes M * N bf16 values flat from out's first element (the library refuses null pointers)
    if tuple(out.shape) != (m, n) or out.dtype != torch.bfloat16 or not out.is_contiguous():
        raise ValueError(f"gemm_split_k: out must be a contiguous bf16 [{m}, {n}] tensor, got "
                         f"{out.dtype} {tuple(out.shape)} with strides {tuple(out.stride())}")
    if out.device != a.device:
        raise ValueError("gemm_split_k: out must be on the operands' device")
    if workspace is None:
        workspace = torch.empty(splits * m * n, dtype=torch.float32, device=a.device)
    if workspace.numel() < splits * m * n or workspace.dtype != torch.float32:
        raise ValueError("gemm_split_k: workspace must be fp32 with splits * M * N elements")
    if workspace.device != a.device or not workspace.is_contiguous():
        raise ValueError("gemm_split_k: workspace must be a contiguous tensor on the operands' device")
    if not a.is_cuda or b.device != a.device:
        raise ValueError("gemm_split_k: a, b, out and workspace must be on one GPU")
    if any(t.data_ptr() % 16 for t in (a, b, out, workspace)):
        raise ValueError("gemm_split_k: a, b, out and workspace must be 16-byte aligned")
    if m == 0 or n == 0:
        return out
    gemm_fn, reduce_fn = _splitk_functions(variant or SPLITK_GEMM_VARIANT)
    stream = torch.cuda.current_stream(a.device).cuda_stream
    if reduce_fn is None:   # the slices are summed inside the GEMM kernel
        tiles = math.ceil(m / 128) * math.ceil(n / 128)
        arr = _arrival_counters(a.device, stream, tiles)
        check(library().wir_gemm_splitk_fused(gemm_fn, a.data_ptr(), b.data_ptr(), out.data_ptr(),
                                              workspace.data_ptr(), workspace.numel(), arr.data_ptr(),
                                              arr.numel(), m, n, k, splits, ctypes.c_void_p(stream)),
              "wir_gemm_splitk_fused")
        return out
    check(library().wir_gemm_splitk(gemm_fn, reduce_fn, a.data_ptr(), b.data_ptr(), out.data_ptr(),
                                    workspace.data_ptr(), workspace.numel(), m, n, k, splits,
                                    ctypes.c_void_p(stream)), "wir_gemm_splitk")
    return out


NOALLOC_SCRATCH_FLOATS = 8 * 1024 * 1024   # WIR_NOALLOC_SCRATCH_FLOATS of include/warpir_rt.h


def gemm_split_k_noalloc(a, b, out, splits: Optional[int] = None, stream=None):
    """``out = a @ b`` by the split-K GEMM and the separate reduction kernel
    (``SPLITK_TWO_LAUNCH_VARIANT``; the same sums, bit for bit, as
    ``gemm_split_k``), with the fp32 partials in the native library's own
    device scratch: no device
    memory is allocated (``wir_gemm_splitk_noalloc``).  ``out`` is required.
    Raises ``HipError`` when ``splits * M * N`` exceeds the scratch
    (``NOALLOC_SCRATCH_FLOATS``).  Calls that overlap on one device share the
    scratch and race; order them on one stream."""
    import torch

    from warpir_amd.runtime import check, library

    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[0]:
        raise ValueError(f"gemm: shapes {tuple(a.shape)} @ {tuple(b.shape)} do not chain")
    m, k = a.shape
    n = b.shape[1]
    if k == 0:
        raise ValueError("gemm_split_k_noalloc: K must be positive (api.gemm takes K = 0)")
    splits = splits or splitk_count(m, n, k)
    for name, t, shape in (("a", a, (m, k)), ("b", b, (k, n)), ("out", out, (m, n))):
        if (not isinstance(t, torch.Tensor) or tuple(t.shape) != shape or t.dtype != torch.bfloat16
                or not t.is_contiguous()):
            raise ValueError(f"gemm_split_k_noalloc: {name} must be a contiguous bf16 {list(shape)} tensor")
    if not a.is_cuda or b.device != a.device or out.device != a.device:
        raise ValueError("gemm_split_k_noalloc: a, b and out must be on one GPU")
    if m == 0 or n == 0:
        return out
    gemm_fn, reduce_fn = _splitk_functions(SPLITK_TWO_LAUNCH_VARIANT)
    if stream is None:
        stream = torch.cuda.current_stream(a.device).cuda_stream
    elif hasattr(stream, "cuda_stream"):
        stream = stream.cuda_stream
    with torch.cuda.device(a.device):
        check(library().wir_gemm_splitk_noalloc(gemm_fn, reduce_fn, a.data_ptr(),
                                                b.data_ptr(), out.data_ptr(), m, n, k, splits,
                                                ctypes.c_void_p(stream)),
              "wir_gemm_splitk_noalloc")
    return out


def _splitk_operands_ok(a, b, out) -> bool:
    """Whether ``gemm_split_k`` accepts these tensors: bf16, contiguous and
    16-byte aligned (it addresses them as dense row-major arrays)."""
    import torch

    return all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.data_ptr() % 16 == 0
               for t in (a, b, out))


def gemm(a, b, out=None, variant: Optional[str] = None, workspace=None):
    """``out[M, N] = a[M, K] @ b[K, N]`` in bf16 with fp32 accumulation.

    The variant follows ``gemm_variant``: 256x256 tiles for outputs that fill
    the chip with them, smaller tiles for others, split-K for few tiles and
    long K.  ``workspace`` (as in ``gemm_split_k``) asks for split-K where
    M <= 128 has at least four slices and is not read elsewhere; a call that
    passes it and ``out`` allocates nothing.  An empty output (M or N = 0)
    launches nothing; K = 0 gives zeros (the kernel's loop runs no step and
    its tile loads read the zero page).
    """
    import torch

    done = None
    if variant is None and workspace is None:
        done = _gemm_plans.run(0, a, b, out)
        if done is not None and done is not False:
            return done
    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[0]:
        raise ValueError(f"gemm: shapes {tuple(a.shape)} @ {tuple(b.shape)} do not chain")
    m, k = a.shape
    n = b.shape[1]
    if k % 8 or n % 8:
        raise ValueError("gemm: K and N must be multiples of 8 (16-byte rows)")
    rec = _gemm_plans.recording(done, a, b, out)
    given = out is not None
    if not given:
        out = rec.alloc(torch.empty(m, n, dtype=torch.bfloat16, device=a.device))
    if variant is None:
        variant, tiled = _gemm_route(m, n, k)
        if workspace is not None:
            # the caller's choice of split-K there; elsewhere it is not read, and no partials are
            # allocated beside it
            variant = SPLITK_GEMM_VARIANT if _always_split(m, n, k) else tiled
        if given and tuple(out.shape) != (m, n):
            # split-K, which short M of long K always took, refuses it; the tiled kernels
            # drop what does not fit and write zeros past the product
            variant = SPLITK_GEMM_VARIANT if _always_split(m, n, k) else tiled
        if variant == SPLITK_GEMM_VARIANT and not _splitk_operands_ok(a, b, out):
            # the split-K entry points take dense operands only; the tiled
            # kernel reads row-strided views through the globals' row stride
            variant = tiled
    if variant == SPLITK_GEMM_VARIANT:
        if rec:
            splits = splitk_count(m, n, k)
            workspace = rec.alloc(torch.empty(splits * m * n, dtype=torch.float32, device=a.device))
        gemm_split_k(a, b, out=out, workspace=workspace)
        if rec:
            _record_split_k(rec, a, b, out, workspace, splits)
            _gemm_plans.add(0, rec, out)
        return out
    rec.kernel(kernels.handle(variant), dict(A=a, B=b, N=k, C_global=out))
    if rec:
        _gemm_plans.add(0, rec, out)
    return out


class _ReduceArgs(ctypes.Structure):   # wir_splitk_reduce
    _fields_ = [("partials", ctypes.c_void_p), ("out", ctypes.c_void_p), ("n", ctypes.c_longlong),
                ("split_stride", ctypes.c_longlong), ("splits", ctypes.c_int)]


def _record_split_k(rec: Recording, a, b, out, ws, splits: int) -> None:
    """The two launches of ``wir_gemm_splitk``: the slices of A and B along
    the depth of their globals, then the reduction."""
    (m, k), n = a.shape, b.shape[1]
    kc = k // splits
    args_type = kernels.handle(SPLITK_GEMM_VARIANT).args_type
    args = args_type(A=GL(0, 1, splits, m, kc, 0, kc, k), B=GL(0, 1, splits, kc, n, 0, kc * n, n), N=kc,
                     C_global=GL(0, 1, splits, m, n, 0, m * n, n))
    gemm_fn, reduce_fn = _splitk_functions(SPLITK_GEMM_VARIANT)
    rec.raw(gemm_fn, (math.ceil(n / 128), math.ceil(m / 128), splits), (256, 1, 1), args,
            [(getattr(args_type, f).offset, rec.slot(t), 0) for f, t in (("A", a), ("B", b), ("C_global", ws))])
    rec.raw(reduce_fn, ((m * n // 8 + 255) // 256, 1, 1), (256, 1, 1), _ReduceArgs(0, 0, m * n, m * n, splits),
            [(_ReduceArgs.partials.offset, rec.slot(ws), 0), (_ReduceArgs.out.offset, rec.slot(out), 0)])


def attention_forward(q, k, v, causal: bool = False, out=None, lse=None,
                      variant: Optional[str] = None) -> Tuple[object, object]:
    """FlashAttention forward over ``[B, H, S, D]`` bf16; returns ``(O, LSE)``.

    ``LSE[b, h, s] = logsumexp_j(q_s . k_j / sqrt(D))`` in fp32 (natural log).
    """
    import torch

    planned = variant is None and type(causal) in (bool, int) and 0 <= causal <= 1   # others are refused below
    done = None
    if planned:
        done = _forward_plans.run(1 if causal else 0, q, k, v, out, lse)
        if done is not None and done is not False:
            return done
    bsz, heads, seq, d = q.shape
    hr = _head_ratio("attention_forward", q, k, v)
    if variant is None:
        variant = {(128, False): "mha_d128", (64, True): "mha_d64_causal",
                   (128, True): "mha_d128_causal", (64, False): "mha_d64"}.get((d, causal))
        if variant is None:
            raise ValueError(f"attention_forward: no kernel variant for D={d}, causal={causal}")
        if hr > 1:
            variant += "_gqa"
        elif variant == "mha_d128" and -(-seq // 128) * heads * bsz <= 256:
            # 256-row blocks leave CUs idle: 128-row blocks of the same softmax, while there is
            # at most one per CU (B1 H16 S2048 49.9 -> 43.4 us, B1 H8 S512 16.7 -> 13.6 us;
            # 336 blocks, B6 H8 S896: 26.5 -> 27.6 us)
            variant = "mha_d128_w4"
    handle = kernels.handle(variant)
    kv_tile = _kv_tile(variant)
    if seq % kv_tile:
        raise ValueError(f"attention_forward: S={seq} must be a multiple of the KV tile {kv_tile}")
    rec = _forward_plans.recording(done, q, k, v, out, lse)
    # (the tiled kernels' grid covers destinations of other shapes: what does not fit is dropped)
    whole = (out is None or out.shape == q.shape) and (lse is None or lse.shape == (bsz, heads, seq))
    if out is None:
        out = rec.alloc(torch.empty_like(q))
    if lse is None:
        lse = rec.alloc(torch.empty(bsz, heads, seq, dtype=torch.float32, device=q.device))
    args = dict(Q=q, K=k, V=v, N=seq, O=out, L=lse)
    if "HR" in handle.args_type.__dict__:
        args["HR"] = hr
    elif hr > 1:
        raise ValueError(f"attention_forward: variant {variant} takes no grouped-query heads")
    packing = rec.pack(handle, args)
    shape = (bsz, heads, seq, d)
    if planned and whole and _split_kv_fits(shape, causal, packing[0]):
        _attention_split_kv(packing, args, shape, hr, causal, rec)
        return out, lse
    rec.kernel(handle, args, packing=packing)
    if rec:
        _forward_plans.add(1 if causal else 0, rec, out, lse)
    return out, lse


# The split attention kernels hold one program of 32 rows per CU at a time.  Up
# to 256 programs they win at every length; up to 512, which start a second
# round of them, where each has enough tiles to walk.  Shortest such S of causal
# launches by programs (up to 320, 384, 448, 512): a causal launch's short
# blocks fill the second round, so it pays earlier with fewer of them.  us,
# tiled -> split, forward D64 H32 S320 9.0 -> 8.7, H44 S320 9.0 -> 9.9, H32 S512
# 10.7 -> 10.1, H64 S256 7.6 -> 8.7; D128 H32 S320 12.3 -> 10.7, H27 S448 14.3 ->
# 15.0, H24 S512 14.8 -> 13.7, H21 S768 19.5 -> 21.2, H18 S896 21.8 -> 20.6;
# dQ + dK/dV D64 H32 S320 27.7 -> 24.0, H53 S192 22.3 -> 24.5, H37 S384 30.0 ->
# 31.6, H32 S448 33.8 -> 27.9; D128 H32 S320 34.4 -> 31.1, H38 S320 36.1 -> 37.1,
# H32 S384 37.2 -> 35.0, H37 S384 39.1 -> 43.0, H36 S448 42.4 -> 41.3.
_SPLIT_CAUSAL_SEQ = {
    ("forward", 64): (320, 320, 448, 448), ("forward", 128): (320, 512, 576, 896),
    ("backward", 64): (320, 320, 448, 448), ("backward", 128): (320, 384, 448, 448),
}


def _split_wins(part: str, programs: int, seq: int, d: int, causal: bool) -> bool:
    """Whether a launch of *programs* blocks of 32 rows is faster in the split
    kernels (``attn_splitkv.hip``, ``attn_bwd_split.hip``) than in the tiled
    ones.  us, tiled -> split, at 128 programs: forward B1 H8 S512 D64 10.3 -> 6.0,
    dQ + dK/dV 32.2 -> 16.3.  Past 256 programs full launches take two whole
    rounds: the forward never wins (S2048 D64 30.0 -> 26.5 but D128 46.5 ->
    48.5), dQ + dK/dV at D64 from S640, or from S512 where the waves' tiles come
    out even (H16 S512 32.4 -> 30.6, S576 34.7 -> 35.8, S640 37.6 -> 36.1), at D128
    from S1024 (67.5 -> 66.4, S768 55.1 -> 56.3)."""
    if not 0 < programs <= 512:
        return False
    if programs <= 256:
        return True
    if causal:
        return seq >= _SPLIT_CAUSAL_SEQ[part, d][(programs - 257) // 64]
    if part == "forward":
        return False
    return seq >= 1024 if d == 128 else seq >= 640 or seq == 512


def _split_kv_fits(shape, causal: bool, packed) -> bool:
    """Whether the forward on Q of *shape* goes to the split-key kernel; its
    lane offsets are 32-bit."""
    bsz, heads, seq, d = shape
    return (_split_wins("forward", bsz * heads * (seq // 32), seq, d, causal)
            and 0 <= packed.K.sr < 1 << 23 and 0 <= packed.V.sr < 1 << 23)


_split_kv_kernels: dict = {}


class _SplitKvArgs(ctypes.Structure):
    _fields_ = [("Q", GL), ("K", GL), ("V", GL), ("N", ctypes.c_int), ("HR", ctypes.c_int), ("O", GL), ("L", GL)]


_SPLIT_KV_POINTERS = [(f, getattr(_SplitKvArgs, f).offset) for f in "QKVOL"]


def _attention_split_kv(packing, args: dict, shape, hr: int, causal: bool, rec) -> None:
    """Launch the split-key forward on what a tiled kernel's handle made of
    *args* (validated, packed; *shape* is Q's), and keep the call's plan."""
    import torch

    packed, _cfg, device, _empty = packing
    bsz, heads, seq, d = shape
    name = f"wir_attn_splitkv_d{d}" + ("_causal" if causal else "")
    kernel = _split_kv_kernels.get(name)
    if kernel is None:
        kernel = _split_kv_kernels.setdefault(name, RawKernel("attn_splitkv.hsaco", name))
    packed = _SplitKvArgs(packed.Q, packed.K, packed.V, args["N"], hr, packed.O, packed.L)
    grid, block = (seq // 32, heads, bsz), (256, 1, 1)
    kernel.launch(grid, block, packed, stream=torch.cuda.current_stream(device).cuda_stream)
    if rec:
        rec.raw(kernel._function, grid, block, packed,
                [(offset, rec.slot(args[f]), 0) for f, offset in _SPLIT_KV_POINTERS])
        _forward_plans.add(1 if causal else 0, rec, args["O"], args["L"])


def _head_ratio(fn: str, q, k, v) -> int:
    """Query heads per key/value head (grouped-query attention); 1 for plain MHA."""
    if q.dim() != 4 or k.dim() != 4 or k.shape != v.shape or q.shape[0] != k.shape[0] \
            or q.shape[2:] != k.shape[2:]:
        raise ValueError(f"{fn}: q [B, H, S, D] and k, v [B, H_kv, S, D] shapes do not match")
    if k.shape[1] < 1 or q.shape[1] % k.shape[1]:
        raise ValueError(f"{fn}: {q.shape[1]} query heads are not a multiple of {k.shape[1]} key/value heads")
    return q.shape[1] // k.shape[1]


def attention_backward(q, k, v, o, lse, do, dq=None, dk=None, dv=None, dvec=None, causal: bool = False,
                       workspace=None):
    """Gradients ``(dQ, dK, dV)`` of ``attention_forward`` over ``[B, H, S, D]``
    bf16, from its outputs ``o`` and ``lse`` and the output gradient ``do``
    (``causal`` must match the forward); S must be a multiple of 64.  With
    grouped-query K and V (``[B, H_kv, S, D]``) the key-major kernel writes
    each query head's fp32 dK / dV contribution into ``workspace`` (fp32, at
    least ``2 * B * H * S * D`` elements, allocated if omitted) and a HIP
    reduction sums the ``H / H_kv`` contributions of every key/value head
    into bf16 ``dK`` / ``dV``.  Two WarpIR kernels (or, for small launches,
    their hand-written split forms, ``attn_bwd_split.hip``) run
    on the current stream: the query-major dQ kernel, which also writes
    ``Dv = rowsum(dO * O)`` (into ``dvec``, fp32 ``[B, H, S]``, allocated if
    omitted) and the LSE in log2 units, and the key-major dK/dV kernel, which
    reads them (the reference's TK backward,
    ``kernel_examples/attention/mha_h100.cu:253-303,482-642``, computes the
    same gradients with dQ by atomic adds)."""
    import torch

    planned = workspace is None
    done = None
    if planned:
        done = _backward_plans.run(1 if causal else 0, q, k, v, o, lse, do, dq, dk, dv, dvec)
        if done is not None and done is not False:
            return done
    if q.dim() != 4 or not (q.shape == o.shape == do.shape):
        raise ValueError("attention_backward: q, o, do must share one [B, H, S, D] shape")
    hr = _head_ratio("attention_backward", q, k, v)
    bsz, heads, seq, d = q.shape
    if d not in (64, 128) or seq % 64:
        raise ValueError(f"attention_backward: D must be 64 or 128 and S a multiple of 64 (got D={d}, S={seq})")
    if tuple(lse.shape) != (bsz, heads, seq) or lse.dtype != torch.float32:
        raise ValueError("attention_backward: lse must be fp32 [B, H, S]")
    rec = _backward_plans.recording(done, q, k, v, o, lse, do, dq, dk, dv, dvec)
    whole = (all(g is None or g.shape == q.shape for g in (dq, dk, dv))   # as in the forward
             and (dvec is None or dvec.shape == lse.shape))
    dq = rec.alloc(torch.empty_like(q)) if dq is None else dq
    dk = rec.alloc(torch.empty_like(k)) if dk is None else dk
    dv = rec.alloc(torch.empty_like(v)) if dv is None else dv
    dvec = rec.alloc(torch.empty(bsz, heads, seq, dtype=torch.float32, device=q.device)) if dvec is None else dvec
    lse2 = rec.alloc(torch.empty_like(lse))   # the LSE in log2 units, for the dK/dV kernel
    sfx = ("_causal" if causal else "") + ("_gqa" if hr > 1 else "")
    dq_args = dict(Q=q, K=k, V=v, dO=do, O=o, L=lse, N=seq, dQ=dq, Dv=dvec, L2=lse2)
    dkdv_args = dict(Q=q, K=k, V=v, dO=do, L2=lse2, Dv=dvec, N=seq)
    views = None
    if hr == 1:
        dkdv_args.update(dK=dk, dV=dv)
    else:
        numel = q.numel()
        if workspace is None:
            workspace = rec.alloc(torch.empty(2 * numel, dtype=torch.float32, device=q.device))
        if workspace.dtype != torch.float32 or workspace.numel() < 2 * numel or not workspace.is_contiguous():
            raise ValueError(f"attention_backward: workspace must be contiguous fp32 with >= {2 * numel} elements")
        dk_part = workspace[:numel].view(q.shape)
        dv_part = workspace[numel:2 * numel].view(q.shape)
        views = {"dK_part": (workspace, 0), "dV_part": (workspace, 4 * numel)}
        dq_args["HR"] = hr
        dkdv_args.update(HR=hr, dK_part=dk_part, dV_part=dv_part)
    # (handle, arguments, views) of each launch in order
    launches = [(kernels.handle(f"mha_bwd_dq_prep_d{d}{sfx}"), dq_args, None),
                (kernels.handle(f"mha_bwd_dkdv_d{d}{sfx}"), dkdv_args, views)]
    if planned and whole and hr == 1 and _split_bwd_fits((bsz, heads, seq, d), causal, q, k, v, do):
        _attention_bwd_split(launches, causal, rec, dvec)
        if rec:
            _backward_plans.add(1 if causal else 0, rec, dq, dk, dv)
        return dq, dk, dv
    for handle, args, seen in launches:
        rec.kernel(handle, args, seen)
    reductions = []
    if hr > 1:
        reductions = [(_group_reduce(dk_part, dk, hr), 0, dk), (_group_reduce(dv_part, dv, hr), 4 * numel, dv)]
    if rec:
        for (grid, args), off, grad in reductions:
            rec.raw(_group_reduce_kernel._function, grid, (256, 1, 1), args,
                    [(type(args).partials.offset, rec.slot(workspace), off), (type(args).out.offset, rec.slot(grad), 0)])
        _backward_plans.add(1 if causal else 0, rec, dq, dk, dv)
    return dq, dk, dv


def _split_bwd_fits(shape, causal: bool, *loaded) -> bool:
    """Whether the backward goes to the split kernels; their lane offsets are
    32-bit."""
    bsz, heads, seq, d = shape
    return (_split_wins("backward", bsz * heads * (seq // 32), seq, d, causal)
            and all(0 <= t.stride(2) < 1 << 23 for t in loaded))


_split_bwd_kernels: dict = {}


def _attention_bwd_split(launches, causal: bool, rec, dvec) -> None:
    """Launch the split dQ and dK/dV kernels on the arguments of the tiled
    kernels in *launches*, which validate and pack them, and record them."""
    import torch

    stream = torch.cuda.current_stream(dvec.device).cuda_stream
    for part, (handle, args, _) in zip(("dq", "dkdv"), launches):
        bsz, heads, seq, d = args["Q"].shape
        name = f"wir_attn_{part}_split_d{d}" + ("_causal" if causal else "")
        kernel = _split_bwd_kernels.get(name)
        if kernel is None:
            kernel = _split_bwd_kernels.setdefault(name, RawKernel("attn_bwd_split.hsaco", name))
        packed = rec.pack(handle, args)[0]
        grid, block = (seq // 32, heads, bsz), (256, 1, 1)
        kernel.launch(grid, block, packed, stream=stream)
        if rec:
            rec.raw(kernel._function, grid, block, packed,
                    [(getattr(handle.args_type, f).offset, rec.slot(x), 0) for f, x in args.items()
                     if isinstance(x, torch.Tensor)])


_group_reduce_kernel = None


class _GroupReduceArgs(ctypes.Structure):
    _fields_ = [("partials", ctypes.c_void_p), ("out", ctypes.c_void_p), ("n", ctypes.c_longlong),
                ("groups", ctypes.c_longlong), ("splits", ctypes.c_int)]


def _group_reduce(partials, out, splits: int):
    """``out[g] = bf16(sum_r partials[g * splits + r])`` over the key/value head
    groups of a ``[B, H, S, D]`` fp32 contribution tensor (``splitk_reduce.hip``)."""
    global _group_reduce_kernel
    if _group_reduce_kernel is None:
        _group_reduce_kernel = RawKernel("splitk_reduce.hsaco", "wir_group_reduce")
    if not out.is_contiguous() or out.dtype.itemsize != 2:
        raise ValueError("attention_backward: dk / dv must be contiguous bf16")
    if out.numel() == 0:
        return None
    if out.device != partials.device or not out.data_ptr():
        raise ValueError("attention_backward: dk / dv must be in the memory of the operands' GPU")
    n = out.shape[-2] * out.shape[-1]
    groups = out.numel() // n
    if n % 8 or partials.numel() != groups * splits * n:
        raise ValueError("attention_backward: grouped reduction needs S * D % 8 == 0 and matching shapes")
    args = _GroupReduceArgs(partials.data_ptr(), out.data_ptr(), n, groups, splits)
    grid = ((groups * n // 8 + 255) // 256, 1, 1)
    _group_reduce_kernel.launch(grid, (256, 1, 1), args)
    return grid, args


def attention_backward_flops(bsz: int, heads: int, seq: int, d: int, causal: bool = False) -> float:
    """Matmul FLOPs of attention backward counted as the five S x S x D
    products of the standard algorithm (S, dP, dV, dK, dQ): 10*B*H*S^2*D,
    halved when causal.  These kernels run seven (dQ recomputes S and dP
    instead of atomics)."""
    f = 10.0 * bsz * heads * seq * seq * d
    return f / 2 if causal else f


def attention_flops(bsz: int, heads: int, seq: int, d: int, causal: bool = False) -> float:
    """Matmul FLOPs of attention forward: 4*B*H*S^2*D (halved when causal)."""
    f = 4.0 * bsz * heads * seq * seq * d
    return f / 2 if causal else f


@functools.lru_cache(maxsize=None)
def _kv_tile(variant: str) -> int:
    from warpir_amd.ir.ops import ForOp

    return next(op for op in kernels.handle(variant).kernel.body if isinstance(op, ForOp)).tile_size


__all__ = ["gemm", "gemm_split_k", "splitk_count", "gemm_variant", "attention_forward", "attention_backward",
           "attention_flops", "attention_backward_flops"]
