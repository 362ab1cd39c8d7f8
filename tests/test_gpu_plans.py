"""Launch plans: a planned call gives what the validating Python path gives,
for every form that path accepts, and every call it refuses stays refused."""
import threading

import pytest
import torch

from oracle.torch_ref import attention_ref, gemm_ref, rel_err, seeded_normal
from warpir_amd import api
from warpir_amd.plans import Plans, native

pytestmark = pytest.mark.gpu


@pytest.fixture
def fresh(monkeypatch):
    """Empty plan tables for one test."""
    for name in ("_gemm_plans", "_forward_plans", "_backward_plans"):
        monkeypatch.setattr(api, name, Plans(name))


def _count(plans):
    return 0 if plans._table is None else native().size(plans._table)


@pytest.mark.parametrize("m,n,k", [(8, 8, 8), (100, 264, 136), (64, 1024, 4096), (300, 520, 264)])
def test_gemm_plan_matches_the_first_call(gpu, fresh, m, n, k):
    a, b = seeded_normal((m, k), 0).cuda(), seeded_normal((k, n), 1).cuda()
    first = api.gemm(a, b)
    assert _count(api._gemm_plans) == 1
    a2, b2 = seeded_normal((m, k), 2).cuda(), seeded_normal((k, n), 3).cuda()
    got = api.gemm(a2, b2)
    assert _count(api._gemm_plans) == 1
    assert rel_err(got.cpu(), gemm_ref(a2.cpu(), b2.cpu())) <= 1e-2
    assert torch.equal(api.gemm(a, b), first)
    out = torch.empty_like(first)
    for _ in range(2):   # a call with `out` has a plan of its own
        assert api.gemm(a, b, out=out.fill_(0)) is out and torch.equal(out, first)
    assert _count(api._gemm_plans) == 2
    wide = torch.zeros(m, k + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, :k] = a
    for _ in range(2):   # another row stride, another plan
        assert rel_err(api.gemm(wide[:, :k], b).cpu(), gemm_ref(a.cpu(), b.cpu())) <= 1e-2
    w = torch.nn.Parameter(b)
    assert torch.equal(api.gemm(a, w), first) and not api.gemm(a, w).requires_grad


@pytest.mark.parametrize("kv,causal,packed", [(6, False, False), (6, True, True), (2, True, False)])
@pytest.mark.parametrize("d", [64, 128])
def test_attention_plans_match_the_first_call(gpu, fresh, d, kv, causal, packed):
    def inputs(seed):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        if packed:
            return torch.randn(2, 192, 3, 6, d, generator=gen, device="cuda", dtype=torch.bfloat16).permute(2, 0, 3, 1, 4)
        return [torch.randn(2, h, 192, d, generator=gen, device="cuda", dtype=torch.bfloat16) for h in (6, kv, kv)]

    def step(seed):
        q, k, v = inputs(seed)
        o, lse = api.attention_forward(q, k, v, causal=causal)
        do = torch.randn(2, 6, 192, d, device="cuda", dtype=torch.bfloat16,
                         generator=torch.Generator(device="cuda").manual_seed(seed + 1))
        return o, lse, *api.attention_backward(q, k, v, o, lse, do, causal=causal)

    first = step(0)
    step(5)
    assert (_count(api._forward_plans), _count(api._backward_plans)) == (1, 1)
    assert all(torch.equal(x, y) for x, y in zip(step(0), first))
    assert [x.stride() for x in step(0)] == [x.stride() for x in first]


def test_a_call_with_one_tensor_twice_leaves_no_plan(gpu, fresh):
    """Its launches cannot tell K from V; later calls must not read K for V."""
    q, k, v = (seeded_normal((1, 2, 128, 128), s).cuda() for s in range(3))
    api.attention_forward(q, k, k)
    assert _count(api._forward_plans) == 0
    for _ in range(2):
        o, _ = api.attention_forward(q, k, v)
        ref, _ = attention_ref(q.cpu(), k.cpu(), v.cpu(), scale=128 ** -0.5)
        assert rel_err(o.cpu(), ref) <= 1e-2
    o, _ = api.attention_forward(q, k, k)   # by the plan of the calls before
    ref, _ = attention_ref(q.cpu(), k.cpu(), k.cpu(), scale=128 ** -0.5)
    assert rel_err(o.cpu(), ref) <= 1e-2


def test_refused_calls_stay_refused_beside_a_plan(gpu, fresh):
    a, b = seeded_normal((64, 64), 0).cuda(), seeded_normal((64, 64), 1).cuda()
    api.gemm(a, b)
    flat = torch.zeros(64 * 64 + 8, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError, match="aligned"):
        api.gemm(flat[1:1 + 64 * 64].view(64, 64), b)
    for bad in (a.cpu(), a.float()):
        with pytest.raises((ValueError, TypeError)):
            api.gemm(bad, b)
    with pytest.raises(ValueError, match="chain"):
        api.gemm(a, b[:32])
    assert api.gemm(a[:0], b).shape == (0, 64)
    assert _count(api._gemm_plans) == 1


def test_plan_follows_the_current_stream_and_capture(gpu, fresh):
    a, b = seeded_normal((64, 4096), 0).cuda(), seeded_normal((4096, 1024), 1).cuda()
    ref = api.gemm(a, b)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = api.gemm(a, b)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = api.gemm(a, b)
    for seed in (4, 5, 6):
        a.copy_(seeded_normal((64, 4096), seed))
        graph.replay()
        assert torch.equal(held, api.gemm(a, b))


def test_tables_are_bounded_and_calls_from_threads_agree(gpu, fresh):
    b = seeded_normal((8, 8), 1).cuda()
    for m in range(1, 300):
        api.gemm(torch.zeros(m, 8, dtype=torch.bfloat16, device="cuda"), b)
    assert _count(api._gemm_plans) <= 256
    a, b = seeded_normal((128, 512), 2).cuda(), seeded_normal((512, 256), 3).cuda()
    ref, bad = api.gemm(a, b), []
    torch.cuda.synchronize()

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                if not torch.equal(api.gemm(a, b), ref):
                    bad.append(1)

    threads = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_a_causal_flag_that_is_no_truth_value_stays_refused_beside_a_plan(gpu, fresh):
    q, k, v = (seeded_normal((1, 2, 128, 64), s).cuda() for s in range(3))
    for causal in (False, True):
        for _ in range(2):
            o, _ = api.attention_forward(q, k, v, causal=causal)
        assert torch.equal(api.attention_forward(q, k, v, causal=int(causal))[0], o)
    for causal in (None, 2, "yes"):
        with pytest.raises(ValueError, match="no kernel variant"):
            api.attention_forward(q, k, v, causal=causal)


class _Subclass(torch.Tensor):
    pass


def _plannable(*tensors):
    """What an empty table says of a call with these tensors."""
    r = native().run(native().table(), 0, *tensors)
    assert r is None or r is False
    return r is False


def _in_mode(mode, *tensors):
    with mode:
        return _plannable(*tensors)


def test_calls_that_can_have_no_plan(gpu, fresh):
    """Active torch-function and dispatch modes, functorch and Python wrappers,
    subclasses, conjugate or misaligned or empty tensors, one tensor twice."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    a, b = seeded_normal((64, 64), 0).cuda(), seeded_normal((64, 64), 1).cuda()
    plan = _plannable
    assert plan(a, b, None) and plan(a, torch.nn.Parameter(b)) and plan(a, b.clone().requires_grad_())
    for mode in (Function(), Dispatch(), torch.device("cuda")):
        assert not _in_mode(mode, a, b)
    assert plan(a, b)
    assert not plan(a, a) and not plan(a, b[:0]) and not plan(a, a.cpu()) and not plan(None, None)
    assert not plan(a, a.flatten()[1:-7].view(8, 511)) and not plan(a, a.as_subclass(_Subclass))
    assert not plan(a, torch._neg_view(b.float())) and not plan(a, b.to_sparse())
    seen = []
    torch.func.vmap(lambda x: seen.append(plan(x, b)) or x)(a[None])
    torch.func.grad(lambda x: seen.append(plan(x, b)) or x.sum())(a.float())
    assert seen == [False, False]
    for mode in (Function(), torch.device("cuda")):   # refused by a table that holds the plan, too
        ref = api.gemm(a, b)
        with mode:
            assert torch.equal(api.gemm(a, b), ref)
    assert torch.equal(api.gemm(a, b.as_subclass(_Subclass)), ref)
    assert _count(api._gemm_plans) == 1


def test_calls_without_a_plan_pack_their_arguments_once(gpu, fresh, monkeypatch):
    """What a call without plans costs: validated and packed on its first call,
    from the handles' caches on later ones, and nothing packed for a plan."""
    from warpir_amd.runtime import KernelHandle

    packed, real = [], KernelHandle.pack
    monkeypatch.setattr(KernelHandle, "pack", lambda self, args: packed.append(self) or real(self, args))

    def twice(call, launches):
        for n in (launches, 0):
            packed.clear()
            call()
            assert len(packed) == n

    x = seeded_normal((64, 64), 0).cuda()
    y = torch.empty_like(x)
    a, b = seeded_normal((64, 4096), 1).cuda(), seeded_normal((4096, 256), 2).cuda()
    twice(lambda: api.gemm(x, x, out=y), 1)
    assert api.gemm_variant(64, 256, 4096) == api.SPLITK_GEMM_VARIANT
    for heads in (2, 600):   # the split and the tiled kernels
        q, k, v, do, o, dq, dk, dv = (seeded_normal((1, heads, 128, 64), s).cuda() for s in range(8))
        flat = torch.empty(heads * 128 + 1, device="cuda")
        lse, dvec = flat[1:].view(1, heads, 128), torch.empty(1, heads, 128, device="cuda")   # lse: 4-byte aligned
        twice(lambda: api.attention_forward(q, k, v, out=o, lse=lse), 1)
        # (its log2 LSE is allocated on every call, where the allocator gives the same memory again)
        twice(lambda: api.attention_backward(q, k, v, o, lse, do, dq, dk, dv, dvec), 2)
    out, z = torch.empty(64, 256, dtype=torch.bfloat16, device="cuda"), torch.empty_like(x)
    with torch.device("cuda"):
        twice(lambda: api.gemm(a, b, out=out), 0)
        twice(lambda: api.gemm(x, y, out=z), 1)
    assert all(_count(p) == 0 for p in (api._gemm_plans, api._forward_plans, api._backward_plans))
    packed.clear()
    api.gemm(x, y)   # a call that leaves a plan packs once as well
    assert len(packed) == 1 and _count(api._gemm_plans) == 1


def test_a_full_table_keeps_part_of_more_signatures_than_it_holds(gpu, fresh, monkeypatch):
    b = seeded_normal((8, 8), 1).cuda()
    rows = [seeded_normal((m, 8), m).cuda() for m in range(1, 321)]
    want = [gemm_ref(a.cpu(), b.cpu()) for a in rows]
    missed, real = [], api._gemm_plans.run

    def run(*args):
        got = real(*args)
        missed.extend([1] * (got is False))
        return got

    monkeypatch.setattr(api._gemm_plans, "run", run)
    for _ in range(4):
        missed.clear()
        for a, w in zip(rows, want):
            assert rel_err(api.gemm(a, b).cpu(), w) <= 1e-2
        assert _count(api._gemm_plans) == 256
    # 256 of 320 held: a random replacement finds most of them, dropping the oldest or all would find none
    assert len(missed) < 200
