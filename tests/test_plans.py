"""The native plan module on the CPU: it takes no call there."""
import os

import pytest
import torch

from warpir_amd import plans
from warpir_amd.runtime import PKG_DIR


@pytest.mark.skipif(not os.path.exists(os.path.join(PKG_DIR, "_wir_plans.so")), reason="not built")
def test_cpu_tensors_and_foreign_arguments_have_no_plan():
    mod = plans.native()
    table, t = mod.table(), torch.zeros(8, 8, dtype=torch.bfloat16)
    for args in ((t, t, None), (None, None), ("x", t), (3,), (torch.zeros(0), t)):
        assert mod.run(table, 0, *args) is None
    assert not mod.add(table, 0, (t, t), [], [(1, (1, 1, 1), (1, 1, 1), 0, b"\0" * 8, [(0, 0, 0)])], [0])
    assert mod.size(table) == 0
    with pytest.raises(ValueError):
        mod.run("no table", 0, t)


def test_recording_finds_a_tensor_by_its_argument():
    a, b, out = (torch.zeros(1) for _ in range(3))
    rec = plans.Recording(a, None, b)
    rec.alloc(out)
    assert [rec.slot(x) for x in (a, b, out)] == [0, 2, 3]


@pytest.mark.skipif(not os.path.exists(os.path.join(PKG_DIR, "_wir_plans.so")), reason="not built")
def test_cpu_calls_record_nothing():
    t = torch.zeros(8, 8, dtype=torch.bfloat16)
    for loaded in (False, True):
        if loaded:
            plans.native()
        table = plans.Plans("x")
        rec = table.recording(table.run(0, t, t.clone()), t)
        assert rec is plans.NO_RECORDING and not rec and rec.alloc(t) is t
