"""Launch plans of the public calls: what a call with given shapes, strides,
dtypes and device allocates and launches, worked out once in Python and
replayed by the native module (``csrc/wir_plans.cpp``).

A plan follows from the call's signature alone.  It holds no tensor, and no
address but those of loaded kernel functions, which live as long as the
process (``kernels.handle``).
"""
from __future__ import annotations

import ctypes
import importlib.util
import os
import threading

_native = None
_lock = threading.Lock()


def native():
    """The native module, loaded on the first GPU call."""
    global _native
    if _native is None:
        with _lock:
            if _native is None:
                import torch

                from warpir_amd.runtime import PKG_DIR, library

                path = os.path.join(PKG_DIR, "_wir_plans.so")
                if not os.path.exists(path):
                    raise RuntimeError(f"{path} is not built: run __graft_entry__.build()")
                spec = importlib.util.spec_from_file_location("_wir_plans", path)
                mod = importlib.util.module_from_spec(spec)
                spec.loader.exec_module(mod)
                mod.init(ctypes.cast(library().wir_launch, ctypes.c_void_p).value, torch._C._cuda_getCurrentRawStream)
                _native = mod
    return _native


class Recording:
    """The launches of one call, by the tensors they take."""

    def __init__(self, *inputs):
        self.inputs = inputs
        self.allocs = []
        self.launches = []
        self._slots = {id(t): i for i, t in enumerate(inputs)}

    def alloc(self, t):
        """Note that the call allocated *t*."""
        self._slots[id(t)] = len(self.inputs) + len(self.allocs)
        self.allocs.append(t)
        return t

    def slot(self, t) -> int:
        return self._slots[id(t)]   # (inputs and allocations outlive the recording)

    def pack(self, handle, args):
        """*args* packed for a ``KernelHandle``, past its cache: the next call
        with this signature takes the plan."""
        return handle.pack(args)

    def kernel(self, handle, args, addend=None, packing=None) -> None:
        """Launch a ``KernelHandle`` on *args* (packed as *packing*) and note
        it; ``addend`` maps an argument that is a view to (the tensor it
        views, its offset in bytes)."""
        import torch

        if packing is None:
            packing = self.pack(handle, args)
        packed, cfg = packing[:2]
        if not handle.launch(packing):
            raise ValueError("an empty launch has no plan")
        pointers = []
        for name, x in args.items():
            if isinstance(x, torch.Tensor):
                base, off = addend[name] if addend and name in addend else (x, 0)
                pointers.append((getattr(handle.args_type, name).offset, self.slot(base), off))
        self.raw(handle._function, cfg.grid, cfg.block, packed, pointers, cfg.dyn_lds)

    def raw(self, function, grid, block, args, pointers, dyn_lds: int = 0) -> None:
        """Note a launch of a loaded function with a ctypes argument structure."""
        self.launches.append((function.value, tuple(grid), tuple(block), dyn_lds, bytes(args), pointers))


class _NoRecording:
    """In the place of the recording of a call that can have no plan."""

    def alloc(self, t):
        return t

    def pack(self, handle, args):
        return handle.packed(args)

    def kernel(self, handle, args, addend=None, packing=None) -> None:
        if packing is None:
            handle(**args)
        else:
            handle.launch(packing)

    def __bool__(self) -> bool:
        return False


NO_RECORDING = _NoRecording()


class Plans:
    """The plans of one public call."""

    def __init__(self, what: str):
        self.what = what
        self._table = None

    def run(self, flags: int, *tensors):
        """The call's results by its plan; False where it has none and can
        leave one, None where it can not."""
        table = self._table
        if table is None:
            if _native is None and not getattr(tensors[0], "is_cuda", False):
                return None
            mod = native()
            with _lock:
                if self._table is None:
                    self._table = mod.table()
                table = self._table
        r = _native.run(table, flags, *tensors)
        if type(r) is int:
            from warpir_amd.runtime import check

            check(r, self.what)
        return r

    @staticmethod
    def recording(missed, *inputs):
        """A recording for a call whose ``run`` gave *missed*: ``NO_RECORDING``
        for None, so that nothing is packed for a plan in vain.  us, without
        plans / recording in vain / now: gemm under
        ``torch.set_default_device`` 28 / 68 / 28, the tiled backward 123 / 289
        / 109."""
        return Recording(*inputs) if missed is False else NO_RECORDING

    def add(self, flags: int, rec: Recording, *results) -> None:
        """Keep the plan of a call that has just run."""
        _native.add(self._table, flags, rec.inputs, rec.allocs, rec.launches, [rec.slot(t) for t in results])


__all__ = ["Plans", "Recording", "NO_RECORDING", "native"]
