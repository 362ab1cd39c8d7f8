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

    def alloc(self, t):
        """Note that the call allocated *t*."""
        self.allocs.append(t)
        return t

    def slot(self, t) -> int:
        for i, x in enumerate(self.inputs):
            if x is t:
                return i
        return len(self.inputs) + next(i for i, x in enumerate(self.allocs) if x is t)

    def kernel(self, handle, addend=None, **args) -> None:
        """A launch of a ``KernelHandle``; ``addend`` maps an argument that is
        a view to (the tensor it views, its offset in bytes)."""
        import torch

        packed, cfg, _device, empty = handle.pack(args)
        if empty or not all(cfg.grid):
            raise ValueError("an empty launch has no plan")
        handle.load()
        pointers = []
        for name, x in args.items():
            if isinstance(x, torch.Tensor):
                base, off = (addend or {}).get(name, (x, 0))
                pointers.append((getattr(handle.args_type, name).offset, self.slot(base), off))
        self.raw(handle._function, cfg.grid, cfg.block, packed, pointers, cfg.dyn_lds)

    def raw(self, function, grid, block, args, pointers, dyn_lds: int = 0) -> None:
        """A launch of a loaded function with a ctypes argument structure."""
        self.launches.append((function.value, tuple(grid), tuple(block), dyn_lds, bytes(args), pointers))


class Plans:
    """The plans of one public call."""

    def __init__(self, what: str):
        self.what = what
        self._table = None

    def run(self, flags: int, *tensors):
        """The call's results by its plan, or None where it has none."""
        table = self._table
        if table is None:
            return None
        r = _native.run(table, flags, *tensors)
        if type(r) is int:
            from warpir_amd.runtime import check

            check(r, self.what)
        return r

    def add(self, flags: int, rec: Recording, *results) -> None:
        """Keep the plan of a call that has just run.  A call that passed one
        tensor twice gives none: its launches do not tell which argument a
        pointer came from."""
        given = [id(t) for t in rec.inputs if t is not None]
        if len(set(given)) != len(given):
            return
        if self._table is None:
            mod = native()
            with _lock:
                if self._table is None:
                    self._table = mod.table()
        _native.add(self._table, flags, rec.inputs, rec.allocs, rec.launches, [rec.slot(t) for t in results])


__all__ = ["Plans", "Recording", "native"]
