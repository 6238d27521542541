"""Shared plumbing of the drop-in modules."""

from __future__ import annotations

import torch
import torch.nn as nn


_CHECK_MODE = False


class check_mode:
    """Context manager / switch for the fp32 check mode: inside it every module's
    `forward` runs the plain fp32 kernels of `check.py` (fp32 tensors in and out,
    results returned as new tensors) instead of the bf16 MFMA path."""

    def __init__(self, enabled: bool = True):
        self.enabled = enabled

    def __enter__(self):
        global _CHECK_MODE
        self._old, _CHECK_MODE = _CHECK_MODE, self.enabled
        return self

    def __exit__(self, *exc):
        global _CHECK_MODE
        _CHECK_MODE = self._old


def in_check_mode() -> bool:
    return _CHECK_MODE


def drop_mesh(args):
    """The reference's distributed classes take a device mesh as their first
    positional argument (e.g. nn/d_attention.py:24); on one GPU it carries no
    information, so it is accepted and ignored."""
    if args and not isinstance(args[0], (int, bool, float)):
        return args[1:]
    return args


def bf16(t: torch.Tensor) -> torch.Tensor:
    return t.detach().to(torch.bfloat16).contiguous()


def f32(t: torch.Tensor) -> torch.Tensor:
    return t.detach().to(torch.float32).contiguous()


def pad_to(w: torch.Tensor, *shape: int) -> torch.Tensor:
    """`w` in the leading corner of a zero tensor of `shape`."""
    out = torch.zeros(shape, dtype=w.dtype, device=w.device)
    out[tuple(slice(0, d) for d in w.shape)] = w.detach()
    return out


def pad_channels(x: torch.Tensor, width: int = 128) -> torch.Tensor:
    """[..., c] -> [..., width] with zeros behind the c real channels (a new tensor)."""
    return torch.nn.functional.pad(x, (0, width - x.shape[-1])).contiguous()


def pad_rows(w: torch.Tensor, multiple: int) -> torch.Tensor:
    rows = w.shape[0]
    target = (rows + multiple - 1) // multiple * multiple
    if target == rows:
        return w.contiguous()
    out = torch.zeros((target,) + tuple(w.shape[1:]), dtype=w.dtype, device=w.device)
    out[:rows] = w
    return out


def pack_swiglu(w1: torch.Tensor, block: int) -> torch.Tensor:
    """Re-order the rows of a GLU weight [2*hidden, c] (silu half first, linear
    half second) into alternating blocks of `block` silu rows and the `block`
    matching linear rows."""
    hidden = w1.shape[0] // 2
    if hidden % block:
        raise ValueError(f"hidden size {hidden} is not a multiple of {block}")
    a = w1[:hidden].reshape(hidden // block, block, -1)
    b = w1[hidden:].reshape(hidden // block, block, -1)
    return torch.cat([a, b], dim=1).reshape(2 * hidden, -1).contiguous()


def fragments(w: torch.Tensor, swap23: bool = False) -> torch.Tensor:
    """A matrix [rows, k] (multiples of 32 and 16) in the order in which MFMA fragments are loaded: 16-byte pieces of 8
    columns, lane by lane, 32 rows x 16 columns at a time.  swap23: with bits 2 and 3 of the row number exchanged (eight
    consecutive rows are then eight consecutive accumulator registers of a lane)."""
    rows, k = w.shape
    v = w.reshape(rows // 32, 2, 2, 2, 4, k // 16, 2, 8)
    return v.permute(0, 5, 6, 1, *((3, 2) if swap23 else (2, 3)), 4, 7).reshape(-1)


def point(s, *fields) -> None:
    """Set address fields of a library structure from packed weights: (field or (field, index), tensor, shape).  The
    structures carry no sizes, so what the operator layer checks of every tensor and packing does not settle (it makes
    contiguous tensors of the types that the library takes) is checked here: the shape, and one device for all, which is
    kept as `s.device` for the operator layer to compare with the activations'."""
    device = s.device
    for name, t, shape in fields:
        if t.shape != shape:
            raise ValueError(f"{name}: expected a weight {shape}, got {tuple(t.shape)}")
        if t.device != device:
            if device is not None:
                raise ValueError(f"{name}: on {t.device}, other weights of the block on {device}")
            s.device = device = t.device
        if name.__class__ is tuple:
            getattr(s, name[0])[name[1]] = t.data_ptr()
        else:
            setattr(s, name, t.data_ptr())


_EVERY = nn.modules.module


def as_written(*modules) -> bool:
    """Whether using each of (module, class) does what the class says and nothing else: no subclass, no forward hook (its
    own or one for all modules), no method replaced on the instance.  A run of modules that goes to the library as one
    call passes its modules by, so it is made for such modules only.  (Asked at every call: 0.2 us a module.)"""
    if _EVERY._global_forward_hooks or _EVERY._global_forward_pre_hooks:
        return False
    for m, cls in modules:
        d = m.__dict__
        if (m.__class__ is not cls or d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d or "run" in d
                or "packed" in d):
            return False
    return True


def packs_of(mods) -> list:
    return [m._packed or m.packed() for m in mods]


class HipModule(nn.Module):
    """A module whose `forward` runs on the HIP kernels.

    The packed device-side weights are derived from the nn.Parameters by
    `load_hip_params()` (the counterpart of the reference's
    `load_xsmm_params()`, e.g. nn/d_triangle_multiplication.py:126-138); it runs
    lazily on the first forward and again after `invalidate()`.  `xsmm_forward`
    and `load_xsmm_params` are kept as aliases so that the reference's plug-in
    loop (run_inference.py:197-218) binds these modules unchanged.
    """

    _native = None      # the packed weights as the library's structures, where a module makes them

    def __init__(self):
        super().__init__()
        self._packed = None

    # What is packed is derived from the parameters and is made again on demand: a copied or stored module is its
    # parameters (the structures hold device addresses, which would mean nothing elsewhere).
    def __getstate__(self):
        state = dict(self.__dict__, _packed=None)
        state.pop("_native", None)
        return state

    def __setstate__(self, state):
        super().__setstate__(state)
        self._packed = self._native = None

    def invalidate(self):
        """Drop the packed weights of this module and of every HIP module below
        it, however deeply nested (blocks usually sit in an nn.ModuleList)."""
        for m in self.modules():
            if isinstance(m, HipModule):
                m._packed = m._native = None

    def _apply(self, fn, *a, **k):  # .to() / .cuda() move parameters: repack afterwards
        self._packed = self._native = None
        return super()._apply(fn, *a, **k)

    def load_state_dict(self, *a, **k):
        self.invalidate()
        return super().load_state_dict(*a, **k)

    def _pack(self):
        raise NotImplementedError

    def _structures(self):
        """The library's structures of a module that has such, made from the packed weights."""

    def load_hip_params(self):
        _pack_all(self)
        return self

    def packed(self):
        if self._packed is None:
            self._packed = self._pack()
        return self._packed

    # reference plug-in protocol
    def load_xsmm_params(self):
        return self.load_hip_params()

    def hip_forward(self, *a, **k):
        return self.forward(*a, **k)

    def xsmm_forward(self, *a, **k):
        return self.forward(*a, **k)


def _pack_all(model: nn.Module) -> int:
    mods = [m for m in model.modules() if isinstance(m, HipModule)]
    for m in mods:
        m._packed = m._pack()
    for m in mods:
        try:
            m._structures()
        except ValueError:      # weights that do not go together: an error of the call that needs them, not of packing
            pass
    return len(mods)


def enable_hip(model: nn.Module) -> int:
    """Counterpart of ModelRunner.enable_xsmm (run_inference.py:197-218): packs
    the weights of every HIP module under `model`.  Returns how many were bound."""
    return _pack_all(model)
