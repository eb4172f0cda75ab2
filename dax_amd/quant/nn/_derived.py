"""GEMM operands derived from a quantised linear's stored state, shared by the dynamic and the static module.

The GEMM reads the weight as bytes ``[N, pad128(K)]`` and the weight scale as an fp32 vector ``[N]``.  The stored
state (``qweight`` [N, K], ``weight_scale`` [1, N] or [1]) already has that form when K is a multiple of 128 and the
scale is per channel; otherwise a zero-padded copy / the scalar written out per channel is kept beside the state,
never saved, rebuilt when the state changes, and built ahead of the first forward wherever the state is set
(conversion, ``load_state_dict``, ``.to(device)``).
"""
from __future__ import annotations

import weakref

import torch
from torch import Tensor

from ... import _capi, ops


def _capturing(t: Tensor) -> bool:
    return t.device.type == "cuda" and torch.cuda.is_current_stream_capturing()


def _refresh_after_load(module, incompatible_keys) -> None:
    module.refresh_derived()


class _Derived(tuple):
    """(what it was made from, tensor): a copy derived from a state tensor, good while that very tensor is still the module's
    state, lives where it lived and has not been written to.  It does not keep the state tensor alive, and a copied or
    unpickled module makes its own."""

    __slots__ = ()

    def __new__(cls, of: Tensor, made: Tensor):
        return super().__new__(cls, ((weakref.ref(of), of.data_ptr(), of._version), made))

    def is_from(self, t: Tensor) -> bool:
        ref, ptr, version = self[0]
        return ref() is t and t.data_ptr() == ptr and t._version == version

    def __reduce__(self):
        return type(None), ()


class DerivedOperands:
    """Mixin for a module with ``qweight``, ``weight_scale`` and ``out_features``."""

    # The forward of a module whose state lives on the device is one native call: every torch call in a forward costs the
    # host a microsecond or two, and a small linear's time is the host's.  The state goes into that call as it stands at the
    # time (a buffer or parameter replaced by assignment, by a hook of an off-loading framework, or through `.data`, and
    # any update in place, show through, and nothing is kept alive); only copies derived from it are kept, and only the
    # codes of the module's settings, with the settings they stand for beside them.
    _fast = None  # (settings, codes or None: these settings need more than the one call)

    def _fast_settings(self):
        """The settings that the codes are made of."""
        raise NotImplementedError

    def _fast_codes(self):
        """(x_fmt, w_fmt, element type of the output, scheme) of the one call, or None where the module needs more."""
        raise NotImplementedError

    def _fast_state(self):
        raise NotImplementedError

    def _fast_forward(self, input: Tensor, scale_fp32: bool):
        """The output, or None where the general forward has to look at the call."""
        if input.__class__ is not Tensor or torch.compiler.is_compiling():
            return None
        f, settings = self._fast, self._fast_settings()
        if f is None or f[0] != settings:
            f = (settings, self._fast_codes())
            object.__setattr__(self, "_fast", f)
        device = input.get_device()
        if f[1] is None or device < 0:
            return None
        wq, sw, bias, in_scale = self._fast_state()
        k = self.in_features
        if k % ops.K_ALIGN:
            d = self._packed
            if d is None or not d.is_from(wq):
                d = self._derive(wq, self._gemm_weight, "_packed")
                if d is None:
                    return None
            wq = d[1]
        d = self._sw_vec  # (per channel there is none)
        if d is not None:
            if not d.is_from(sw):
                self._sw_vec = None
                d = self._derive(sw, self._weight_scale_vector, "_sw_vec") if sw.numel() == 1 else None
            if d is not None:
                sw = d[1]
        if device not in _capi._checked_devices:
            _capi.require_gfx950(device)
        out = (_capi._native or _capi.native()).linear(input, wq, sw, bias, in_scale, k, *f[1], scale_fp32, _capi._kernel_arg)
        if out.__class__ is int:
            _capi.check(out, "linear")
        if out is None and d is None and sw.numel() == 1 and self._derive(sw, self._weight_scale_vector, "_sw_vec") is not None:
            return self._fast_forward(input, scale_fp32)  # (a scalar scale whose vector did not exist yet)
        return out

    def _derive(self, of: Tensor, make, name: str):
        """The copy derived from a state tensor, made now; None where none can be kept."""
        if of.device.type != "cuda" or of.is_inference() or ops.is_tracing(of) or torch.cuda.is_current_stream_capturing():
            return None
        make()
        return getattr(self, name)

    def _init_derived(self) -> None:
        self._packed = None  # _Derived: K-padded byte copy of qweight
        self._sw_vec = None  # _Derived: per-tensor weight scale once per output channel
        self.register_load_state_dict_post_hook(_refresh_after_load)

    def _apply(self, fn, recurse=True):
        out = super()._apply(fn, recurse)  # .to(device) / .cuda(): the derived operands follow the state
        if not torch.compiler.is_compiling():
            self.refresh_derived()
        return out

    def refresh_derived(self) -> None:
        """Builds the derived operands and the codes of the native call now, so that a forward launches nothing but its
        kernels.  A module that does not live on a ROCm device (yet) builds them at its first forward there."""
        self._packed = self._sw_vec = None
        qw, ws = self.qweight, self.weight_scale
        if qw.device.type == "cuda":
            if qw.shape[1] % ops.K_ALIGN or not qw.is_contiguous():
                self._gemm_weight()
            if ws.numel() == 1:
                self._weight_scale_vector()
            object.__setattr__(self, "_fast", (self._fast_settings(), self._fast_codes()))

    def _gemm_weight(self) -> Tensor:
        """qweight as the byte matrix [N, pad128(K)] the GEMM reads."""
        qw = self.qweight.detach()
        if qw.dtype != torch.int8:
            qw = qw.view(torch.uint8)
        k = qw.shape[1]
        kp = ops.pad_k(k)
        if kp == k and qw.is_contiguous():
            return qw
        if ops.is_tracing(qw):
            # a traced graph cannot key a cache on the storage address: pad inside the graph
            return torch.nn.functional.pad(qw, (0, kp - k)).contiguous()
        if self._packed is None or not self._packed.is_from(self.qweight):
            buf = torch.zeros((qw.shape[0], kp), dtype=qw.dtype, device=qw.device)
            buf[:, :k] = qw
            if _capturing(qw):
                # recorded, not executed: the buffer belongs to the graph's pool and holds data only after a
                # replay, so it must not be kept for later eager calls
                return buf
            self._packed = _Derived(self.qweight, buf)
        return self._packed[1]

    def _weight_scale_vector(self) -> Tensor:
        """weight_scale as the fp32 [N] vector the GEMM reads."""
        ws = self.weight_scale
        if ws.numel() != 1:
            return ws.view(-1)
        if ops.is_tracing(ws):
            return ops.broadcast_f32(ws.reshape(1).contiguous(), self.out_features)
        if self._sw_vec is None or not self._sw_vec.is_from(ws):
            vec = ops.broadcast_f32(ws.reshape(1).contiguous(), self.out_features)
            if _capturing(ws):
                return vec
            self._sw_vec = _Derived(ws, vec)
        return self._sw_vec[1]

    def _check_device(self, dev) -> None:
        if self.qweight.device != dev:
            raise RuntimeError(f"Expected all tensors to be on the same device, but the input is on {dev} and this "
                               f"module's qweight on {self.qweight.device} (move the quantised model with .to(device))")
