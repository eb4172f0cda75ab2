"""GEMM operands derived from a quantised linear's stored state, shared by the dynamic and the static module.

The GEMM reads the weight as bytes ``[N, pad128(K)]`` and the weight scale as an fp32 vector ``[N]``.  The stored
state (``qweight`` [N, K], ``weight_scale`` [1, N] or [1]) already has that form when K is a multiple of 128 and the
scale is per channel; otherwise a zero-padded copy / the scalar written out per channel is kept beside the state,
never saved, rebuilt when the state changes, and built ahead of the first forward wherever the state is set
(conversion, ``load_state_dict``, ``.to(device)``).
"""
from __future__ import annotations

import torch
from torch import Tensor

from ... import _capi, ops


def _capturing(t: Tensor) -> bool:
    return t.device.type == "cuda" and torch.cuda.is_current_stream_capturing()


def _refresh_after_load(module, incompatible_keys) -> None:
    module.refresh_derived()


class DerivedOperands:
    """Mixin for a module with ``qweight``, ``weight_scale`` and ``out_features``."""

    # A module whose forward is quantiser + GEMM and whose state lives on the device keeps the arguments of that one call
    # ready: every torch call in a forward costs the host a microsecond or two, and a small linear's time is the host's.
    # The tensors alias the module's state (or are derived from it), so in-place updates of the aliased ones show through;
    # the tuple also remembers which state tensors it was built from, where they lived and, where a derived copy stands
    # for one, at which version, and a forward that finds anything else (a buffer or parameter replaced by assignment, by a
    # hook of an off-loading framework, or through `.data`) rebuilds it.  Whatever sets the state afresh
    # (conversion, load_state_dict, .to()) rebuilds it too.  Plain data only: a module must stay deep-copyable, and a
    # copy finds the addresses changed and rebuilds.
    _fast = None

    def _fast_arguments(self):
        """(x_fmt, w_fmt, element type of the output, scheme) of the one call, or None where the module needs more."""
        raise NotImplementedError

    def _fast_state(self):
        raise NotImplementedError

    def _build_fast(self) -> None:
        object.__setattr__(self, "_fast", None)
        args = self._fast_arguments()
        qw, ws, bp, xs = self._fast_state()
        if (args is None or qw.device.type != "cuda" or not qw.is_contiguous() or ops.is_tracing(qw)
                or torch.cuda.is_current_stream_capturing()):
            return
        wq, sw = self._gemm_weight(), self._weight_scale_vector()
        # (a tensor made in inference mode counts no versions: nothing can be derived from it that stays checkable)
        derived = [t for t, of in ((qw, wq), (ws, sw)) if of.data_ptr() != t.data_ptr()]
        if any(t.is_inference() for t in derived):
            return
        bias = None if bp is None else bp.detach()
        in_scale = None if xs is None else xs.detach()
        object.__setattr__(self, "_fast", (
            (wq, sw, bias, in_scale, self.in_features, *args), qw.device.index, qw, ws, bp, xs, qw.data_ptr(), ws.data_ptr(),
            0 if bp is None else bp.data_ptr(), 0 if xs is None else xs.data_ptr(),
            tuple((t, t._version) for t in derived)))

    def _fast_forward(self, input: Tensor, scale_fp32: bool):
        """The output, or None where the general forward has to look at the call."""
        f = self._fast
        if f is None or input.__class__ is not Tensor or torch.compiler.is_compiling():
            return None
        qw, ws, bp, xs = self._fast_state()
        if (qw is not f[2] or ws is not f[3] or bp is not f[4] or xs is not f[5] or qw.data_ptr() != f[6] or ws.data_ptr() != f[7]
                or (bp is not None and bp.data_ptr() != f[8]) or (xs is not None and xs.data_ptr() != f[9])
                or any(t._version != v for t, v in f[10])):
            self.refresh_derived()
            f = self._fast
            if f is None:
                return None
        if f[1] not in _capi._checked_devices:
            _capi.require_gfx950(f[1])
        out = _capi.native().linear(input, *f[0], scale_fp32, _capi.kernel_arg())
        if out is not None and out.__class__ is int:
            _capi.check(out, "linear")
        return out

    def _init_derived(self) -> None:
        self._packed = None  # (key, K-padded byte view of qweight)
        self._sw_vec = None  # (key, per-tensor weight scale once per output channel)
        self.register_load_state_dict_post_hook(_refresh_after_load)

    def _apply(self, fn, recurse=True):
        out = super()._apply(fn, recurse)  # .to(device) / .cuda(): the derived operands follow the state
        if not torch.compiler.is_compiling():
            self.refresh_derived()
        return out

    def refresh_derived(self) -> None:
        """Builds the derived operands now, so that a forward launches nothing but its kernels.  A module that
        does not live on a ROCm device (yet) builds them at its first forward there."""
        self._packed = self._sw_vec = None
        if self.qweight.device.type == "cuda":
            self._gemm_weight()
            self._weight_scale_vector()
        self._build_fast()

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
        key = (self.qweight.data_ptr(), self.qweight._version, str(qw.device))
        if self._packed is None or self._packed[0] != key:
            buf = torch.zeros((qw.shape[0], kp), dtype=qw.dtype, device=qw.device)
            buf[:, :k] = qw
            if _capturing(qw):
                # recorded, not executed: the buffer belongs to the graph's pool and holds data only after a
                # replay, so it must not be kept for later eager calls
                return buf
            self._packed = (key, buf)
        return self._packed[1]

    def _weight_scale_vector(self) -> Tensor:
        """weight_scale as the fp32 [N] vector the GEMM reads."""
        ws = self.weight_scale
        if ws.numel() != 1:
            return ws.view(-1)
        if ops.is_tracing(ws):
            return ops.broadcast_f32(ws.reshape(1).contiguous(), self.out_features)
        key = (ws.data_ptr(), ws._version, str(ws.device))
        if self._sw_vec is None or self._sw_vec[0] != key:
            vec = ops.broadcast_f32(ws.reshape(1).contiguous(), self.out_features)
            if _capturing(ws):
                return vec
            self._sw_vec = (key, vec)
        return self._sw_vec[1]

    def _check_device(self, dev) -> None:
        if self.qweight.device != dev:
            raise RuntimeError(f"Expected all tensors to be on the same device, but the input is on {dev} and this "
                               f"module's qweight on {self.qweight.device} (move the quantised model with .to(device))")
