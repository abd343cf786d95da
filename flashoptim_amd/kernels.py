"""Host launch wrappers: plain functions of torch tensors and Python scalars that enqueue the HIP kernels.

This is the boundary the optimizer classes call.  Names, argument order and error behaviour follow the
launch wrappers of the reference (``/root/reference/flashoptim/optimizers.py``, cited as ``ref:``):
``quantize`` (ref:2446), ``dequantize`` (ref:2501), ``reconstruct_fp32_param`` (ref:2835),
``compute_ecc_bits`` (ref:2895), ``_fused_adam_step`` (ref:2203), ``_fused_momentum_step`` (ref:1535).
All of them are asynchronous on the current stream of the tensors' device and mutate their outputs in place.
"""

from __future__ import annotations

import ctypes
from bisect import bisect_left, bisect_right
from typing import Optional

import torch

from . import _hostscan, _native
from ._native import DTYPE_CODE

GROUP_SIZE = 32

_NUM_MANTISSA_BITS = {torch.float16: 10, torch.bfloat16: 7, torch.float32: 23}


def _require_device(t: torch.Tensor, what: str) -> None:
    if not t.is_cuda:
        raise NotImplementedError(
            f"{what}: flashoptim_amd only runs on a ROCm GPU; got a {t.dtype} tensor on {t.device} with "
            f"shape {tuple(t.shape)}."
        )


def _require_same_device(ref: torch.Tensor, other: Optional[torch.Tensor], what: str) -> None:
    """The kernels dereference raw addresses: a tensor on another device (or the host) would fault the GPU."""
    if other is not None and other.device != ref.device:
        raise ValueError(f"{what} is on {other.device}, expected {ref.device}.")


def _ecc_bytes(errors: Optional[torch.Tensor]) -> int:
    """Width of the correction term: 0 (none), 1 (int8, 24-bit master) or 2 (int16, 32-bit master);
    same rule as ``_ecc_kernel_params`` (ref:1514-1524)."""
    if errors is None:
        return 0
    width = errors.element_size()
    if width not in (1, 2):
        raise ValueError(f"Errors must have width 1 or 2, not {width}.")
    return width


def _check_group_size(group_size: int) -> None:
    if group_size != GROUP_SIZE:
        raise ValueError(f"group_size is fixed at {GROUP_SIZE} in the HIP kernels; got {group_size}.")


# ------------------------------------------------------------------------------------------ group codec


def _check_values(x: torch.Tensor) -> None:
    _require_device(x, "quantize")
    if x.dtype not in DTYPE_CODE:
        raise ValueError(f"quantize expects fp32, bf16 or fp16 input, got {x.dtype}.")


def quantize(
    x_float: torch.Tensor,
    out_int8: Optional[torch.Tensor] = None,
    out_scales: Optional[torch.Tensor] = None,
    signed: bool = True,
    group_size: int = 32,
    sqrt: bool = False,
    softsign: bool = True,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Group-quantise a floating tensor to 8-bit codes plus one fp16 scale per 32 elements.

    Returns ``(codes, scales)``: codes have the shape of ``x_float`` (int8 when ``signed`` else uint8),
    scales are fp16 ``[ceil(N/32)]`` (ref:2476-2498).
    """
    _check_group_size(group_size)
    _check_values(x_float)
    x = x_float if x_float.is_contiguous() else x_float.contiguous()
    n = x.numel()
    if out_int8 is None:
        out_int8 = torch.empty_like(x, dtype=torch.int8 if signed else torch.uint8)
    if out_scales is None:
        out_scales = torch.empty((n + GROUP_SIZE - 1) // GROUP_SIZE, device=x.device, dtype=torch.float16)
    if out_int8.numel() != n or not out_int8.is_contiguous() or out_int8.element_size() != 1:
        raise ValueError("out_int8 must be a contiguous 1-byte tensor with as many elements as the input")
    if (out_scales.numel() < (n + GROUP_SIZE - 1) // GROUP_SIZE or out_scales.dtype != torch.float16
            or not out_scales.is_contiguous()):
        raise ValueError("out_scales must be contiguous fp16 with at least ceil(N/32) elements")
    _require_same_device(x, out_int8, "out_int8")
    _require_same_device(x, out_scales, "out_scales")
    if n > 0:
        with _native.device_guard(x.device):
            rc = _native.lib().fo_quantize(
                x.data_ptr(), DTYPE_CODE[x.dtype], out_int8.data_ptr(), out_scales.data_ptr(), n,
                int(signed), int(sqrt), int(softsign), _native.current_stream_ptr(x.device),
            )
        _native.check(rc, "fo_quantize")
    return out_int8, out_scales


def _check_codes(codes: torch.Tensor, scales: torch.Tensor, signed: bool) -> None:
    _require_device(codes, "dequantize")
    if codes.dtype != (torch.int8 if signed else torch.uint8):
        raise ValueError(f"codes must be {'int8' if signed else 'uint8'} for signed={signed}, got {codes.dtype}.")
    if scales.dtype != torch.float16:
        raise ValueError(f"scales must be fp16, got {scales.dtype}.")
    if scales.numel() < (codes.numel() + GROUP_SIZE - 1) // GROUP_SIZE:
        raise ValueError("too few scales for the number of codes")
    _require_same_device(codes, scales, "in_scales")


def dequantize(
    in_int8: torch.Tensor,
    in_scales: torch.Tensor,
    out_float: Optional[torch.Tensor] = None,
    signed: bool = True,
    group_size: int = 32,
    sqrt: bool = False,
    softsign: bool = True,
) -> torch.Tensor:
    """Inverse of :func:`quantize`; returns fp32 with the shape of the codes (ref:2529-2538)."""
    _check_group_size(group_size)
    _check_codes(in_int8, in_scales, signed)
    codes = in_int8 if in_int8.is_contiguous() else in_int8.contiguous()
    scales = in_scales if in_scales.is_contiguous() else in_scales.contiguous()
    n = codes.numel()
    if out_float is None:
        out_float = torch.empty_like(codes, dtype=torch.float32)
    if out_float.dtype != torch.float32 or out_float.numel() != n or not out_float.is_contiguous():
        raise ValueError("out_float must be a contiguous fp32 tensor with as many elements as the codes")
    _require_same_device(codes, out_float, "out_float")
    if n > 0:
        with _native.device_guard(codes.device):
            rc = _native.lib().fo_dequantize(
                codes.data_ptr(), scales.data_ptr(), out_float.data_ptr(), n, int(signed), int(sqrt),
                int(softsign), _native.current_stream_ptr(codes.device),
            )
        _native.check(rc, "fo_dequantize")
    return out_float


# --------------------------------------------------------------------------- conversions of many tensors


def _codec_flags(signed: bool, sqrt: bool, softsign: bool) -> int:  # fo_codec_flags
    return (1 if signed else 0) | (2 if sqrt else 0) | (4 if softsign else 0)


class _Spans:
    """A set of addresses, held as disjoint spans in ascending order."""

    __slots__ = ("_first", "_end")

    def __init__(self) -> None:
        self._first: list = []
        self._end: list = []

    def meets(self, first: int, end: int) -> bool:
        i = bisect_right(self._first, first)
        return (i > 0 and self._end[i - 1] > first) or (i < len(self._first) and self._first[i] < end)

    def add(self, first: int, end: int) -> None:
        starts, ends = self._first, self._end
        i = bisect_right(starts, first)
        if (i == 0 or ends[i - 1] <= first) and (i == len(starts) or starts[i] >= end):
            starts.insert(i, first)
            ends.insert(i, end)
            return
        lo, hi = bisect_right(ends, first), bisect_left(starts, end)  # the spans it overlaps
        starts[lo:hi], ends[lo:hi] = [min(first, starts[lo])], [max(end, ends[hi - 1])]


def _span(t: torch.Tensor) -> tuple[int, int]:
    """First and end address of the elements of a tensor (strides are never negative)."""
    extent = t.numel()
    if extent and not t.is_contiguous():
        extent = 1 + sum((size - 1) * stride for size, stride in zip(t.shape, t.stride()))
    first = t.data_ptr()
    return first, first + extent * t.element_size()


# Bytes of copies (a host value's device copy, a checkpoint's cast values) that a ConversionBatch keeps alive before it
# launches what it has: such a list would otherwise need the memory of all its copies at once.  A launch over this much takes
# 70 us and more, beside which its own cost of a few us does not count, least of all next to the copies.
_COPIES_HELD = 256 << 20


class ConversionBatch:
    """Conversions of many tensors, issued as one launch per kind, dtype and device (up to 64 tensors each) instead of
    one or two launches per tensor.

    A method allocates its output and returns it at once; the values are there, in stream order, after ``launch()``.
    A batch is used by one thread, inside one call of this package.

    ``lasting``: the id()s of the inputs that outlive the batch; others are copies that nobody else holds.  None: every
    input outlives it, but for those a caller names (``hold_copy``).
    """

    def __init__(self, lasting: Optional[set] = None) -> None:
        self._lasting = lasting
        self._copied = 0  # bytes of the copies it keeps alive
        self._jobs: dict = {}  # (entry point, *its leading arguments, device) -> flat list of fo_convert_job words
        self._keepalive: list = []  # inputs must outlive the launch
        # memory that pending imports read and write: addresses, since one memory can belong to several storage objects
        # (dlpack, tensors of other libraries)
        self._import_sources, self._import_targets = _Spans(), _Spans()
        self._importing = False

    def _add(self, entry: tuple, device: torch.device, src: torch.Tensor, src2, dst: torch.Tensor, dst2, flags: int = 0) -> None:
        ptr = _native.ptr
        self._jobs.setdefault((entry, device), []).extend(
            (src.data_ptr(), ptr(src2) or 0, dst.data_ptr(), ptr(dst2) or 0, dst.numel(), flags))
        self._keepalive.append((src, src2, dst, dst2))

    def hold_copy(self, t: torch.Tensor) -> torch.Tensor:
        """`t`, the next input, which is freed with the launch."""
        size = t.numel() * t.element_size()
        if self._copied + size > _COPIES_HELD:
            self.launch()
        self._copied += size
        return t

    def _dense(self, t: torch.Tensor) -> torch.Tensor:
        return t if t.is_contiguous() else self.hold_copy(t.contiguous())

    def dequantize_bf16(self, codes: torch.Tensor, scales: torch.Tensor, signed: bool, sqrt: bool, softsign: bool) -> torch.Tensor:
        """``dequantize(codes, scales, ...).to(torch.bfloat16)``."""
        _check_codes(codes, scales, signed)
        codes, scales = codes.contiguous(), scales.contiguous()  # a state's always are
        out = torch.empty_like(codes, dtype=torch.bfloat16)
        if codes.numel() > 0:
            self._add(("fo_dequantize_many", DTYPE_CODE[torch.bfloat16]), codes.device, codes, scales, out, None,
                      _codec_flags(signed, sqrt, softsign))
        return out

    def widen_int8(self, values: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
        """``values.to(dtype)`` of an int8 tensor, dtype bf16 or fp16."""
        if (type(values) is not torch.Tensor or not values.is_cuda or values.dtype != torch.int8 or values.is_neg()
                or not values.is_contiguous() or dtype not in (torch.bfloat16, torch.float16)):
            return values.to(dtype=dtype)
        out = torch.empty_like(values, dtype=dtype)
        if values.numel() > 0:
            self._add(("fo_int8_widen_many", DTYPE_CODE[dtype]), values.device, values, None, out, None)
        return out

    def quantize(self, x: torch.Tensor, signed: bool, sqrt: bool, softsign: bool) -> tuple[torch.Tensor, torch.Tensor]:
        """:func:`quantize` of one tensor."""
        _check_values(x)
        if not x.is_contiguous():
            x = self.hold_copy(x.contiguous())
        elif self._lasting is not None and id(x) not in self._lasting:
            self.hold_copy(x)
        n = x.numel()
        codes = torch.empty_like(x, dtype=torch.int8 if signed else torch.uint8)
        scales = torch.empty((n + GROUP_SIZE - 1) // GROUP_SIZE, device=x.device, dtype=torch.float16)
        if n > 0:
            self._add(("fo_quantize_many", DTYPE_CODE[x.dtype]), x.device, x, None, codes, scales, _codec_flags(signed, sqrt, softsign))
        return codes, scales

    def narrow_to_int8(self, values: torch.Tensor) -> torch.Tensor:
        """``values.to(torch.int8)`` of a bf16 or fp16 tensor."""
        if (type(values) is not torch.Tensor or not values.is_cuda or not values.is_contiguous() or values.is_neg()
                or values.dtype not in (torch.bfloat16, torch.float16)):
            return values.to(dtype=torch.int8)
        out = torch.empty_like(values, dtype=torch.int8)
        if values.numel() > 0:
            if self._lasting is not None and id(values) not in self._lasting:
                self.hold_copy(values)
            self._add(("fo_int8_narrow_many", DTYPE_CODE[values.dtype]), values.device, values, None, out, None)
        return out

    def import_fp32(self, x: torch.Tensor, narrow: torch.Tensor, error_bits: torch.Tensor) -> Optional[torch.Tensor]:
        """``narrow.copy_(x)`` and the new correction term ``compute_ecc_bits(x, narrow, ...)`` of `error_bits`' width in
        one pass; None (and nothing done) where the tensors are not laid out for it."""
        if (not type(x) is type(narrow) is torch.Tensor or x.dtype != torch.float32 or x.shape != narrow.shape
                or not x.is_contiguous() or not narrow.is_contiguous() or not narrow.is_cuda or x.device != narrow.device
                or x.is_neg() or narrow.is_neg() or narrow.dtype not in (torch.bfloat16, torch.float16) or error_bits.element_size() not in (1, 2)):
            return None
        width = error_bits.element_size()
        out = torch.empty(narrow.shape, dtype=torch.int8 if width == 1 else torch.int16, device=narrow.device)
        n = narrow.numel()
        if n == 0:
            return out
        source, target = x.data_ptr(), narrow.data_ptr()
        source_end, target_end = source + 4 * n, target + 2 * n
        if source < target_end and target < source_end:
            return None
        if self._importing:
            self._order_spans(source, source_end, target, target_end)
        self._import_sources.add(source, source_end)
        self._import_targets.add(target, target_end)
        self._importing = True
        self._add(("fo_ecc_narrow_many", DTYPE_CODE[narrow.dtype], width), narrow.device, x, None, narrow, out)
        return out

    def reconstruct_fp32(self, param: torch.Tensor, error_bits: torch.Tensor) -> torch.Tensor:
        """:func:`reconstruct_fp32_param` of one parameter."""
        _check_join(param, error_bits)
        out = torch.empty(param.shape, dtype=torch.float32, device=param.device)
        if param.numel() > 0:
            self._add(("fo_ecc_join_many", DTYPE_CODE[param.dtype], error_bits.element_size()), param.device,
                      self._dense(param), self._dense(error_bits), out, None)
        return out

    def launch(self) -> None:
        """Enqueue everything collected so far on the current stream of each device."""
        jobs, self._jobs = self._jobs, {}
        for ((name, *args), device), words in jobs.items():
            table = (ctypes.c_int64 * len(words))(*words)
            with _native.device_guard(device):
                rc = getattr(_native.lib(), name)(table, len(words) // 6, *args, _native.current_stream_ptr(device))
            _native.check(rc, name)
        self._keepalive.clear()
        self._copied = 0
        if self._importing:
            self._import_sources, self._import_targets = _Spans(), _Spans()
            self._importing = False

    def order_import(self, value: torch.Tensor, param: torch.Tensor) -> None:
        """``launch()`` if a pending import writes the memory of `value`, or reads or writes that of `param`: tensors that
        share memory keep the order of the calls, and jobs of one launch have none.  Parameters carved from one buffer
        side by side share a launch."""
        if not self._importing:
            return
        if not type(value) is type(param) is torch.Tensor:  # whose memory cannot be asked for
            self.launch()
            return
        self._order_spans(*_span(value), *_span(param))

    def _order_spans(self, source: int, source_end: int, target: int, target_end: int) -> None:
        writes = self._import_targets
        if writes.meets(target, target_end) or writes.meets(source, source_end) or self._import_sources.meets(target, target_end):
            self.launch()


# ------------------------------------------------------------------------------------------------- ECC


def _check_join(param: torch.Tensor, error_bits: torch.Tensor) -> None:
    if param.dtype == torch.float32:
        raise ValueError(
            "param is already fp32; ECC reconstruction is only meaningful for narrow dtypes (bf16, fp16). "
            f"Got {param.dtype}."
        )
    if param.dtype not in _NUM_MANTISSA_BITS:
        raise ValueError(f"Unsupported param dtype {param.dtype}; expected one of {list(_NUM_MANTISSA_BITS)}.")
    if error_bits.dtype not in (torch.int8, torch.int16):
        raise ValueError(f"error_bits must be int8 or int16, got {error_bits.dtype}.")
    _require_device(param, "reconstruct_fp32_param")
    if error_bits.numel() != param.numel():
        raise ValueError("error_bits must have as many elements as param")
    _require_same_device(param, error_bits, "error_bits")


def reconstruct_fp32_param(param: torch.Tensor, error_bits: torch.Tensor) -> torch.Tensor:
    """fp32 master weights from a bf16/fp16 parameter and its int8/int16 correction term (ref:2835-2892)."""
    batch = ConversionBatch()
    out = batch.reconstruct_fp32(param, error_bits)
    batch.launch()
    return out


def compute_ecc_bits(
    fp32_param: torch.Tensor, narrow_param: torch.Tensor, master_bytewidth: int = 4
) -> torch.Tensor:
    """Correction term (int8 for 3-byte, int16 for 4-byte masters) such that
    ``reconstruct_fp32_param(narrow_param, result)`` approximates ``fp32_param`` (ref:2895-2970)."""
    if fp32_param.dtype != torch.float32:
        raise ValueError(f"fp32_param must be float32, got {fp32_param.dtype}.")
    if narrow_param.dtype not in (torch.bfloat16, torch.float16):
        raise ValueError(f"narrow_param must be bf16 or fp16, got {narrow_param.dtype}.")
    narrow_bytes = narrow_param.element_size()
    num_err_bytes = master_bytewidth - narrow_bytes
    if num_err_bytes not in (1, 2):
        raise ValueError(
            f"Unsupported dtype combination: master_bytewidth={master_bytewidth} to {narrow_param.dtype} "
            f"({narrow_bytes} bytes). Error byte width {num_err_bytes} must be 1 or 2."
        )
    _require_device(narrow_param, "compute_ecc_bits")
    if fp32_param.numel() != narrow_param.numel():
        raise ValueError("fp32_param and narrow_param must have the same number of elements")
    out = torch.empty(
        narrow_param.shape, dtype=torch.int8 if num_err_bytes == 1 else torch.int16, device=narrow_param.device
    )
    n = narrow_param.numel()
    if n > 0:
        x = fp32_param.to(narrow_param.device).resolve_neg().contiguous()
        narrow = narrow_param.contiguous()
        with _native.device_guard(narrow.device):
            rc = _native.lib().fo_ecc_split(
                x.data_ptr(), narrow.data_ptr(), DTYPE_CODE[narrow.dtype], out.data_ptr(), num_err_bytes, n,
                _native.current_stream_ptr(narrow.device),
            )
        _native.check(rc, "fo_ecc_split")
    return out


# ------------------------------------------------------------------------------------------ fused steps


def _check_step_tensors(param: torch.Tensor, grad: torch.Tensor, errors: Optional[torch.Tensor]) -> None:
    """Everything the step kernels assume about param / grad / ECC and cannot check from raw addresses."""
    _require_device(param, "fused step")
    if param.dtype not in DTYPE_CODE:
        raise ValueError(f"Unsupported parameter dtype {param.dtype}.")
    if grad.dtype != param.dtype:
        raise ValueError(f"grad dtype {grad.dtype} must match param dtype {param.dtype}.")
    if grad.numel() != param.numel():
        raise ValueError("grad and param must have the same number of elements")
    if grad.device != param.device:
        raise ValueError("grad and param must be on the same device")
    if not param.is_contiguous() or not grad.is_contiguous():
        raise RuntimeError("the fused kernels need contiguous param and grad tensors")
    if errors is not None:
        if errors.numel() != param.numel():
            raise ValueError("error_bits and param must have the same number of elements")
        if not errors.is_contiguous():
            raise RuntimeError("the fused kernels need a contiguous error_bits tensor")
        _require_same_device(param, errors, "error_bits")


def _check_moment(param: torch.Tensor, values: torch.Tensor, scales: Optional[torch.Tensor], quantized: bool,
                  signed: bool, name: str) -> None:
    """One optimizer state as the step kernels read and write it: 8-bit codes with fp16 group scales, or a tensor
    of the parameter's dtype."""
    n = param.numel()
    if values.numel() != n or not values.is_contiguous():
        raise ValueError(f"{name} must be contiguous with as many elements as param ({n}), got {values.numel()}.")
    _require_same_device(param, values, name)
    if not quantized:
        if values.dtype != param.dtype:
            raise ValueError(f"unquantised {name} must have the parameter's dtype {param.dtype}, got {values.dtype}.")
        return
    if values.dtype != (torch.int8 if signed else torch.uint8):
        raise ValueError(f"quantised {name} must be {'int8' if signed else 'uint8'}, got {values.dtype}.")
    if scales is None or scales.dtype != torch.float16 or not scales.is_contiguous():
        raise ValueError(f"{name} scales must be a contiguous fp16 tensor.")
    if scales.numel() < (n + GROUP_SIZE - 1) // GROUP_SIZE:
        raise ValueError(f"{name} scales hold {scales.numel()} groups, {(n + GROUP_SIZE - 1) // GROUP_SIZE} needed.")
    _require_same_device(param, scales, f"{name} scales")


def _step_args(param: torch.Tensor, grad: torch.Tensor, errors: Optional[torch.Tensor], mom: Optional[torch.Tensor],
               mom_scales: Optional[torch.Tensor], var: Optional[torch.Tensor], var_scales: Optional[torch.Tensor],
               quantized: bool) -> tuple:
    """The checked arguments of a single-tensor step: addresses of mom, mom_scales, var, var_scales, param, grad, errors,
    then elements, dtype code, ECC bytes.  The checks run in C++ where the helper is built (0.4 instead of 4 us); what
    it does not vouch for comes here, and the exceptions are raised here."""
    if _hostscan.step_args is not None:
        args = _hostscan.step_args(param, grad, errors, mom, mom_scales, var, var_scales, quantized)
        if args is not None:
            return args
    _check_step_tensors(param, grad, errors)
    if mom is not None:
        _check_moment(param, mom, mom_scales, quantized, True, "mom" if var is not None else "momentum")
    if var is not None:
        _check_moment(param, var, var_scales, quantized, False, "var")
    ecc_bytes = _ecc_bytes(errors)
    ptr = _native.ptr
    return (ptr(mom), ptr(mom_scales) if quantized else None, ptr(var), ptr(var_scales) if quantized else None,
            param.data_ptr(), grad.data_ptr(), ptr(errors), param.numel(), DTYPE_CODE[param.dtype], ecc_bytes)


def _fused_adam_step(
    mom: torch.Tensor,
    mom_scales_f16: torch.Tensor,
    var: torch.Tensor,
    var_scales_f16: torch.Tensor,
    param: torch.Tensor,
    grad: torch.Tensor,
    errors: Optional[torch.Tensor],
    lr: float,
    beta1: float,
    beta2: float,
    eps: float,
    weight_decay: float,
    decoupled: bool,
    step: int,
    quantize_optim_states: bool = True,
    group_size: int = 32,
    exact_update: bool = False,
) -> None:
    """One fused Adam/AdamW step on one contiguous tensor (ref:2203-2251).  ``weight_decay`` is already
    multiplied by lr (or lr/initial_lr) for the decoupled optimizers.

    ``exact_update`` (not in the reference): evaluate the update operation by operation as the reference writes it
    on every element of every variant; every output bit then equals an IEEE evaluation of the reference's formulas.
    The default already does so except for bf16 parameters with an int8 correction term and 2-byte parameters
    without one, whose folded update keeps every master weight within one unit of master precision."""
    _check_group_size(group_size)
    n = param.numel()
    if n == 0:
        return
    args = _step_args(param, grad, errors, mom, mom_scales_f16, var, var_scales_f16, quantize_optim_states)
    with _native.device_guard(param.device):
        entry = _native.lib().fo_adam_step_exact if exact_update else _native.lib().fo_adam_step
        rc = entry(*args, int(quantize_optim_states), lr, beta1, beta2, eps, weight_decay, int(decoupled), int(step),
                   _native.current_stream_ptr(param.device))
    _native.check(rc, "fo_adam_step")


def _fused_momentum_step(
    momentum: torch.Tensor,
    scales_f16: torch.Tensor,
    param: torch.Tensor,
    grad: torch.Tensor,
    errors: Optional[torch.Tensor],
    lr: float,
    mom_coef: float,
    update_coef: float,
    weight_decay: float,
    decoupled: bool = False,
    nesterov: bool = False,
    do_lion: bool = False,
    quantize_optim_states: bool = True,
    group_size: int = 32,
) -> None:
    """One fused SGD/SGDW/Nesterov/Lion step on one contiguous tensor (ref:1535-1579)."""
    _check_group_size(group_size)
    n = param.numel()
    if n == 0:
        return
    mom_ptr, scales_ptr, _, _, *args = _step_args(param, grad, errors, momentum, scales_f16, None, None, quantize_optim_states)
    with _native.device_guard(param.device):
        rc = _native.lib().fo_momentum_step(
            mom_ptr, scales_ptr, *args, int(quantize_optim_states), lr, mom_coef, update_coef, weight_decay,
            int(decoupled), int(nesterov), int(do_lion), _native.current_stream_ptr(param.device),
        )
    _native.check(rc, "fo_momentum_step")


def _sgd_plain_step(
    param: torch.Tensor,
    grad: torch.Tensor,
    errors: Optional[torch.Tensor],
    lr: float,
    weight_decay: float,
    decoupled: bool = False,
) -> None:
    """Momentum-free SGD step: the branch the reference evaluates with eager PyTorch ops (ref:1447-1465),
    here one kernel."""
    n = param.numel()
    if n == 0:
        return
    args = _step_args(param, grad, errors, None, None, None, None, False)
    with _native.device_guard(param.device):
        rc = _native.lib().fo_sgd_plain_step(*args[4:], lr, weight_decay, int(decoupled), _native.current_stream_ptr(param.device))
    _native.check(rc, "fo_sgd_plain_step")


def absmax_many(tensors) -> list:
    """Largest magnitude of every tensor with one launch per (device, dtype); see ``launcher.absmax_many``."""
    from .launcher import absmax_many as _impl

    return _impl(tensors)


def copy_bytes(dst: torch.Tensor, src: torch.Tensor) -> None:
    """Device copy with the step kernels' access shape; a measurement aid (counter calibration, attainable
    streaming rate)."""
    _require_device(src, "copy_bytes")
    _require_same_device(src, dst, "dst")
    nbytes = src.numel() * src.element_size()
    if dst.numel() * dst.element_size() != nbytes:
        raise ValueError("dst and src must have the same size in bytes")
    if not src.is_contiguous() or not dst.is_contiguous():
        raise ValueError("copy_bytes needs contiguous tensors")
    with _native.device_guard(src.device):
        diag = _native.diag_lib()
        rc = diag.fo_copy_bytes(dst.data_ptr(), src.data_ptr(), nbytes, _native.current_stream_ptr(src.device))
    _native.check(rc, "fo_copy_bytes", diag)
