"""Tensor-level wrappers over the C ABI (include/mxfp8.h).

PyTorch is used for device memory and the current HIP stream only; every computation is a
call into libmxfp8_gfx950.so.  There is no fallback path: CPU tensors are rejected.
"""
from __future__ import annotations

import os
from ctypes import c_int32, c_int64
from typing import NamedTuple

import torch

from . import _lib
from ._lib import MX_SCALE_FLOOR, MX_SCALE_RCEIL, MX_SCALES_MFMA, MX_SCALES_ROWMAJOR

BLOCK = 32  # torchtitan/components/quantization/__init__.py:36

SCALE_MODES = {"floor": MX_SCALE_FLOOR, "rceil": MX_SCALE_RCEIL}


class MXData(NamedTuple):
    """e4m3 codes [rows, cols] (uint8) + E8M0 scales, blocks of 32 along `cols`."""

    codes: torch.Tensor
    scales: torch.Tensor
    scale_order: int  # MX_SCALES_ROWMAJOR: [rows, cols/32]; MX_SCALES_MFMA: flat re-laid buffer


class KernelTimer:
    """Optional per-launch timing with HIP events on the launch stream (used by bench.py).

    While a timer is installed with ``set_kernel_timer`` every library call is bracketed by two
    events recorded on the stream it is launched on; ``summary()`` synchronises once and
    returns {kernel name: (launches, mean milliseconds)}.
    """

    def __init__(self):
        self.records = []

    def bracket(self, name: str, device):
        start = torch.cuda.Event(enable_timing=True)
        stop = torch.cuda.Event(enable_timing=True)
        self.records.append((name, start, stop))
        return start, stop

    def summary(self):
        torch.cuda.synchronize()
        acc: dict[str, list[float]] = {}
        for name, a, b in self.records:
            acc.setdefault(name, []).append(a.elapsed_time(b))
        return {k: (len(v), sum(v) / len(v)) for k, v in acc.items()}


_timer: KernelTimer | None = None


def set_kernel_timer(timer: KernelTimer | None) -> None:
    global _timer
    _timer = timer


_entry_points: dict = {}  # C-ABI name -> bound function


def _call(name: str, tag: str, device, *args) -> None:
    """Run one C-ABI entry point on `device`'s current stream and raise on a non-zero status."""
    fn = _entry_points.get(name)
    if fn is None:
        fn = _entry_points[name] = getattr(_lib.load(), name)
    if _timer is None and device.index == _current_device():
        st = fn(*args)
    else:
        with torch.cuda.device(device):
            if _timer is None:
                st = fn(*args)
            else:
                start, stop = _timer.bracket(tag, device)
                start.record()
                st = fn(*args)
                stop.record()
    if st:
        _lib.check(st, name)


def _single(x: torch.Tensor) -> bool:
    """A launch on x may go through the native module, which makes the outputs and passes the pointers on in a third of
    the time (8 to 10 us a launch here); it returns None for operands that are not plain."""
    return x.is_cuda and _timer is None and not _watched()


def _mode(mode) -> int:
    if isinstance(mode, str):
        return SCALE_MODES[mode]
    if mode not in (MX_SCALE_FLOOR, MX_SCALE_RCEIL):
        raise ValueError(f"unknown scale mode {mode!r}")
    return int(mode)


# (device ordinal -> current stream as an address, without a torch.cuda.Stream object around it)
_current_device = getattr(torch._C, "_cuda_getDevice", lambda: -1)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t: torch.Tensor) -> int:
    return _raw_stream(t.device.index)


def _ptr(t: torch.Tensor) -> int:
    return t.data_ptr()


def _wrote(out: torch.Tensor) -> torch.Tensor:
    """A library write into a caller's tensor is an in-place op that autograd did not see: bump
    the version counter so that whatever is keyed on it (saved-tensor checks, the activation cast
    reuse of mx_tensor) notices the new contents."""
    torch.autograd.graph.increment_version(out)
    return out


def _check_hp(x: torch.Tensor) -> torch.Tensor:
    if not x.is_cuda:
        raise _lib.MXLibraryError("the MXFP8 kernels run on the GPU only; got a CPU tensor")
    if x.dtype != torch.bfloat16:
        raise TypeError(f"to_mx expects bfloat16, got {x.dtype}")
    if x.dim() != 2:
        raise ValueError("to_mx expects a 2-D tensor")
    if x.stride(1) != 1:
        x = x.contiguous()
    return x


def mfma_scale_bytes(rows: int, nblk: int) -> int:
    return ((rows + 127) // 128) * ((nblk + 1) // 2) * 256


def _alloc_scales(rows: int, nblk: int, order: int, device) -> torch.Tensor:
    if order == MX_SCALES_MFMA:
        return torch.empty(mfma_scale_bytes(rows, nblk), dtype=torch.uint8, device=device)
    return torch.empty((rows, nblk), dtype=torch.uint8, device=device)


def to_mx_dim0(x: torch.Tensor, mode="floor", order: int = MX_SCALES_ROWMAJOR) -> MXData:
    """Row-wise cast: blocks of 32 along the last dim of x [R, C]."""
    x = _check_hp(x)
    R, C = x.shape
    if C % BLOCK:
        raise ValueError(f"last dim {C} is not a multiple of {BLOCK}")
    codes = torch.empty((R, C), dtype=torch.uint8, device=x.device)
    scales = _alloc_scales(R, C // BLOCK, order, x.device)
    _call("mx_cast_dim0", "cast_dim0", x.device, _ptr(x), R, C, x.stride(0), _ptr(codes), _ptr(scales), _mode(mode), order, _stream(x))
    return MXData(codes, scales, order)


def to_mx_dim1(x: torch.Tensor, mode="floor", order: int = MX_SCALES_ROWMAJOR) -> MXData:
    """Column-wise cast of x [R, C]: codes [C, R], blocks of 32 down the rows of x."""
    x = _check_hp(x)
    R, C = x.shape
    if R % BLOCK:
        raise ValueError(f"first dim {R} is not a multiple of {BLOCK}")
    codes = torch.empty((C, R), dtype=torch.uint8, device=x.device)
    scales = _alloc_scales(C, R // BLOCK, order, x.device)
    _call("mx_cast_dim1", "cast_dim1", x.device, _ptr(x), R, C, x.stride(0), _ptr(codes), _ptr(scales), _mode(mode), order, _stream(x))
    return MXData(codes, scales, order)


# Row pitch of GEMM operands: codes whose rows lie a whole number of 4 KB apart (K = 4096, 14336,
# 16384 ...) put the lines a GEMM fetches together -- one 128-byte K block of 512 rows -- on few
# channels of the L2; 128 bytes between the end of a row and the start of the next spread them
# (measured on the dense GEMM inside the benchmark step: 2.4 % less time per launch).
# (MXFP8_CODE_PITCH_PAD in the environment: another multiple of 128, 0 = dense codes; for measurements.)
CODE_PITCH_PAD = int(os.environ.get("MXFP8_CODE_PITCH_PAD", "128"))


def _code_rows(rows: int, cols: int, pad: int, device, stack: int = 0) -> torch.Tensor:
    """uint8 [rows, cols] (or [stack, rows, cols]) whose rows lie cols + pad bytes apart."""
    shape = (rows, cols + pad) if not stack else (stack, rows, cols + pad)
    return torch.empty(shape, dtype=torch.uint8, device=device)[..., :cols]


def _pitch_ok(pad: int) -> int:
    """The row pitch padding the tile casts take: a multiple of 16 bytes (else none)."""
    return pad if pad > 0 and pad % 16 == 0 else 0


WHOLE_BLOCK = 128  # depth of the persistent GEMM's K blocks


def _operand_input(x: torch.Tensor, f32_ok: bool = False) -> torch.Tensor:
    """`x` as the tile casts read it: 16-byte aligned rows (a copy where they are not); bf16, or float32
    where the caller's kernel takes it."""
    if f32_ok and x.dtype == torch.float32 and x.is_cuda and x.dim() == 2:
        x = x if x.stride(1) == 1 else x.contiguous()
    else:
        x = _check_hp(x)
    if x.shape[1] % 8:
        return torch.nn.functional.pad(x, (0, -x.shape[1] % 8))
    if x.stride(0) * x.element_size() % 16 or x.data_ptr() % 16 or x.stride(0) < x.shape[1]:  # (expanded rows)
        return x.clone(memory_format=torch.contiguous_format)
    return x


class Operand:
    """One operand of the dense GEMMs, e4m3 codes [rows, k] and their MFMA-order scales, in one
    allocation: rows `ld` bytes apart from byte `at` on, scales from byte `scales_at` on.  Reads as
    an `MXData` (`codes`, `scales`, `scale_order`; views made when asked for).  `k` is the contraction in
    whole 128-deep blocks, `depth` how much of it is not zero fill: what the other operand must agree
    with.  One buffer and plain
    numbers instead of two to four tensors and their views: at small sizes making those takes the
    host longer than the GPU needs for the cast.  (`scales_buf`: the scales' own buffer, where they have
    one: an operand `around` two tensors.)"""

    __slots__ = ("buf", "rows", "k", "ld", "at", "scales_at", "depth", "scales_buf")
    scale_order = MX_SCALES_MFMA

    def __init__(self, buf: torch.Tensor, layout, scales_buf: torch.Tensor | None = None):
        self.buf = buf
        self.scales_buf = buf if scales_buf is None else scales_buf
        self.rows, self.k, self.ld, self.at, self.scales_at, self.depth = layout

    @property
    def layout(self):
        """What, with the buffer, makes the operand: for a backward that gets the buffer back."""
        return self.rows, self.k, self.ld, self.at, self.scales_at, self.depth

    @property
    def codes(self) -> torch.Tensor:
        return self.buf[self.at:self.at + self.rows * self.ld].view(self.rows, self.ld)[:, :self.k]

    @property
    def scales(self) -> torch.Tensor:
        return self.scales_buf[self.scales_at:self.scales_at + mfma_scale_bytes(self.rows, self.k // BLOCK)]

    @property
    def codes_ptr(self) -> int:
        return self.buf.data_ptr() + self.at

    @property
    def scales_ptr(self) -> int:
        return self.scales_buf.data_ptr() + self.scales_at

    def first_rows(self, n: int) -> "Operand":
        """The operand's first n rows (n rounds up to the same multiple of 128)."""
        return Operand(self.buf, (n, self.k, self.ld, self.at, self.scales_at, self.depth), self.scales_buf)

    @classmethod
    def of(cls, q: MXData) -> "Operand":
        """A copy of dense codes in whole blocks with MFMA-order scales as an operand."""
        rows, k = q.codes.shape
        if k % WHOLE_BLOCK or q.scale_order != MX_SCALES_MFMA:
            raise ValueError("an operand has whole blocks along its contraction and MFMA-order scales")
        out = _new_operand(rows, k, 0, q.codes.device)
        out.codes.copy_(q.codes)
        out.scales.copy_(q.scales)
        return out

    @classmethod
    def around(cls, codes: torch.Tensor, scales: torch.Tensor, depth: int) -> "Operand":
        """Dense codes [rows, whole blocks] of a contraction of `depth`, and their scales, as they lie."""
        rows, k = codes.shape
        return cls(codes, (rows, k, k, 0, 0, depth), scales)

    def data(self) -> MXData:
        return MXData(self.codes, self.scales, MX_SCALES_MFMA)


def saved_operand(buf: torch.Tensor, layout, device) -> Operand:
    """An operand from the buffer that a backward gets back and the layout that its forward kept.  The buffer may have
    been through hooks on saved tensors: strides that the kernels would not follow are laid out anew, another device,
    type or size is an error."""
    rows, k, _, _, scales_at, _ = layout
    need = scales_at + mfma_scale_bytes(rows, k // BLOCK)
    if buf.device != device or buf.dtype != torch.uint8 or buf.numel() < need:
        raise RuntimeError(f"a saved MXFP8 operand came back as {buf.dtype} x {buf.numel()} on {buf.device}; "
                           f"expected torch.uint8 x {need} on {device}")
    return Operand(buf if buf.is_contiguous() else buf.contiguous(), layout)


def saved_matrix(t: torch.Tensor | None, device) -> torch.Tensor | None:
    """`t`, which a backward gets back, as the kernels read it: dense, on `device` (see `saved_operand`)."""
    if t is not None and t.device != device:
        raise RuntimeError(f"a saved tensor came back on {t.device}; expected {device}")
    return t if t is None else t.contiguous()


def _new_operand(rows: int, cols: int, pad: int, device) -> Operand:
    """An operand of `rows` rows with a contraction of `cols` rounded up to whole 128-deep blocks."""
    k = -(-cols // WHOLE_BLOCK) * WHOLE_BLOCK
    ld = k + pad
    scales_at = (rows * ld + 255) & ~255
    buf = torch.empty(scales_at + ((rows + 127) & ~127) * (k // BLOCK), dtype=torch.uint8, device=device)
    return Operand(buf, (rows, k, ld, 0, scales_at, cols))


def _new_operand_pair(rows: int, cols: int, pad: int, device):
    """Two operands of one shape in one buffer, codes and then scales stacked."""
    k = -(-cols // WHOLE_BLOCK) * WHOLE_BLOCK
    ld, scale_bytes = k + pad, ((rows + 127) & ~127) * (k // BLOCK)
    scales_at = (2 * rows * ld + 255) & ~255
    buf = torch.empty(scales_at + 2 * scale_bytes, dtype=torch.uint8, device=device)
    return (Operand(buf, (rows, k, ld, 0, scales_at, cols)),
            Operand(buf, (rows, k, ld, rows * ld, scales_at + scale_bytes, cols)))


def to_operands(x: torch.Tensor, mode="floor", rows: bool = True, cols: bool = True, pitch_pad: int = 0):
    """GEMM operands of x [R, C] (bf16; float32 is rounded to bf16 in the cast), any R: (row-wise `Operand` or None, column-wise `Operand` or None), each
    with its contraction rounded up to a multiple of 128 by zero codes (`mx_cast_pad`) -- codes
    [R, C up to 128] and [C, R up to 128], `pitch_pad` as for `to_mx_dim0_dim1`.  Both operands of a
    product come from here, so that they agree on the rounded contraction."""
    C = x.shape[1]
    x = _operand_input(x, f32_ok=True)
    (R, Cx), dev, pad = x.shape, x.device, _pitch_ok(pitch_pad)
    r = _new_operand(R, C, pad, dev) if rows else None
    c = _new_operand(Cx, R, pad, dev) if cols else None
    _call("mx_cast_pad", "cast_dim0_dim1" if rows and cols else "cast_dim0" if rows else "cast_dim1", dev,
          x.data_ptr(), x.dtype == torch.float32, R, Cx, x.stride(0),
          *((r.codes_ptr, r.ld, r.scales_ptr) if rows else (None, 0, None)),
          *((c.codes_ptr, c.ld, c.scales_ptr) if cols else (None, 0, None)), _mode(mode), _stream(x))
    if cols and Cx != C:
        c = c.first_rows(C)
    return r, c


CAST_LIST = 8  # matrices or stacks that one launch casts


class CastList:
    """Both forms of up to `CAST_LIST` tensors, written by one launch: `add` makes the outputs, `launch`
    fills them.

    The operands of a product are independent and mostly small, and a launch of its own for each has the
    chip fill and drain every time."""

    def __init__(self, mode="floor"):
        self._mode, self._table, self._held, self._device = _mode(mode), [], [], None

    def _entry(self, x, G, R, C, ldx, *outputs):
        if len(self._held) == CAST_LIST:
            raise _lib.MXLibraryError(f"a cast list holds {CAST_LIST} tensors")
        if self._device is None:
            self._device = x.device
        elif x.device != self._device:
            raise _lib.MXLibraryError("a cast list is of one device")
        self._held.append(x)
        self._table += (x.data_ptr(), x.dtype == torch.float32, G, R, C, ldx, *outputs)

    def add(self, x: torch.Tensor, pitch_pad: int = 0):
        """A matrix, bf16 or float32: (row-wise, column-wise) as `to_operands` gives them."""
        pad, cols = _pitch_ok(pitch_pad), x.shape[1]
        x = _operand_input(x, f32_ok=True)
        R, C = x.shape
        r, c = _new_operand(R, cols, pad, x.device), _new_operand(C, R, pad, x.device)
        self._entry(x, 1, R, C, x.stride(0), r.codes_ptr, r.ld, r.scales_ptr, c.codes_ptr, c.ld, c.scales_ptr)
        return r, c if C == cols else c.first_rows(cols)

    def add_stack(self, x: torch.Tensor):
        """A contiguous stack [G, R, C], R and C multiples of 128: (row-wise, column-wise) as
        `to_mx_dim0_dim1_batched` gives them; float32 is rounded to bf16 in the cast."""
        if x.dim() != 3 or x.dtype not in (torch.bfloat16, torch.float32) or not x.is_cuda:
            raise TypeError("expected a 3-D bf16 or float32 GPU tensor")
        G, R, C = x.shape
        if R % WHOLE_BLOCK or C % WHOLE_BLOCK or not x.is_contiguous():
            raise ValueError(f"expected a contiguous stack of whole 128 x 128 tiles, got {tuple(x.shape)}")
        x = x if x.data_ptr() % 16 == 0 else x.clone()
        new = lambda *shape: torch.empty(shape, dtype=torch.uint8, device=x.device)
        r = MXData(new(G, R, C), new(G * R * C // BLOCK), MX_SCALES_MFMA)
        c = MXData(new(G, C, R), new(G * R * C // BLOCK), MX_SCALES_MFMA)
        self._entry(x, G, R, C, C, r.codes.data_ptr(), C, r.scales.data_ptr(), c.codes.data_ptr(), R, c.scales.data_ptr())
        return r, c

    def launch(self) -> None:
        if self._held:
            _call("mx_cast_pad_many", "cast_dim0_dim1", self._device, len(self._held), _host_table(self._table, c_int64),
                  self._mode, _stream(self._held[0]))
            self._held, self._table, self._device = [], [], None


def swiglu_to_operands(a: torch.Tensor, b: torch.Tensor, mode="floor", cols: bool = True, pitch_pad: int = 0):
    """`to_operands` of silu(a) * b (see `swiglu_to_mx_dim0_dim1`), any number of rows."""
    a, b = _operand_input(a), _operand_input(b)
    if a.shape != b.shape:
        raise ValueError(f"shape mismatch: {tuple(a.shape)} vs {tuple(b.shape)}")
    (R, C), pad, dev = a.shape, _pitch_ok(pitch_pad), a.device
    r = _new_operand(R, C, pad, dev)
    c = _new_operand(C, R, pad, dev) if cols else None
    _call("mx_swiglu_cast_pad", "swiglu_cast_dim0_dim1", dev, a.data_ptr(), b.data_ptr(), R, C, a.stride(0), b.stride(0),
          r.codes_ptr, r.ld, r.scales_ptr, *((c.codes_ptr, c.ld, c.scales_ptr) if cols else (None, 0, None)),
          _mode(mode), _stream(a))
    return r, c


def swiglu_bwd_to_operands(dg: torch.Tensor, a: torch.Tensor, b: torch.Tensor, mode="floor", pitch_pad: int = 0):
    """Both operand forms of both gradients of silu(a) * b (see `swiglu_bwd_to_mx_dim0_dim1`), any number
    of rows: ((da row-wise, da column-wise), (db row-wise, db column-wise))."""
    dg, a, b = _operand_input(dg), _operand_input(a), _operand_input(b)
    if a.shape != b.shape or a.shape != dg.shape:
        raise ValueError(f"shape mismatch: {tuple(dg.shape)}, {tuple(a.shape)}, {tuple(b.shape)}")
    (R, C), pad, dev = a.shape, _pitch_ok(pitch_pad), a.device
    ra, rb = _new_operand_pair(R, C, pad, dev)
    ca, cb = _new_operand_pair(C, R, pad, dev)
    _call("mx_swiglu_bwd_cast_pad", "swiglu_bwd_cast_dim0_dim1", dev, dg.data_ptr(), a.data_ptr(), b.data_ptr(), R, C,
          dg.stride(0), a.stride(0), b.stride(0), ra.codes_ptr, ra.ld, ra.scales_ptr, ca.codes_ptr, ca.ld, ca.scales_ptr,
          _mode(mode), _stream(a))
    return (ra, ca), (rb, cb)


def rms_norm_to_operands(x: torch.Tensor, weight: torch.Tensor, eps: float, mode="floor", pitch_pad: int = 0):
    """(row-wise, column-wise, rstd) of rms_norm(x) * weight (see `rms_norm_to_mx`), any number of rows."""
    x = _operand_input(x)
    if weight.dtype != torch.bfloat16 or weight.shape != (x.shape[1],) or weight.device != x.device:
        raise TypeError("the norm weight must be bf16 [cols] on x's device")
    weight = weight.contiguous()
    (R, C), pad, dev = x.shape, _pitch_ok(pitch_pad), x.device
    r, c = _new_operand(R, C, pad, dev), _new_operand(C, R, pad, dev)
    rstd = torch.empty(R, dtype=torch.float32, device=dev)
    _call("mx_rmsnorm_cast_pad", "rmsnorm_cast_dim0_dim1", dev, x.data_ptr(), weight.data_ptr(), eps, R, C, x.stride(0),
          rstd.data_ptr(), r.codes_ptr, r.ld, r.scales_ptr, c.codes_ptr, c.ld, c.scales_ptr, _mode(mode), _stream(x))
    return r, c, rstd


def to_mx_dim0_dim1(x: torch.Tensor, mode="floor", order: int = MX_SCALES_ROWMAJOR, pitch_pad: int = 0,
                    whole_blocks: bool = False, cast_list: CastList | None = None):
    """Both casts from one read of x; returns (row-wise MXData, column-wise MXData).  With
    `pitch_pad` the rows of both code matrices lie that many bytes further apart than they are
    long (`codes.stride(0)` says so; only `mx_gemm_nt` takes such operands), where the tile kernel
    takes the input; otherwise the codes are dense.  `whole_blocks`: as `to_operands` gives them, with
    `cast_list` by that list's launch."""
    if cast_list is not None:
        if not whole_blocks:
            raise ValueError("a cast list makes whole-block operands")
        return cast_list.add(x, pitch_pad)
    if whole_blocks:
        return to_operands(x, mode, True, True, pitch_pad)
    x = _check_hp(x)
    R, C = x.shape
    if R % BLOCK or C % BLOCK:
        raise ValueError(f"both dims of {tuple(x.shape)} must be multiples of {BLOCK}")
    scales = _alloc_scales(R, C // BLOCK, order, x.device)
    scales_t = _alloc_scales(C, R // BLOCK, order, x.device)
    if pitch_pad and pitch_pad % 16 == 0 and x.data_ptr() % 16 == 0 and C % 8 == 0 and x.stride(0) % 8 == 0:
        codes = torch.empty((R, C + pitch_pad), dtype=torch.uint8, device=x.device)[:, :C]
        codes_t = torch.empty((C, R + pitch_pad), dtype=torch.uint8, device=x.device)[:, :R]
        _call("mx_cast_dim0_dim1_ld", "cast_dim0_dim1", x.device, _ptr(x), R, C, x.stride(0), _ptr(codes),
              codes.stride(0), _ptr(scales), _ptr(codes_t), codes_t.stride(0), _ptr(scales_t), _mode(mode), order,
              _stream(x))
        return MXData(codes, scales, order), MXData(codes_t, scales_t, order)
    codes = torch.empty((R, C), dtype=torch.uint8, device=x.device)
    codes_t = torch.empty((C, R), dtype=torch.uint8, device=x.device)
    _call("mx_cast_dim0_dim1", "cast_dim0_dim1", x.device, _ptr(x), R, C, x.stride(0), _ptr(codes), _ptr(scales), _ptr(codes_t), _ptr(scales_t), _mode(mode), order, _stream(x))
    return MXData(codes, scales, order), MXData(codes_t, scales_t, order)


def to_mx_rows_gathered(x: torch.Tensor, row_index: torch.Tensor, mode="floor",
                        order: int = MX_SCALES_ROWMAJOR, want_cols: bool = True,
                        row_scale: torch.Tensor | None = None):
    """Casts of x[row_index] (index -1, or any index outside x, = a row of zeros) without forming
    the gathered tensor; returns (row-wise MXData, column-wise MXData or None).  `row_scale`
    (float32, one per output row) multiplies the rows in float32, rounded to bf16, first."""
    x = _check_hp(x)
    if row_scale is not None:
        if row_scale.dtype != torch.float32 or row_scale.shape != row_index.shape or row_scale.device != x.device:
            raise TypeError("row_scale must be float32 with one entry per output row on x's device")
        row_scale = row_scale.contiguous()
    if row_index.dtype != torch.int64 or row_index.dim() != 1 or row_index.device != x.device:
        raise TypeError("row_index must be a 1-D int64 tensor on x's device")
    row_index = row_index.contiguous()
    R, C = row_index.numel(), x.shape[1]
    if C % BLOCK or (want_cols and R % BLOCK):
        raise ValueError(f"dims {R}, {C} must be multiples of {BLOCK}")
    codes = torch.empty((R, C), dtype=torch.uint8, device=x.device)
    scales = _alloc_scales(R, C // BLOCK, order, x.device)
    codes_t = scales_t = None
    if want_cols:
        codes_t = torch.empty((C, R), dtype=torch.uint8, device=x.device)
        scales_t = _alloc_scales(C, R // BLOCK, order, x.device)
    _call("mx_cast_rows_gathered", "cast_rows_gathered", x.device, _ptr(x), _ptr(row_index),
          _ptr(row_scale) if row_scale is not None else None, x.shape[0],
          R, C, x.stride(0), _ptr(codes), _ptr(scales), _ptr(codes_t) if want_cols else None,
          _ptr(scales_t) if want_cols else None, _mode(mode), order, _stream(x))
    return MXData(codes, scales, order), (MXData(codes_t, scales_t, order) if want_cols else None)


def moe_route_plan(counts: torch.Tensor, order: torch.Tensor, scores: torch.Tensor | None, top_k: int,
                   alignment: int, length_multiple: int = 1):
    """(padded inclusive group ends int32 [E], token of every padded row int64 [max_len] (-1 =
    padding), score of every padded row float32 [max_len], padded row of every (token, choice)
    pair int64 [pairs]) for tokens-per-expert `counts` and the expert-sorted pair order; the
    padded length is the static bound `plan_length`."""
    if not counts.is_cuda:
        raise _lib.MXLibraryError("moe_route_plan runs on the GPU only")
    dev = counts.device
    c32 = counts.to(torch.int32).contiguous()
    E, R = c32.numel(), order.numel()
    if order.dtype != torch.int64 or order.device != dev:
        raise TypeError("order must be int64 on the counts' device")
    order = order.contiguous()
    if scores is not None:
        if scores.dtype != torch.float32 or scores.numel() != R or scores.device != dev:
            raise TypeError("scores must be float32 with one entry per pair")
        scores = scores.contiguous()
    max_len = plan_length(R, E, alignment, length_multiple)
    offs = torch.empty(E, dtype=torch.int32, device=dev)
    src_row = torch.empty(max_len, dtype=torch.int64, device=dev)
    row_score = torch.empty(max_len, dtype=torch.float32, device=dev)
    pos = torch.full((R,), -1, dtype=torch.int64, device=dev)
    _call("mx_moe_route_plan", "moe_route_plan", dev, _ptr(c32), E, _ptr(order),
          _ptr(scores) if scores is not None else None, R, top_k, max_len, alignment, _ptr(offs),
          _ptr(src_row), _ptr(row_score), _ptr(pos), _stream(counts))
    return offs, src_row, row_score, pos


ROUTE_MAX_EXPERTS = 512
ROUTE_MAX_TOP_K = 16
_ROUTE_TOKENS = 16  # tokens of one workgroup (mx_route_blocks)


GATE_MAX_EXPERTS = 128


def gate_shape_ok(tokens: int, experts: int, dim: int) -> bool:
    """The gate kernels' shapes: at most 128 experts in whole eights, `dim` in whole 128s."""
    return tokens > 0 and 8 <= experts <= GATE_MAX_EXPERTS and experts % 8 == 0 and dim >= 128 and dim % 128 == 0


def _gate_rows(t: torch.Tensor) -> torch.Tensor:
    """bf16 [rows, dim] on the GPU with 16-byte aligned rows (a copy where they are not)."""
    t = _check_hp(t)
    if t.stride(0) % 8 or t.data_ptr() % 16 or t.stride(0) < t.shape[1]:
        return t.clone(memory_format=torch.contiguous_format)
    return t


def _gate_check(x: torch.Tensor, experts: int, *others: torch.Tensor) -> None:
    if not gate_shape_ok(x.shape[0], experts, x.shape[1]):
        raise ValueError(f"no gate kernel for {x.shape[0]} x {x.shape[1]}, {experts} experts")
    if any(o.device != x.device for o in others):
        raise ValueError("operands on different devices")


def gate_logits(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """float32 [tokens, experts] = x w^T for bf16 x [tokens, dim], w [experts, dim], as a float32 matmul."""
    if _single(x) and (out := _lib.blocks().gate_logits(x, w)) is not None:
        return out
    x, w = _gate_rows(x), _gate_rows(w)
    if w.shape[1] != x.shape[1]:
        raise ValueError(f"column mismatch: {x.shape[1]} vs {w.shape[1]}")
    _gate_check(x, w.shape[0], w)
    (T, D), E = x.shape, w.shape[0]
    logits = torch.empty((T, E), dtype=torch.float32, device=x.device)
    _call("mx_gate_logits", "gate_logits", x.device, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), T, E, D,
          logits.data_ptr(), _stream(x))
    return logits


def _gate_grad(dlogits: torch.Tensor, T: int, E: int) -> torch.Tensor:
    if dlogits.dtype != torch.float32 or dlogits.shape != (T, E):
        raise TypeError(f"dlogits must be float32 [{T}, {E}]")
    dlogits = dlogits.contiguous()
    return dlogits.clone() if dlogits.data_ptr() % 16 else dlogits


def gate_dx(dlogits: torch.Tensor, w: torch.Tensor, base: torch.Tensor | None = None) -> torch.Tensor:
    """bf16 [tokens, dim] = dlogits w, summed in float32; with `base` (bf16 of that shape) the bf16 sum of both."""
    if _single(w) and (out := _lib.blocks().gate_dx(dlogits, w, base)) is not None:
        return out
    w = _gate_rows(w)
    (E, D), T = w.shape, dlogits.shape[0]
    dlogits = _gate_grad(dlogits, T, E)
    if base is not None:
        base = _gate_rows(base)
        if base.shape != (T, D):
            raise ValueError(f"base must be [{T}, {D}]")
    out = torch.empty((T, D), dtype=torch.bfloat16, device=w.device)
    _gate_check(out, E, w, dlogits, *(() if base is None else (base,)))
    _call("mx_gate_dx", "gate_dx", w.device, dlogits.data_ptr(), w.data_ptr(), w.stride(0),
          None if base is None else base.data_ptr(), 0 if base is None else base.stride(0), T, E, D, out.data_ptr(),
          _stream(w))
    return out


def gate_dw(dlogits: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """bf16 [experts, dim] = dlogits^T x, summed in float32."""
    if _single(x) and (out := _lib.blocks().gate_dw(dlogits, x)) is not None:
        return out
    x = _gate_rows(x)
    (T, D), E = x.shape, dlogits.shape[1]
    dlogits = _gate_grad(dlogits, T, E)
    _gate_check(x, E, dlogits)
    work = torch.empty(_lib.load().mx_gate_dw_workspace(T, E, D), dtype=torch.uint8, device=x.device)
    out = torch.empty((E, D), dtype=torch.bfloat16, device=x.device)
    _call("mx_gate_dw", "gate_dw", x.device, dlogits.data_ptr(), x.data_ptr(), x.stride(0), T, E, D, work.data_ptr(),
          out.data_ptr(), _stream(x))
    return out


def route_topk(logits: torch.Tensor, bias: torch.Tensor | None, top_k: int, softmax: bool, norm: bool, scale: float):
    """Token-choice routing from float32 logits [T, E] (`mx_route_topk`): (weights of the chosen experts
    float32 [T, k], the experts int64 [T, k] in falling order of score + bias, pairs per expert int64
    [E], and what `route_fill` needs to place the pairs)."""
    if _single(logits) and (out := _lib.blocks().route_topk(logits, bias, top_k, bool(softmax), bool(norm), scale)) is not None:
        return out
    T, E = logits.shape
    dev = logits.device
    if logits.dtype != torch.float32 or not logits.is_cuda:
        raise TypeError("expected float32 logits on the GPU")
    logits = logits.contiguous()
    if bias is not None:
        if bias.dtype != torch.float32 or bias.shape != (E,) or bias.device != dev:
            raise TypeError("the routing bias must be float32 [experts] on the logits' device")
        bias = bias.contiguous()
    top = torch.empty((T, top_k), dtype=torch.float32, device=dev)
    selected = torch.empty((T, top_k), dtype=torch.int64, device=dev)
    counts = torch.empty(E, dtype=torch.int64, device=dev)
    block_counts = torch.empty(E * -(-T // _ROUTE_TOKENS), dtype=torch.int32, device=dev)
    _call("mx_route_topk", "route_topk", dev, _ptr(logits), T, E, None if bias is None else _ptr(bias), top_k,
          int(softmax), int(norm), scale, _ptr(top), _ptr(selected), _ptr(counts), _ptr(block_counts), _stream(logits))
    return top, selected, counts, block_counts


def route_topk_bwd(logits: torch.Tensor, selected: torch.Tensor, dtop: torch.Tensor, softmax: bool, norm: bool,
                   scale: float) -> torch.Tensor:
    """Gradient of `route_topk`'s weights with respect to the logits, float32 [T, E]."""
    if _single(logits):
        out = _lib.blocks().route_topk_bwd(logits, selected, dtop, bool(softmax), bool(norm), scale)
        if out is not None:
            return out
    T, E = logits.shape
    if selected.device != logits.device or dtop.device != logits.device:
        raise ValueError("operands on different devices")
    logits, selected, dtop = logits.contiguous(), selected.contiguous(), dtop.contiguous()
    out = torch.empty((T, E), dtype=torch.float32, device=logits.device)
    _call("mx_route_topk_bwd", "route_topk_bwd", logits.device, _ptr(logits), T, E, selected.shape[1], int(softmax),
          int(norm), scale, _ptr(selected), _ptr(dtop), _ptr(out), _stream(logits))
    return out


def plan_length(pairs, experts: int, alignment: int, length_multiple: int = 1):
    """Rows of the padded layout of `pairs` rows in groups aligned to `alignment`: a static bound, in multiples of
    `length_multiple`, and one more where its 128s (the persistent kernel's layout) come to whole 512s, but for the
    powers of two below 65536.  The column-wise codes have rows of this many bytes, and a weight gradient reads 128-byte
    pieces of 512 of them at a time: where rows lie a whole number of KB apart those fall on few channels of the L2 (128
    experts 768 x 2048 and 2048 x 768 over 131 072 pairs: 265 and 267 us with 135168 rows = 33 x 4096; with 1024 more 251
    and 256, 512 more 240 and 245, 256 more 238 and 240, 128 more 235 and 240).  Rows a power of two apart spread better,
    and the additional row of tiles opens another round of launches that fill theirs: below 65536 that costs more.
    All GPU work of the experts forward and backward, 1536 to 135680 rows, five sets of experts (8 to 128 of 1024 x 512 ..
    2048 x 1024), time without the additional rows over the time with them:
        odd 512s              0.99 .. 1.03, about 1.00 below 65536      odd 1024s, 2048s   0.99 .. 1.04
        multiples of 3 x 4096  1.00 .. 1.08 (24576, 32 experts of 2048 x 768: 776 and 731 us)
        2048                  1.00 .. 1.01                              4096               0.96 .. 1.00
        8192                  0.94 .. 1.01                              16384              0.96 .. 1.00
        32768                 0.97 .. 1.02                              65536, 131072      1.00 .. 1.04
    (Without a branch on the length, which may be symbolic.)"""
    step = max(alignment, length_multiple)
    if step % alignment:
        raise ValueError("length_multiple must be a multiple of the alignment")
    rows = -(-(pairs + alignment * experts) // step) * step
    if length_multiple != WHOLE_BLOCK:
        return rows
    whole_512s, least = (3 - rows // step % 4) // 3, min if type(rows) is int else torch.sym_min
    return rows + step * whole_512s * least(1, (rows & (rows - 1)) + rows // 65536)


def route_fill(selected: torch.Tensor, scores: torch.Tensor, counts: torch.Tensor, block_counts: torch.Tensor,
               alignment: int, length_multiple: int = 1):
    """The plan of `moe_route_plan` (same outputs, pos [T, k]) from `route_topk`'s, without a sort."""
    T, k = selected.shape
    E, dev = counts.numel(), selected.device
    max_len = plan_length(T * k, E, alignment, length_multiple)
    scores = scores.contiguous()
    offs = torch.empty(E, dtype=torch.int32, device=dev)
    src_row = torch.empty(max_len, dtype=torch.int64, device=dev)
    row_score = torch.empty(max_len, dtype=torch.float32, device=dev)
    pos = torch.empty((T, k), dtype=torch.int64, device=dev)
    _call("mx_route_fill", "route_fill", dev, _ptr(selected), _ptr(scores), T, k, E, _ptr(block_counts), _ptr(counts),
          max_len, alignment, _ptr(offs), _ptr(src_row), _ptr(row_score), _ptr(pos), _stream(selected))
    return offs, src_row, row_score, pos


def moe_combine(y: torch.Tensor, pos: torch.Tensor, weights: torch.Tensor | None = None,
                y2: torch.Tensor | None = None) -> torch.Tensor:
    """out[t] = sum_j weights[t, j] * y[pos[t, j]] (float32, j in order; plain sum without
    weights), bf16 [tokens, cols].  y: bf16 [rows, cols]; pos: int64 [tokens, top_k]; a position
    outside y contributes nothing.  With y2 (y's shape) the rows are bf16(y + y2)."""
    y = _check_hp(y)
    if y2 is not None:
        y2 = _check_hp(y2)
        if y2.shape != y.shape or y2.stride(0) != y.stride(0):
            raise ValueError("y2 must have y's shape and row stride")
    if pos.dtype != torch.int64 or pos.dim() != 2 or pos.device != y.device:
        raise TypeError("pos must be a 2-D int64 tensor on y's device")
    pos = pos.contiguous()
    T, k = pos.shape
    if weights is not None:
        if weights.dtype != torch.float32 or weights.shape != pos.shape or weights.device != y.device:
            raise TypeError("weights must be float32 of pos's shape on y's device")
        weights = weights.contiguous()
    out = torch.empty((T, y.shape[1]), dtype=torch.bfloat16, device=y.device)
    _call("mx_moe_combine", "moe_combine", y.device, _ptr(y), _ptr(y2) if y2 is not None else None,
          y.shape[0], y.stride(0), _ptr(pos),
          _ptr(weights) if weights is not None else None, T, k, y.shape[1], _ptr(out), out.stride(0),
          _stream(y))
    return out


MOE_DOT_MAX_TOP_K = 16  # choices per token whose dot products one wave keeps


def moe_combine_dot(y: torch.Tensor, pos: torch.Tensor, x: torch.Tensor, weights: torch.Tensor | None = None,
                    combine: bool = True):
    """(`moe_combine(y, pos, weights)`, <y[pos[t, j]], x[t]> as float32 [tokens, top_k]) from one read of
    y; x: bf16 [tokens, cols].  Without `combine` the first is None.  At most MOE_DOT_MAX_TOP_K choices."""
    y, x = _check_hp(y), _check_hp(x)
    if pos.dtype != torch.int64 or pos.dim() != 2 or pos.device != y.device or x.device != y.device:
        raise TypeError("pos must be a 2-D int64 tensor, and x a tensor, on y's device")
    T, k = pos.shape
    if x.shape != (T, y.shape[1]):
        raise ValueError(f"x must be [{T}, {y.shape[1]}], got {tuple(x.shape)}")
    pos = pos.contiguous()
    if weights is not None:
        if weights.dtype != torch.float32 or weights.shape != pos.shape or weights.device != y.device:
            raise TypeError("weights must be float32 of pos's shape on y's device")
        weights = weights.contiguous()
    out = torch.empty((T, y.shape[1]), dtype=torch.bfloat16, device=y.device) if combine else None
    dots = torch.empty((T, k), dtype=torch.float32, device=y.device)
    _call("mx_moe_combine_dot", "moe_combine_dot", y.device, _ptr(y), y.shape[0], y.stride(0), _ptr(pos),
          _ptr(weights) if weights is not None else None, _ptr(x), x.stride(0), T, k, y.shape[1],
          _ptr(out) if combine else None, out.stride(0) if combine else 0, _ptr(dots), _stream(y))
    return out, dots


def moe_row_dot(a: torch.Tensor, ia: torch.Tensor, b: torch.Tensor, ib: torch.Tensor,
                a2: torch.Tensor | None = None) -> torch.Tensor:
    """out[i] = <a[ia[i]], b[ib[i]]> in float32 for bf16 matrices a, b with equal column counts;
    an index outside its matrix gives 0.  With a2 (a's shape) a's rows are bf16(a + a2)."""
    a, b = _check_hp(a), _check_hp(b)
    if a2 is not None:
        a2 = _check_hp(a2)
        if a2.shape != a.shape or a2.stride(0) != a.stride(0):
            raise ValueError("a2 must have a's shape and row stride")
    if a.shape[1] != b.shape[1]:
        raise ValueError(f"column mismatch: {a.shape[1]} vs {b.shape[1]}")
    for idx in (ia, ib):
        if idx.dtype != torch.int64 or idx.device != a.device:
            raise TypeError("indices must be int64 on the matrices' device")
    if ia.shape != ib.shape:
        raise ValueError("index shapes differ")
    ia_c, ib_c = ia.contiguous().view(-1), ib.contiguous().view(-1)
    out = torch.empty(ia.shape, dtype=torch.float32, device=a.device)
    _call("mx_moe_row_dot", "moe_row_dot", a.device, _ptr(a), _ptr(a2) if a2 is not None else None,
          a.shape[0], a.stride(0), _ptr(ia_c), _ptr(b),
          b.shape[0], b.stride(0), _ptr(ib_c), ia_c.numel(), a.shape[1], _ptr(out), _stream(a))
    return out


def mx_dequant(d: MXData, out: torch.Tensor | None = None) -> torch.Tensor:
    """bf16 [rows, cols] values of row-wise MXFP8 data (codes [rows, cols], blocks along cols)."""
    codes = d.codes
    if codes.dtype != torch.uint8 or codes.dim() != 2 or not codes.is_cuda:
        raise TypeError("expected 2-D uint8 codes on the GPU")
    codes = codes.contiguous()
    rows, cols = codes.shape
    if cols % BLOCK:
        raise ValueError(f"cols {cols} is not a multiple of {BLOCK}")
    if out is None:
        out = torch.empty((rows, cols), dtype=torch.bfloat16, device=codes.device)
    else:
        _wrote(out)
    scales = d.scales.contiguous()
    _call("mx_dequant", "dequant", codes.device, _ptr(codes), _ptr(scales), rows, cols, d.scale_order,
          _ptr(out), out.stride(0), _stream(codes))
    return out


def _host_table(values, kind):
    """Host array of 64-bit (pointers, counts) or 32-bit entries for the library's list entry points."""
    return (kind * len(values))(*values)


def to_mx_rows_many(tensors, mode="floor"):
    """Row-wise `MXData` (codes of the tensor's shape, row-major scales [..., last/32]) of every tensor in the
    list -- bf16 or float32, one device, last dimension a multiple of 32 -- in one launch."""
    tensors = list(tensors)
    if tensors and _single(tensors[0]) and (out := _lib.blocks().rows_many(tensors, _mode(mode))) is not None:
        return [MXData(codes, scales, MX_SCALES_ROWMAJOR) for codes, scales in out]
    tensors = [t.contiguous() if t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)
               for t in tensors]
    if not tensors:
        return []
    dev = tensors[0].device
    out = []
    for t in tensors:
        if not t.is_cuda or t.device != dev:
            raise _lib.MXLibraryError("the MXFP8 kernels run on the GPU only, one device per call")
        if t.dtype not in (torch.bfloat16, torch.float32):
            raise TypeError(f"expected bfloat16 or float32, got {t.dtype}")
        if t.shape[-1] % BLOCK:
            raise ValueError(f"last dim {t.shape[-1]} is not a multiple of {BLOCK}")
        out.append(MXData(torch.empty(t.shape, dtype=torch.uint8, device=dev),
                          torch.empty((*t.shape[:-1], t.shape[-1] // BLOCK), dtype=torch.uint8, device=dev),
                          MX_SCALES_ROWMAJOR))
    _call("mx_cast_rows_many", "cast_rows_many", dev, len(out), _host_table([_ptr(t) for t in tensors], c_int64),
          _host_table([t.numel() for t in tensors], c_int64),
          _host_table([int(t.dtype == torch.float32) for t in tensors], c_int32),
          _host_table([_ptr(q.codes) for q in out], c_int64), _host_table([_ptr(q.scales) for q in out], c_int64),
          _mode(mode), _stream(tensors[0]))
    return out


def mx_dequant_many(data) -> list:
    """bf16 values of every row-wise `MXData` with row-major scales in the list (any shapes), in one launch."""
    data = list(data)
    if data and _single(data[0].codes) and all(q.scale_order == MX_SCALES_ROWMAJOR for q in data):
        out = _lib.blocks().dequant_many([q.codes for q in data], [q.scales for q in data])
        if out is not None:
            return out
    data = [MXData(q.codes.contiguous(), q.scales.contiguous(), q.scale_order) for q in data]
    if not data:
        return []
    dev = data[0].codes.device
    for q in data:
        if q.codes.dtype != torch.uint8 or not q.codes.is_cuda or q.codes.device != dev:
            raise TypeError("expected uint8 codes on one GPU")
        if (q.scale_order != MX_SCALES_ROWMAJOR or q.codes.shape[-1] % BLOCK
                or q.scales.numel() * BLOCK != q.codes.numel()):
            raise ValueError("expected row-major scales, one per 32 codes of a row")
    out = [torch.empty(q.codes.shape, dtype=torch.bfloat16, device=dev) for q in data]
    _call("mx_dequant_many", "dequant_many", dev, len(out), _host_table([_ptr(q.codes) for q in data], c_int64),
          _host_table([_ptr(q.scales) for q in data], c_int64), _host_table([q.codes.numel() for q in data], c_int64),
          _host_table([_ptr(t) for t in out], c_int64), _stream(out[0]))
    return out


def _logprob_splits(rows: int, vocab: int) -> int:
    """Parts that the forward cuts every row of logits into: enough for one workgroup per CU, none
    of less than 12 288 logits (a workgroup asks for 16 384 at once; smaller parts cost more in
    reductions than they spread).  Vocabulary 151 936, uncut against so cut: 16 rows 13.4 -> 6.7 us,
    64 rows 16.8 -> 9.2, 200 rows 17.5 -> 16.2; 300 rows 23.6 -> 20.2 at best, 457 rows 24.6 -> 27.0."""
    return max(1, min(-(-256 // rows), vocab // 12288))


def token_logprob_fwd(logits: torch.Tensor, target: torch.Tensor):
    """(log-probability of target[r] under softmax(logits[r]), log-sum-exp of row r), float32
    [rows], from bf16 logits [rows, vocab] read once."""
    if logits.dim() == 2 and logits.shape[0] and _single(logits):
        out = _lib.blocks().token_logprob_fwd(logits, target, _logprob_splits(*logits.shape))
        if out is not None:
            return out
    logits = _check_hp(logits)
    if target.dtype != torch.int64 or target.shape != (logits.shape[0],) or target.device != logits.device:
        raise TypeError("target must be int64 [rows] on the logits' device")
    target = target.contiguous()
    (rows, vocab), ld = logits.shape, logits.stride(0)
    if ld < vocab:  # rows that overlap
        logits, ld = logits.clone(memory_format=torch.contiguous_format), vocab
    lp = torch.empty(rows, dtype=torch.float32, device=logits.device)
    lse = torch.empty(rows, dtype=torch.float32, device=logits.device)
    splits = _logprob_splits(rows, vocab) if rows else 1
    partial = torch.empty(2 * rows * splits, dtype=torch.float32, device=logits.device) if splits > 1 else None
    _call("mx_token_logprob_fwd_split", "token_logprob_fwd", logits.device, _ptr(logits), rows, vocab,
          ld, _ptr(target), _ptr(lp), _ptr(lse), splits, _ptr(partial) if splits > 1 else None,
          _stream(logits))
    return lp, lse


def token_logprob_bwd(logits: torch.Tensor, target: torch.Tensor, lse: torch.Tensor,
                      grad_logprob: torch.Tensor) -> torch.Tensor:
    """Gradient of `token_logprob_fwd`'s first output with respect to the logits, bf16."""
    if _single(logits) and (out := _lib.blocks().token_logprob_bwd(logits, target, lse, grad_logprob)) is not None:
        return out
    logits = _check_hp(logits)
    (rows, vocab), ld = logits.shape, logits.stride(0)
    if ld < vocab:
        logits, ld = logits.clone(memory_format=torch.contiguous_format), vocab
    g = grad_logprob.to(torch.float32).contiguous()
    lse, target = lse.contiguous(), target.contiguous()
    out = torch.empty((rows, -(-vocab // 8) * 8), dtype=torch.bfloat16, device=logits.device)
    if vocab % 8:
        out = out[:, :vocab]
    step, ldo = 65535, out.stride(0)  # (one grid row per token row)
    for lo in range(0, rows, step):
        _call("mx_token_logprob_bwd_any", "token_logprob_bwd", logits.device, _ptr(logits) + 2 * lo * ld,
              min(step, rows - lo), vocab, ld, _ptr(target) + 8 * lo, _ptr(lse) + 4 * lo, _ptr(g) + 4 * lo,
              _ptr(out) + 2 * lo * ldo, ldo, _stream(logits))
    return out


def rms_norm_to_mx(x: torch.Tensor, weight: torch.Tensor, eps: float, mode="floor",
                   order: int = MX_SCALES_ROWMAJOR, want_y: bool = False, pitch_pad: int = 0):
    """Both casts of y = rms_norm(x) * weight (float32 arithmetic, one rounding to bf16) without
    y passing through memory; returns (row-wise MXData, column-wise MXData, rstd float32 [rows],
    y or None).  `pitch_pad`: as for `to_mx_dim0_dim1`."""
    x = _check_hp(x)
    if weight.dtype != torch.bfloat16 or weight.shape != (x.shape[1],) or weight.device != x.device:
        raise TypeError("the norm weight must be bf16 [cols] on x's device")
    weight = weight.contiguous()
    R, C = x.shape
    if R % BLOCK or C % BLOCK:
        raise ValueError(f"both dims of {tuple(x.shape)} must be multiples of {BLOCK}")
    pad = _pitch_ok(pitch_pad)
    codes = _code_rows(R, C, pad, x.device)
    scales = _alloc_scales(R, C // BLOCK, order, x.device)
    codes_t = _code_rows(C, R, pad, x.device)
    scales_t = _alloc_scales(C, R // BLOCK, order, x.device)
    rstd = torch.empty(R, dtype=torch.float32, device=x.device)
    y = torch.empty((R, C), dtype=torch.bfloat16, device=x.device) if want_y else None
    _call("mx_rmsnorm_cast_dim0_dim1_ld", "rmsnorm_cast_dim0_dim1", x.device, _ptr(x), _ptr(weight),
          eps, R, C, x.stride(0), _ptr(rstd), _ptr(y) if y is not None else None,
          _ptr(codes), codes.stride(0), _ptr(scales), _ptr(codes_t), codes_t.stride(0), _ptr(scales_t),
          _mode(mode), order, _stream(x))
    return MXData(codes, scales, order), MXData(codes_t, scales_t, order), rstd, y


def swiglu_to_mx_dim0_dim1(a: torch.Tensor, b: torch.Tensor, mode="floor",
                           order: int = MX_SCALES_ROWMAJOR, want_g: bool = False, pitch_pad: int = 0):
    """Both casts of g = silu(a) * b (bf16, every step rounded to bf16) without g passing through
    memory; returns (row-wise MXData, column-wise MXData, g or None).  `pitch_pad`: as for
    `to_mx_dim0_dim1`."""
    a, b = _check_hp(a), _check_hp(b)
    if a.shape != b.shape:
        raise ValueError(f"shape mismatch: {tuple(a.shape)} vs {tuple(b.shape)}")
    R, C = a.shape
    if R % BLOCK or C % BLOCK:
        raise ValueError(f"both dims of {tuple(a.shape)} must be multiples of {BLOCK}")
    pad = _pitch_ok(pitch_pad)
    codes = _code_rows(R, C, pad, a.device)
    scales = _alloc_scales(R, C // BLOCK, order, a.device)
    codes_t = _code_rows(C, R, pad, a.device)
    scales_t = _alloc_scales(C, R // BLOCK, order, a.device)
    g = torch.empty((R, C), dtype=torch.bfloat16, device=a.device) if want_g else None
    _call("mx_swiglu_cast_dim0_dim1_ld", "swiglu_cast_dim0_dim1", a.device, _ptr(a), _ptr(b), R, C,
          a.stride(0), b.stride(0), _ptr(codes), codes.stride(0), _ptr(scales), _ptr(codes_t), codes_t.stride(0),
          _ptr(scales_t), _ptr(g) if g is not None else None, _mode(mode), order, _stream(a))
    return MXData(codes, scales, order), MXData(codes_t, scales_t, order), g


def _scale_count(rows: int, nblk: int, order: int) -> int:
    return mfma_scale_bytes(rows, nblk) if order == MX_SCALES_MFMA else rows * nblk


def swiglu_bwd_to_mx_dim0_dim1(dg: torch.Tensor, a: torch.Tensor, b: torch.Tensor, mode="floor",
                               order: int = MX_SCALES_ROWMAJOR, want_grads: bool = False, pitch_pad: int = 0):
    """Backward of g = silu(a) * b with both casts of each gradient from one pass over dg, a, b.

    Returns ((da row-wise, da column-wise), (db row-wise, db column-wise), stacked bf16 [2, R, C]
    gradients or None).  The two row-wise (column-wise) results are the halves of one buffer.
    `pitch_pad`: as for `to_mx_dim0_dim1`."""
    dg, a, b = _check_hp(dg), _check_hp(a), _check_hp(b)
    if a.shape != b.shape or a.shape != dg.shape:
        raise ValueError(f"shape mismatch: {tuple(dg.shape)}, {tuple(a.shape)}, {tuple(b.shape)}")
    R, C = a.shape
    if R % BLOCK or C % BLOCK:
        raise ValueError(f"both dims of {tuple(a.shape)} must be multiples of {BLOCK}")
    dev = a.device
    n_s, n_st = _scale_count(R, C // BLOCK, order), _scale_count(C, R // BLOCK, order)
    pad = _pitch_ok(pitch_pad)
    codes = _code_rows(R, C, pad, dev, stack=2)
    codes_t = _code_rows(C, R, pad, dev, stack=2)
    scales = torch.empty(2 * n_s, dtype=torch.uint8, device=dev)
    scales_t = torch.empty(2 * n_st, dtype=torch.uint8, device=dev)
    dab = torch.empty((2, R, C), dtype=torch.bfloat16, device=dev) if want_grads else None
    _call("mx_swiglu_bwd_cast_dim0_dim1_ld", "swiglu_bwd_cast_dim0_dim1", dev, _ptr(dg), _ptr(a), _ptr(b),
          R, C, dg.stride(0), a.stride(0), b.stride(0), _ptr(codes), codes.stride(1), _ptr(scales), _ptr(codes_t),
          codes_t.stride(1), _ptr(scales_t), _ptr(dab) if dab is not None else None, _mode(mode), order, _stream(a))

    def half(i):
        s, st = scales[i * n_s:(i + 1) * n_s], scales_t[i * n_st:(i + 1) * n_st]
        if order == MX_SCALES_ROWMAJOR:
            s, st = s.view(R, C // BLOCK), st.view(C, R // BLOCK)
        return MXData(codes[i], s, order), MXData(codes_t[i], st, order)

    return half(0), half(1), dab


def scale_layout(scales: torch.Tensor) -> torch.Tensor:
    """Row-major [rows, nblk] scales -> flat buffer in MFMA order."""
    rows, nblk = scales.shape
    scales = scales.contiguous()
    out = torch.empty(mfma_scale_bytes(rows, nblk), dtype=torch.uint8, device=scales.device)
    _call("mx_scale_layout", "scale_layout", scales.device, _ptr(scales), rows, nblk, _ptr(out), _stream(scales))
    return out


def scale_unlayout(laid: torch.Tensor, rows: int, nblk: int) -> torch.Tensor:
    out = torch.empty((rows, nblk), dtype=torch.uint8, device=laid.device)
    _call("mx_scale_unlayout", "scale_unlayout", laid.device, _ptr(laid), rows, nblk, _ptr(out), _stream(laid))
    return out


def _as_mfma(d: MXData) -> torch.Tensor:
    return d.scales if d.scale_order == MX_SCALES_MFMA else scale_layout(d.scales)


_gemm_workspace: dict = {}  # (device index, M, N, K, query) -> bytes the library would split with


def _common_pitch(*codes, multiple: int = 128):
    """(the code matrices as the kernels take them, bytes between their rows): unit inner stride
    and one row pitch for all of them, a multiple of `multiple` where it is not the row length
    (copies are made where they differ)."""
    pitch = codes[0].stride(0)
    K = codes[0].shape[1]
    if any(c.stride(1) != 1 or c.stride(0) != pitch for c in codes) or (pitch != K and pitch % multiple):
        codes = tuple(c.contiguous() for c in codes)
        pitch = K
    return codes, pitch


def _split_workspace(device, M: int, N: int, K: int, query: str = "mx_gemm_nt_workspace_bytes"):
    """Float32 partial sums for the shapes whose contraction the library splits (few output tiles, long
    contraction), else None."""
    key = (device.index, M, N, K, query)
    need = _gemm_workspace.get(key)
    if need is None:
        with torch.cuda.device(device):
            need = _gemm_workspace[key] = int(getattr(_lib.load(), query)(M, N, K))
    return torch.empty(need, dtype=torch.uint8, device=device) if need else None


def _gemm_nt_into(a_codes, a_scales, b_codes, b_scales, out):
    M, K = a_codes.shape
    N = b_codes.shape[0]
    (a_codes, b_codes), ldk = _common_pitch(a_codes, b_codes, multiple=16)  # (the tile kernels take any such pitch)
    ws = _split_workspace(out.device, M, N, K)
    if ldk != K:
        _call("mx_gemm_nt_ld", "gemm_nt" if ws is None else "gemm_nt_splitk", out.device, _ptr(a_codes), _ptr(a_scales),
              _ptr(b_codes), _ptr(b_scales), _ptr(out), M, N, K, ldk, out.stride(0),
              None if ws is None else _ptr(ws), 0 if ws is None else ws.numel(), _stream(out))
        return out
    if ws is not None:
        _call("mx_gemm_nt_ws", "gemm_nt_splitk", out.device, _ptr(a_codes), _ptr(a_scales), _ptr(b_codes),
              _ptr(b_scales), _ptr(out), M, N, K, out.stride(0), _ptr(ws), ws.numel(), _stream(out))
        return out
    _call("mx_gemm_nt", "gemm_nt", out.device, _ptr(a_codes), _ptr(a_scales), _ptr(b_codes),
          _ptr(b_scales), _ptr(out), M, N, K, out.stride(0), _stream(out))
    return out


def _operands(*qs) -> bool:
    """All of them `Operand`s with one row pitch the persistent kernel takes: their pointers go to the
    library as they are."""
    ld = getattr(qs[0], "ld", 1)
    if ld % 128:
        return False
    for q in qs:
        if type(q) is not Operand or q.ld != ld:
            return False
    return True


def _depth(q) -> int:
    """The contraction that `q` was cast from: its codes' row length but for the zero fill of an `Operand`."""
    return q.depth if type(q) is Operand else q.codes.shape[-1]


def _gemm_operands(a: Operand, b: Operand, out: torch.Tensor) -> torch.Tensor:
    M, N, K = a.rows, b.rows, a.k
    dev = out.device
    ws = _split_workspace(dev, M, N, K)
    _call("mx_gemm_nt_ld", "gemm_nt" if ws is None else "gemm_nt_splitk", dev, a.codes_ptr, a.scales_ptr, b.codes_ptr,
          b.scales_ptr, out.data_ptr(), M, N, K, a.ld, out.stride(0), None if ws is None else ws.data_ptr(),
          0 if ws is None else ws.numel(), _stream(out))
    return out


def mx_gemm_nt_as(a: MXData, b: MXData, dtype: torch.dtype) -> torch.Tensor:
    """`mx_gemm_nt` in `dtype`: the bf16 result, for float32 written as such by the product itself where it takes
    the shape (147456 x 2048 of float32 gradient: 8 of the 12 bytes an element that the product and a
    conversion move)."""
    if dtype == torch.float32 and _operands(a, b) and not _watched() and a.depth == b.depth:
        M, N, K, dev = a.rows, b.rows, a.k, a.buf.device
        if M > 64 and N > 128 and N % 8 == 0 and max(N * 1024, a.ld * 256) < 1 << 31:
            out = torch.empty((M, N), dtype=torch.float32, device=dev)
            ws = _split_workspace(dev, M, N, K)
            _call("mx_gemm_nt_f32_ld", "gemm_nt" if ws is None else "gemm_nt_splitk", dev, a.codes_ptr, a.scales_ptr,
                  b.codes_ptr, b.scales_ptr, out.data_ptr(), M, N, K, a.ld, N, None if ws is None else ws.data_ptr(),
                  0 if ws is None else ws.numel(), _stream(out))
            return out
    out = mx_gemm_nt(a, b)
    return out if out.dtype == dtype else out.to(dtype)


FEW_ROWS = 32             # rows that `mx_few_rows` takes
FEW_ROWS_VALUES = 65536   # values of x, rows counted in whole 16s, up to which it is chosen
FEW_ROWS_COLUMNS = 16384  # columns of all products, up to which it is chosen


def few_rows_size(rows: int, cols: int, columns: int) -> bool:
    """The sizes of x and of all products' columns that `few_rows_ok` allows."""
    return 0 < rows <= FEW_ROWS and columns <= FEW_ROWS_COLUMNS and (rows + 15 & ~15) * cols <= FEW_ROWS_VALUES


def few_rows_ok(x: torch.Tensor, columns: int) -> bool:
    """`mx_few_rows` runs the products of x with weights of `columns` rows in all: bf16 rows on the GPU in whole
    blocks of 32, few enough of them, and no dispatch mode that would want to see the GEMM.  Every workgroup
    casts all of x, so the line is where that costs more than the launch it saves (a cast of its own: 3.7 us
    on the GPU, about 10 on the host): 16 x 4096 -> 4096 10.7 us in one launch, 3.7 + 7.5 in two; 32 x 2048 ->
    6144 12.6, 3.7 + 7.4; 32 x 14336 -> 4096 42, 3.8 + 27; and where the workgroups outnumber the CUs: 16 x 2048
    -> 16384 14.0 and 14.2, -> 2 x 14336 25.8 and 23.5, -> 151936 123 and 80 us."""
    return (x.dtype == torch.bfloat16 and x.is_cuda and x.dim() == 2 and few_rows_size(*x.shape, columns)
            and x.shape[1] % BLOCK == 0 and x.shape[1] > 0 and x.stride(1) == 1 and not _watched())


def mx_few_rows(x: torch.Tensor, w: Operand, mode="floor", w2: Operand | None = None) -> torch.Tensor:
    """bf16 mx(x) @ deq(w)^T with the cast of x inside the product's launch; with `w2` (of w's shape) both
    products, stacked.  Callers check `few_rows_ok` first."""
    x = _operand_input(x)
    (M, K), N = x.shape, w.rows
    if w.depth != K:
        raise ValueError(f"contraction mismatch: {K} vs {w.depth}")
    if w2 is not None and (w2.rows, w2.depth, w2.ld) != (N, K, w.ld):
        raise ValueError("both weights must have the same shape and pitch")
    out = torch.empty((M, N) if w2 is None else (2, M, N), dtype=torch.bfloat16, device=x.device)
    d = out.data_ptr()
    _call("mx_few_rows", "few_rows", x.device, x.data_ptr(), M, K, x.stride(0), w.codes_ptr, w.scales_ptr,
          *((None, None) if w2 is None else (w2.codes_ptr, w2.scales_ptr)), N, w.ld, d,
          None if w2 is None else d + 2 * M * N, N, _mode(mode), _stream(x))
    return out


def _gemm_nt_op(a_codes, a_scales, b_codes, b_scales):
    out = torch.empty((a_codes.shape[0], b_codes.shape[0]), dtype=torch.bfloat16, device=a_codes.device)
    return _gemm_nt_into(a_codes, a_scales, b_codes, b_scales, out)


def _grouped_2d3d_into(a_codes, a_scales, a_order, b_codes, b_scales, offs, out):
    T, K = a_codes.shape
    G, N, _ = b_codes.shape
    _call("mx_grouped_gemm_2d3d", "grouped_gemm_2d3d", out.device, _ptr(a_codes), _ptr(a_scales),
          _ptr(b_codes), _ptr(b_scales), _ptr(offs), _ptr(out), T, N, K, G, out.stride(0), a_order,
          _stream(out))
    return out


def _grouped_2d3d_op(a_codes, a_scales, a_order, b_codes, b_scales, offs):
    out = torch.empty((a_codes.shape[0], b_codes.shape[1]), dtype=torch.bfloat16, device=a_codes.device)
    return _grouped_2d3d_into(a_codes, a_scales, a_order, b_codes, b_scales, offs, out)


def _grouped_2d3d_rows_out_op(a_codes, a_scales, b_codes, b_scales, offs, out_offs, out_rows, second=None):
    T, K = a_codes.shape
    G, N, _ = b_codes.shape
    out = torch.empty((out_rows, N), dtype=torch.bfloat16, device=a_codes.device)
    extra = [_ptr(t) for t in second] if second is not None else [None] * 4
    _call("mx_grouped_gemm_2d3d_rows_out", "grouped_gemm_2d3d_rows_out", out.device, _ptr(a_codes), _ptr(a_scales),
          _ptr(b_codes), _ptr(b_scales), *extra, _ptr(offs), _ptr(out_offs), _ptr(out), T, out_rows, N, K, G, N,
          _stream(out))
    return out


# The GEMMs whose output a forward pass hands on are also registered with torch's dispatcher, so
# that a per-op activation-checkpoint policy (torch.utils.checkpoint's selective contexts, which
# watch dispatched ops) can name them and keep their outputs instead of running them again in
# the recomputation.  The registered form is only taken while some dispatch mode is active; the
# plain eager path keeps calling the library directly.
_dispatcher_ops = torch.library.Library("torchtitan_amd", "DEF")
_dispatcher_ops.define("mx_gemm_nt(Tensor a_codes, Tensor a_scales, Tensor b_codes, Tensor b_scales) -> Tensor")
_dispatcher_ops.define("mx_grouped_gemm_2d3d(Tensor a_codes, Tensor a_scales, int a_order, Tensor b_codes, "
                       "Tensor b_scales, Tensor offs) -> Tensor")
_dispatcher_ops.define("mx_grouped_gemm_2d3d_rows_out(Tensor a_codes, Tensor a_scales, Tensor b_codes, "
                       "Tensor b_scales, Tensor offs, Tensor out_offs, int out_rows) -> Tensor")
_dispatcher_ops.impl("mx_gemm_nt", _gemm_nt_op, "CUDA")
_dispatcher_ops.impl("mx_grouped_gemm_2d3d", _grouped_2d3d_op, "CUDA")
_dispatcher_ops.impl("mx_grouped_gemm_2d3d_rows_out", _grouped_2d3d_rows_out_op, "CUDA")


_dispatch_depth = getattr(torch._C, "_len_torch_dispatch_stack", None)


def _watched() -> bool:
    """True while some TorchDispatchMode is active (a selective-checkpoint context is one)."""
    return _dispatch_depth is not None and _dispatch_depth() > 0


def _transformed() -> bool:
    """True under a function transform (vmap, jvp, ...) or forward-mode AD: tensors may be wrappers or carry
    tangents, which a library call would not see."""
    return torch._C._functorch.peek_interpreter_stack() is not None or torch.autograd.forward_ad._current_level >= 0


def native_block_ok(x: torch.Tensor, *widths: int) -> bool:
    """A block on x may run its launches from one native call (`_lib.blocks`): a plain tensor, nobody who would
    want to see the single steps (a dispatch mode, a function transform, a kernel timer), and no side narrower
    than a tile of the GEMMs, where other kernels and other combinations of launches run."""
    return (type(x) is torch.Tensor and x.is_cuda and min(widths) > 128 and _timer is None and not _watched()
            and not _transformed())


def op_sac_save_list() -> set:
    """The dispatcher ops of this package whose outputs a per-op activation-checkpoint policy may
    save (the forward GEMMs): add them to the model's save list
    (torchtitan/models/llama3/parallelize.py:44-60) to keep MXFP8 GEMM outputs through the
    recomputation, as the bf16 path keeps its `aten.mm` outputs.  Casts stay recomputed."""
    return {torch.ops.torchtitan_amd.mx_gemm_nt.default,
            torch.ops.torchtitan_amd.mx_grouped_gemm_2d3d.default,
            torch.ops.torchtitan_amd.mx_grouped_gemm_2d3d_rows_out.default}


def mx_gemm_nt(a: MXData, b: MXData, out: torch.Tensor | None = None) -> torch.Tensor:
    """bf16 D[M,N] = deq(a)[M,K] @ deq(b)[N,K]^T with fp32 accumulation."""
    if out is None and _operands(a, b) and not _watched():
        if a.depth != b.depth:
            raise ValueError(f"contraction mismatch: {a.depth} vs {b.depth}")
        return _gemm_operands(a, b, torch.empty((a.rows, b.rows), dtype=torch.bfloat16, device=a.buf.device))
    M, K = a.codes.shape
    N, Kb = b.codes.shape
    if K != Kb or _depth(a) != _depth(b):
        raise ValueError(f"contraction mismatch: {_depth(a)} vs {_depth(b)}")
    sa, sb = _as_mfma(a), _as_mfma(b)
    if out is None:
        if _watched():
            return torch.ops.torchtitan_amd.mx_gemm_nt(a.codes, sa, b.codes, sb)
        return _gemm_nt_op(a.codes, sa, b.codes, sb)
    if out.shape != (M, N) or out.dtype != torch.bfloat16 or out.stride(1) != 1:
        raise ValueError("out must be a bf16 [M, N] tensor with unit inner stride")
    return _gemm_nt_into(a.codes, sa, b.codes, sb, _wrote(out))


def mx_gemm_nt_pair(a: MXData, b: MXData, a2: MXData, b2: MXData) -> torch.Tensor:
    """bf16 deq(a) @ deq(b)^T + deq(a2) @ deq(b2)^T: one GEMM whose output tiles accumulate both
    products before they are rounded and written, where the persistent kernel takes the shape;
    otherwise two GEMMs and a bf16 add.  Few tiles and a long contraction run in slices of K, as
    in `mx_gemm_nt`."""
    if _operands(a, b, a2, b2):
        M, N, K = a.rows, b.rows, a.k
        if a2.rows != M or b2.rows != N or not a.depth == b.depth == a2.depth == b2.depth:
            raise ValueError("both operand sets must have the same shapes")
        if not _persistent_shape(M, N, K):
            return mx_gemm_nt(a, b) + mx_gemm_nt(a2, b2)
        out = torch.empty((M, N), dtype=torch.bfloat16, device=a.buf.device)
        _call_pair((a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr, a2.codes_ptr, a2.scales_ptr, b2.codes_ptr,
                    b2.scales_ptr), M, N, K, a.ld, out)
        return out
    M, K = a.codes.shape
    N = b.codes.shape[0]
    if (a2.codes.shape != (M, K) or b2.codes.shape != (N, K) or b.codes.shape[1] != K
            or not _depth(a) == _depth(b) == _depth(a2) == _depth(b2)):
        raise ValueError("both operand sets must have the same shapes")
    if not _persistent_shape(M, N, K):
        return mx_gemm_nt(a, b) + mx_gemm_nt(a2, b2)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=a.codes.device)
    sa, sb, sa2, sb2 = _as_mfma(a), _as_mfma(b), _as_mfma(a2), _as_mfma(b2)  # kept alive over the launch
    (ac, bc, a2c, b2c), ldk = _common_pitch(a.codes, b.codes, a2.codes, b2.codes)
    _call_pair((_ptr(ac), _ptr(sa), _ptr(bc), _ptr(sb), _ptr(a2c), _ptr(sa2), _ptr(b2c), _ptr(sb2)), M, N, K, ldk, out)
    return out


def _call_pair(args, M: int, N: int, K: int, ldk: int, out: torch.Tensor) -> None:
    ws = _split_workspace(out.device, M, N, K, "mx_gemm_nt_pair_workspace_bytes")
    if ws is None:
        _call("mx_gemm_nt_pair_ld", "gemm_nt_pair", out.device, *args, out.data_ptr(), M, N, K, ldk, N, _stream(out))
    else:
        _call("mx_gemm_nt_pair_ws", "gemm_nt_pair", out.device, *args, out.data_ptr(), M, N, K, ldk, N, ws.data_ptr(),
              ws.numel(), _stream(out))


def _persistent_shape(M: int, N: int, K: int) -> bool:
    return M > 128 and N > 128 and K % 128 == 0 and N % 8 == 0


def mx_gemm_nt_shared_a(a: MXData, b: MXData, b2: MXData) -> torch.Tensor:
    """bf16 [2, M, N]: deq(a) @ deq(b)^T and deq(a) @ deq(b2)^T.  One launch in which the panels
    of `a` are fetched once for both products where the persistent kernel takes the shape (never split
    along K: bit-identical to `mx_gemm_nt` where that is not split either), otherwise two GEMMs."""
    if _operands(a, b, b2) and not _watched():
        M, N, K = a.rows, b.rows, a.k
        if b2.rows != N or not a.depth == b.depth == b2.depth:
            raise ValueError("both second operands must have the same shape")
        out = torch.empty((2, M, N), dtype=torch.bfloat16, device=a.buf.device)
        if not _persistent_shape(M, N, K):
            _gemm_operands(a, b, out[0])
            _gemm_operands(a, b2, out[1])
            return out
        _call("mx_gemm_nt_shared_a_ld", "gemm_nt_shared_a", out.device, a.codes_ptr, a.scales_ptr, b.codes_ptr,
              b.scales_ptr, b2.codes_ptr, b2.scales_ptr, out.data_ptr(), out.data_ptr() + 2 * M * N, M, N, K, a.ld, N,
              _stream(out))
        return out
    M, K = a.codes.shape
    N = b.codes.shape[0]
    if b2.codes.shape != b.codes.shape or b.codes.shape[1] != K or not _depth(a) == _depth(b) == _depth(b2):
        raise ValueError("both second operands must have the same shape")
    if _watched():  # as dispatcher ops, so that a per-op checkpoint policy can keep the outputs
        return torch.stack((mx_gemm_nt(a, b), mx_gemm_nt(a, b2)))
    out = torch.empty((2, M, N), dtype=torch.bfloat16, device=a.codes.device)
    if not _persistent_shape(M, N, K):
        mx_gemm_nt(a, b, out[0])
        mx_gemm_nt(a, b2, out[1])
        return out
    sa, sb, sb2 = _as_mfma(a), _as_mfma(b), _as_mfma(b2)
    (ac, bc, b2c), ldk = _common_pitch(a.codes, b.codes, b2.codes)
    _call("mx_gemm_nt_shared_a_ld", "gemm_nt_shared_a", out.device, _ptr(ac), _ptr(sa), _ptr(bc), _ptr(sb),
          _ptr(b2c), _ptr(sb2), _ptr(out[0]), _ptr(out[1]), M, N, K, ldk, N, _stream(out))
    return out


def mx_gemm_nt_swiglu(a: MXData, b: MXData, b2: MXData, mode="floor", planned: bool = False):
    """The row-wise operand of ``silu(deq(a) @ deq(b)^T) * (deq(a) @ deq(b2)^T)`` in one launch, the same bits as
    `swiglu_to_operands` makes of `mx_gemm_nt_shared_a`'s products; None where those two launches are predicted to be faster
    (`planned`: not asked) or the operands are not for it."""
    if not _operands(a, b, b2) or _watched() or a.depth != b.depth or a.depth != b2.depth or b.rows != b2.rows:
        return None
    M, N = a.rows, b.rows
    if M <= 128 or N <= 128 or N % 8 or not (planned or _lib.load().mx_gemm_nt_swiglu_planned(M, N, a.k)):
        return None
    out = _new_operand(M, N, a.ld - a.k, a.buf.device)
    _call("mx_gemm_nt_swiglu_ld", "gemm_nt_swiglu", out.buf.device, a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr,
          b2.codes_ptr, b2.scales_ptr, out.codes_ptr, out.ld, out.scales_ptr, M, N, a.k, a.ld, _mode(mode), _stream(out.buf))
    return out


def mx_gemm_nt_shared_b(a: MXData, a2: MXData, b: MXData) -> torch.Tensor:
    """bf16 [2, M, N]: deq(a) @ deq(b)^T and deq(a2) @ deq(b)^T, as `mx_gemm_nt_shared_a` with the
    roles of the operands swapped."""
    if _operands(a, a2, b):
        M, N, K = a.rows, b.rows, a.k
        if a2.rows != M or not a.depth == a2.depth == b.depth:
            raise ValueError("both first operands must have the same shape")
        out = torch.empty((2, M, N), dtype=torch.bfloat16, device=a.buf.device)
        if not _persistent_shape(M, N, K):
            _gemm_operands(a, b, out[0])
            _gemm_operands(a2, b, out[1])
            return out
        _call("mx_gemm_nt_shared_b_ld", "gemm_nt_shared_b", out.device, a.codes_ptr, a.scales_ptr, a2.codes_ptr,
              a2.scales_ptr, b.codes_ptr, b.scales_ptr, out.data_ptr(), out.data_ptr() + 2 * M * N, M, N, K, a.ld, N,
              _stream(out))
        return out
    M, K = a.codes.shape
    N = b.codes.shape[0]
    if a2.codes.shape != a.codes.shape or b.codes.shape[1] != K or not _depth(a) == _depth(a2) == _depth(b):
        raise ValueError("both first operands must have the same shape")
    out = torch.empty((2, M, N), dtype=torch.bfloat16, device=a.codes.device)
    if not _persistent_shape(M, N, K):
        mx_gemm_nt(a, b, out[0])
        mx_gemm_nt(a2, b, out[1])
        return out
    sa, sa2, sb = _as_mfma(a), _as_mfma(a2), _as_mfma(b)
    (ac, a2c, bc), ldk = _common_pitch(a.codes, a2.codes, b.codes)
    _call("mx_gemm_nt_shared_b_ld", "gemm_nt_shared_b", out.device, _ptr(ac), _ptr(sa), _ptr(a2c), _ptr(sa2),
          _ptr(bc), _ptr(sb), _ptr(out[0]), _ptr(out[1]), M, N, K, ldk, N, _stream(out))
    return out


# --------------------------------------------------------------------------- 3-D weights
def to_mx_dim0_batched(w: torch.Tensor, mode="floor", order: int = MX_SCALES_MFMA) -> MXData:
    """Row-wise cast of every matrix of w [G, R, C]: codes [G, R, C], one scale block each.

    A 3-D weight is G stacked matrices, so this is one row-wise cast of the [G*R, C] view; in
    MFMA order that equals G per-matrix blocks only when R is a multiple of 128, otherwise the
    matrices are cast one by one.
    """
    G, R, C = w.shape
    if order == MX_SCALES_MFMA and R % 128:
        parts = [to_mx_dim0(w[g], mode, order) for g in range(G)]
        return MXData(torch.stack([p.codes for p in parts]), torch.cat([p.scales for p in parts]), order)
    d = to_mx_dim0(w.reshape(G * R, C), mode, order)
    scales = d.scales if order == MX_SCALES_MFMA else d.scales.view(G, R, C // BLOCK)
    return MXData(d.codes.view(G, R, C), scales, order)


def to_mx_dim1_batched(w: torch.Tensor, mode="floor", order: int = MX_SCALES_MFMA) -> MXData:
    """Column-wise cast of every matrix of w [G, R, C]: codes [G, C, R]."""
    if w.dim() != 3 or w.dtype != torch.bfloat16 or not w.is_cuda:
        raise TypeError("expected a 3-D bf16 GPU tensor")
    w = w.contiguous()
    G, R, C = w.shape
    if R % BLOCK:
        raise ValueError(f"dim 1 ({R}) is not a multiple of {BLOCK}")
    codes = torch.empty((G, C, R), dtype=torch.uint8, device=w.device)
    per = mfma_scale_bytes(C, R // BLOCK) if order == MX_SCALES_MFMA else C * (R // BLOCK)
    scales = torch.empty(G * per, dtype=torch.uint8, device=w.device)
    _call("mx_cast_dim1_batched", "cast_dim1_batched", w.device, _ptr(w), G, R, C, C, _ptr(codes), _ptr(scales), _mode(mode), order, _stream(w))
    if order == MX_SCALES_ROWMAJOR:
        scales = scales.view(G, C, R // BLOCK)
    return MXData(codes, scales, order)


def to_mx_dim0_dim1_batched(w: torch.Tensor, mode="floor", order: int = MX_SCALES_MFMA):
    """Both casts of every matrix of w [G, R, C] from one read."""
    if w.dim() != 3 or w.dtype != torch.bfloat16 or not w.is_cuda:
        raise TypeError("expected a 3-D bf16 GPU tensor")
    w = w.contiguous()
    G, R, C = w.shape
    if R % BLOCK or C % BLOCK:
        raise ValueError(f"dims {R}, {C} must be multiples of {BLOCK}")
    codes = torch.empty((G, R, C), dtype=torch.uint8, device=w.device)
    codes_t = torch.empty((G, C, R), dtype=torch.uint8, device=w.device)
    if order == MX_SCALES_MFMA:
        per, per_t = mfma_scale_bytes(R, C // BLOCK), mfma_scale_bytes(C, R // BLOCK)
    else:
        per, per_t = R * (C // BLOCK), C * (R // BLOCK)
    scales = torch.empty(G * per, dtype=torch.uint8, device=w.device)
    scales_t = torch.empty(G * per_t, dtype=torch.uint8, device=w.device)
    _call("mx_cast_dim0_dim1_batched", "cast_dim0_dim1_batched", w.device, _ptr(w), G, R, C, C, _ptr(codes), _ptr(scales), _ptr(codes_t), _ptr(scales_t), _mode(mode), order, _stream(w))
    if order == MX_SCALES_ROWMAJOR:
        scales, scales_t = scales.view(G, R, C // BLOCK), scales_t.view(G, C, R // BLOCK)
    return MXData(codes, scales, order), MXData(codes_t, scales_t, order)


# --------------------------------------------------------------------------- grouped GEMMs
FAST_MAX_GROUPS = 510   # groups the persistent kernel keeps a table of in LDS
FAST_LENGTH_MULTIPLE = 128  # its operands' token axis: whole 128-deep K blocks / 128-row scale groups


def mx_grouped_gemm_2d3d(a: MXData, b: MXData, offs: torch.Tensor,
                         out: torch.Tensor | None = None) -> torch.Tensor:
    """out[rows of group g] = deq(a[rows of g]) @ deq(b[g])^T; rows past offs[-1] are zero.

    a: codes [T, K]; b: codes [G, N, K] with MFMA-order scales (G per-matrix blocks); offs:
    int32 [G] inclusive cumulative group sizes on the device.  With row-major scales for a the
    groups may end anywhere; with MFMA-order scales for a every group must end at a multiple
    of 32 rows (checked on the device: a violation fills the output with NaN) and the
    persistent kernel (csrc/mx_gemm32.hip) runs.
    """
    T, K = a.codes.shape
    G, N, Kb = b.codes.shape
    if K != Kb:
        raise ValueError(f"contraction mismatch: {K} vs {Kb}")
    if b.scale_order != MX_SCALES_MFMA:
        raise ValueError("2d3d expects MFMA-order scales for b")
    if offs.dtype != torch.int32 or offs.numel() != G:
        raise ValueError("offs must be int32 with one entry per group")
    if out is None:
        if _watched():
            return torch.ops.torchtitan_amd.mx_grouped_gemm_2d3d(a.codes, a.scales, a.scale_order,
                                                                 b.codes, b.scales, offs)
        return _grouped_2d3d_op(a.codes, a.scales, a.scale_order, b.codes, b.scales, offs)
    return _grouped_2d3d_into(a.codes, a.scales, a.scale_order, b.codes, b.scales, offs, _wrote(out))


def mx_grouped_gemm_2d3d_pair(a: MXData, b: MXData, a2: MXData, b2: MXData, offs: torch.Tensor,
                              out: torch.Tensor | None = None) -> torch.Tensor:
    """out[rows of g] = deq(a[rows of g]) @ deq(b[g])^T + deq(a2[rows of g]) @ deq(b2[g])^T, both
    sets with MFMA-order scales and 32-aligned groups (the persistent kernel); other layouts:
    two grouped GEMMs and a bf16 add."""
    T, K = a.codes.shape
    G, N, _ = b.codes.shape
    if a2.codes.shape != a.codes.shape or b2.codes.shape != b.codes.shape:
        raise ValueError("both operand sets must have the same shapes")
    fast = all(d.scale_order == MX_SCALES_MFMA for d in (a, b, a2, b2))
    if not fast or K % 128 or N % 8 or T % 32 or G > FAST_MAX_GROUPS:
        both = mx_grouped_gemm_2d3d(a, b, offs) + mx_grouped_gemm_2d3d(a2, b2, offs)
        return both if out is None else out.copy_(both)
    if offs.dtype != torch.int32 or offs.numel() != G:
        raise ValueError("offs must be int32 with one entry per group")
    if out is None:
        out = torch.empty((T, N), dtype=torch.bfloat16, device=a.codes.device)
    else:
        _wrote(out)
    _call("mx_grouped_gemm_2d3d_pair", "grouped_gemm_2d3d_pair", out.device, _ptr(a.codes), _ptr(a.scales),
          _ptr(b.codes), _ptr(b.scales), _ptr(a2.codes), _ptr(a2.scales), _ptr(b2.codes), _ptr(b2.scales),
          _ptr(offs), _ptr(out), T, N, K, G, out.stride(0), _stream(out))
    return out


def mx_grouped_gemm_2d3d_rows_out(a: MXData, b: MXData, offs: torch.Tensor, out_offs: torch.Tensor,
                                  out_rows: int, a2: MXData | None = None,
                                  b2: MXData | None = None) -> torch.Tensor:
    """bf16 [out_rows, N]: the grouped product (with a2, b2: the sum of two, as
    `mx_grouped_gemm_2d3d_pair`) of operands whose groups are padded, written without the padding:
    the first out_offs[g] - out_offs[g-1] rows of group g go to rows [out_offs[g-1], out_offs[g])
    (out_offs: int32 [G] inclusive ends on the device), rows from out_offs[-1] on are zero.

    Takes the place of the grouped GEMM followed by a gather of the unpadded rows (the second
    half of the padding wrapper, torchtitan/models/common/moe/utils.py:85-89 and :116).  MFMA-order scales and 32-aligned
    padded groups only (the persistent kernel); `rows_out_supported` tells.  The zero rows need
    a.codes to have at least as many rows behind its last group as the output has."""
    T, K = a.codes.shape
    G, N, _ = b.codes.shape
    if not rows_out_supported(a, b, a2, b2):
        raise ValueError("unpadded output needs MFMA-order scales, K % 128 == 0, N % 8 == 0, T % 32 == 0")
    for o in (offs, out_offs):
        if o.dtype != torch.int32 or o.numel() != G:
            raise ValueError("offs and out_offs must be int32 with one entry per group")
    if not 0 <= out_rows <= T:
        raise ValueError("the output cannot have more rows than the padded operand")
    if a2 is None:
        if _watched():  # as a dispatcher op: a forward GEMM whose output a checkpoint policy may keep
            return torch.ops.torchtitan_amd.mx_grouped_gemm_2d3d_rows_out(a.codes, a.scales, b.codes, b.scales,
                                                                          offs, out_offs, out_rows)
        return _grouped_2d3d_rows_out_op(a.codes, a.scales, b.codes, b.scales, offs, out_offs, out_rows)
    if a2.codes.shape != a.codes.shape or b2.codes.shape != b.codes.shape:
        raise ValueError("both operand sets must have the same shapes")
    return _grouped_2d3d_rows_out_op(a.codes, a.scales, b.codes, b.scales, offs, out_offs, out_rows,
                                     (a2.codes, a2.scales, b2.codes, b2.scales))


def rows_out_supported(a: MXData, b: MXData, a2: MXData | None = None, b2: MXData | None = None) -> bool:
    T, K = a.codes.shape
    G, N, _ = b.codes.shape
    every = [d for d in (a, b, a2, b2) if d is not None]
    return (len(every) in (2, 4) and all(d.scale_order == MX_SCALES_MFMA for d in every)
            and K % 128 == 0 and N % 8 == 0 and T % 32 == 0 and G <= FAST_MAX_GROUPS)


def mx_grouped_gemm_2d3d_shared_a(a: MXData, b: MXData, b2: MXData, offs: torch.Tensor) -> torch.Tensor:
    """bf16 [2, T, N]: grouped a x b[g]^T and grouped a x b2[g]^T.  One launch of the persistent
    kernel over both products when every scale buffer is in MFMA order (32-aligned groups),
    otherwise two grouped GEMMs; bit-identical either way."""
    T, K = a.codes.shape
    G, N, _ = b.codes.shape
    if b2.codes.shape != b.codes.shape:
        raise ValueError("both weight stacks must have the same shape")
    if offs.dtype != torch.int32 or offs.numel() != G:
        raise ValueError("offs must be int32 with one entry per group")
    if _watched():  # as dispatcher ops, so that a per-op checkpoint policy can keep the outputs
        return torch.stack((mx_grouped_gemm_2d3d(a, b, offs), mx_grouped_gemm_2d3d(a, b2, offs)))
    out = torch.empty((2, T, N), dtype=torch.bfloat16, device=a.codes.device)
    fast = all(d.scale_order == MX_SCALES_MFMA for d in (a, b, b2))
    if not fast or K % 128 or N % 8 or T % 32 or G > FAST_MAX_GROUPS:
        mx_grouped_gemm_2d3d(a, b, offs, out[0])
        mx_grouped_gemm_2d3d(a, b2, offs, out[1])
        return out
    _call("mx_grouped_gemm_2d3d_shared_a", "grouped_gemm_2d3d_shared_a", out.device, _ptr(a.codes), _ptr(a.scales),
          _ptr(b.codes), _ptr(b.scales), _ptr(b2.codes), _ptr(b2.scales), _ptr(offs), _ptr(out[0]), _ptr(out[1]),
          T, N, K, G, N, _stream(out))
    return out


def mx_grouped_gemm_2d2d_shared_b(at: MXData, at2: MXData, bt: MXData, offs: torch.Tensor) -> torch.Tensor:
    """bf16 [2, G, N, K]: out[0][g] = at[:, tokens of g] x bt[:, tokens of g]^T and out[1][g] the
    same with at2.  One launch of the persistent kernel when the scales are in MFMA order,
    otherwise two grouped GEMMs; bit-identical either way."""
    N, T = at.codes.shape
    K = bt.codes.shape[0]
    if at2.codes.shape != at.codes.shape or bt.codes.shape[1] != T:
        raise ValueError("operand shapes do not match")
    G = offs.numel()
    out = torch.empty((2, G, N, K), dtype=torch.bfloat16, device=at.codes.device)
    fast = all(d.scale_order == MX_SCALES_MFMA for d in (at, at2, bt))
    if not fast or T == 0 or T % 128 or K % 8:
        mx_grouped_gemm_2d2d(at, bt, offs, out[0])
        mx_grouped_gemm_2d2d(at2, bt, offs, out[1])
        return out
    _call("mx_grouped_gemm_2d2d_shared_b", "grouped_gemm_2d2d_shared_b", out.device, _ptr(at.codes), _ptr(at.scales),
          _ptr(at2.codes), _ptr(at2.scales), _ptr(bt.codes), _ptr(bt.scales), _ptr(offs), _ptr(out[0]), _ptr(out[1]),
          T, N, K, G, _stream(out))
    return out


def mx_grouped_gemm_2d2d(at: MXData, bt: MXData, offs: torch.Tensor,
                         out: torch.Tensor | None = None) -> torch.Tensor:
    """out[g] = deq(at[:, tokens of g]) @ deq(bt[:, tokens of g])^T  ->  [G, N, K] bf16.

    at: codes [N, T], bt: codes [K, T] (column-wise casts), scales of both in the same order.
    Groups may be any multiple of 32 tokens (checked on the device: a violation gives NaN).
    MFMA order: T a multiple of 128 (the token axis may run past the last group) and the
    persistent kernel (csrc/mx_gemm32.hip) runs.
    """
    N, T = at.codes.shape
    K, Tb = bt.codes.shape
    if T != Tb:
        raise ValueError(f"token count mismatch: {T} vs {Tb}")
    if at.scale_order != bt.scale_order:
        raise ValueError("2d2d expects both scale buffers in the same order")
    G = offs.numel()
    if out is None:
        out = torch.empty((G, N, K), dtype=torch.bfloat16, device=at.codes.device)
    else:
        _wrote(out)
    _call("mx_grouped_gemm_2d2d", "grouped_gemm_2d2d", out.device, _ptr(at.codes), _ptr(at.scales), _ptr(bt.codes), _ptr(bt.scales), _ptr(offs), _ptr(out), T, N, K, G, at.scale_order, _stream(out))
    return out


def group_offsets_pad(counts: torch.Tensor, experts_per_rank: int, num_ranks: int, max_len: int,
                      alignment: int):
    """(permuted_indices int64 [max_len], m_sizes int32 [E], m_offsets int32 [E]); one launch."""
    if not counts.is_cuda:
        raise _lib.MXLibraryError("group_offsets_pad runs on the GPU only")
    c32 = counts.to(torch.int32).contiguous()
    perm = torch.empty(max_len, dtype=torch.int64, device=counts.device)
    m_sizes = torch.empty(experts_per_rank, dtype=torch.int32, device=counts.device)
    m_offsets = torch.empty(experts_per_rank, dtype=torch.int32, device=counts.device)
    _call("mx_group_offsets_pad", "group_offsets_pad", counts.device, _ptr(c32), experts_per_rank, num_ranks, max_len, alignment, _ptr(perm), _ptr(m_sizes), _ptr(m_offsets), _stream(counts))
    return perm, m_sizes, m_offsets
