"""Weight wrapper that re-routes ``F.linear`` and ``torch._grouped_mm`` to the MXFP8 kernels.

After conversion a target weight is still an ordinary trainable high-precision parameter
(optimizer, ``init_weights``, ``to_empty`` and checkpointing keep working on it), but it is an
instance of ``MXFP8TrainingWeight``; its ``__torch_function__`` sends the two GEMM entry points
to autograd functions that quantize dynamically and call the HIP library in forward and
backward.  This is the role the reference gives to the external tensor subclass installed by
its converter (torchtitan/components/quantization/mx.py:27-31,93-96,119-125).

Passes of one linear with W [N, K], X [M, K], dY [M, N]  (every GEMM is "NT"):
    forward  Y  = cast_dim0(X)  x cast_dim0(W)        contraction K
    dgrad    dX = cast_dim0(dY) x cast_dim1(W)        contraction N
    wgrad    dW = cast_dim1(dY) x cast_dim1(X)        contraction M
X and W are read once in forward (fused row+column cast) and their column-wise forms are what
is saved for backward; dY is read once in backward.
"""
from __future__ import annotations

import weakref

import torch
import torch.nn.functional as F

from . import _lib, ops
from .ops import MX_SCALES_MFMA, MX_SCALES_ROWMAJOR, MXData


class MXFP8Config:
    """Per-weight recipe: scale mode and whether grouped GEMMs pad token groups to 32."""

    __slots__ = ("scale_mode", "pad_token_groups_for_grouped_mm", "fuse_swiglu_cast", "cache_weight_casts",
                 "fuse_rmsnorm_cast")

    def __init__(self, scale_mode: str = "rceil", pad_token_groups_for_grouped_mm: bool = True,
                 fuse_swiglu_cast: bool = True, cache_weight_casts: bool = False,
                 fuse_rmsnorm_cast: bool = False):
        if scale_mode not in ops.SCALE_MODES:
            raise ValueError(f"unknown scale mode {scale_mode!r}")
        self.scale_mode = scale_mode
        self.pad_token_groups_for_grouped_mm = pad_token_groups_for_grouped_mm
        self.fuse_swiglu_cast = fuse_swiglu_cast
        self.cache_weight_casts = cache_weight_casts
        self.fuse_rmsnorm_cast = fuse_rmsnorm_cast

    def __repr__(self):
        return (f"MXFP8Config(scale_mode={self.scale_mode!r}, "
                f"pad_token_groups_for_grouped_mm={self.pad_token_groups_for_grouped_mm})")


# ----------------------------------------------------------------------------- cast reuse
def _capture(x: torch.Tensor) -> int:
    """The graph capture that work on x is part of now (0: none)."""
    if not x.is_cuda or not torch.cuda.is_current_stream_capturing():
        return 0
    return _lib.blocks().capture_id(ops._stream(x))


def _place(x: torch.Tensor):
    """Where work on x goes now: the current stream of its GPU, and the graph capture that it is part of."""
    return (ops._stream(x), _capture(x)) if x.is_cuda else None


class _ActivationCastCache:
    """Remembers the fused cast of the last activation tensor.

    w1(x) and w3(x) of a SwiGLU block, or wq/wk/wv of attention, receive the same tensor object;
    the second and third linear reuse the codes instead of re-reading x.  The entry is keyed on
    object identity, the tensor's version counter and its address, on the stream that the cast was
    launched on, and holds only a weak reference to the activation.

    What keeps a hit from being stale: an entry lives for one forward at most.  It is dropped at
    the start of every backward of a converted linear and by `clear_cast_cache()`, and serves
    neither another stream, whose work is not ordered behind the cast and which the codes' memory
    does not belong to, nor anything outside the graph capture that it was made in (an entry made by
    an eager warm-up or in another capture is never reused under capture, so every graph records the
    casts that it needs, and an entry made under capture is never reused by eager code).  Writes through this package's `out=` arguments
    bump the destination's version counter.  A caller that overwrites an activation behind
    autograd's back (`.data`, a foreign kernel) between two forwards without a backward in between
    must call `clear_cast_cache()`.

    There is one entry for all threads, replaced and dropped as a whole: two threads cost each other
    their hits, and autograd's own threads drop the forward's entry.
    """

    def __init__(self):
        self._entry = None  # (weak reference to the activation, key, cast)

    @staticmethod
    def _key(x: torch.Tensor, mode):
        return x._version, mode, x.data_ptr(), _place(x)

    def get(self, x: torch.Tensor, mode):
        entry = self._entry
        if entry is not None and entry[0]() is x and entry[1] == self._key(x, mode):
            return entry[2]
        return None

    def put(self, x: torch.Tensor, mode, value):
        self._entry = weakref.ref(x), self._key(x, mode), value

    def clear(self):
        self._entry = None


_cast_cache = _ActivationCastCache()


def clear_cast_cache() -> None:
    """Forget the remembered activation cast (see `_ActivationCastCache`)."""
    _cast_cache.clear()


def _cast_activation(x2: torch.Tensor, src: torch.Tensor, mode: str, need_cols: bool, pitch_pad: int = 0):
    """(row-wise, column-wise or None) GEMM operands of the 2-D activation `x2` (any number of
    tokens), remembered for sibling linears that receive the same tensor `src`."""
    key = (mode, pitch_pad)
    hit = _cast_cache.get(src, key)
    if hit is not None and (hit[1] is not None or not need_cols):
        return hit
    q = ops.to_operands(x2, mode, True, need_cols, pitch_pad)
    _cast_cache.put(src, key, q)
    return q


# ----------------------------------------------------------------------------- weight casts
def _follow(done: torch.cuda.Event, *casts) -> None:
    """Orders the current stream behind `done`, an event behind the casts, and keeps their memory until the stream has
    read them.  (Not under capture, which begins with the device idle and cannot wait for work outside it.)"""
    if torch.cuda.is_current_stream_capturing():
        return
    for q in casts:
        if q is None:
            continue
        for t in (q.buf, q.scales_buf) if type(q) is ops.Operand else (q.codes, q.scales):
            here = torch.cuda.current_stream(t.device)
            here.wait_event(done)
            t.record_stream(here)


class _WeightCastCache:
    """MXFP8 forms of weights that have not changed since they were cast.

    A weight changes once per optimizer step but is cast in every forward; with gradient
    accumulation, several forwards per step, or a hand-over of the weights in MXFP8 form, the
    casts after the first are repeats.  An entry is keyed on the weight's memory (address, shape,
    strides) and valid while that storage is alive and its version counter is unchanged: every
    in-place update (optimizer step, ``copy_``, init) invalidates it.  A cast made under graph capture
    exists once that graph has run: its entry serves that capture only.  A hit on another stream than the
    one that cast orders that stream behind the cast.  Off unless the converter
    is built with ``cache_weight_casts=True``; holds 2 bytes per weight element, 1 where only forwards without gradients
    have read a frozen weight (`cached_weights`)."""

    def __init__(self):
        self._entries = {}

    @staticmethod
    def _key(w: torch.Tensor, mode):
        return (w.data_ptr(), tuple(w.shape), tuple(w.stride()), w.dtype, mode)

    def get(self, w: torch.Tensor, mode):
        e = self._entries.get(self._key(w, mode))
        if e is None:
            return None
        ref, version, capture, stream, done, rows, cols = e
        if ref.expired() or version != w._version or (capture and capture != _capture(w)):
            return None
        if done is not None and stream[1] != ops._raw_stream(stream[0]):
            _follow(done, rows, cols)
        return rows, cols

    def put(self, w: torch.Tensor, mode, rows: MXData, cols):
        from torch.multiprocessing.reductions import StorageWeakRef

        own = self._key(w, mode)
        dead = [k for k, e in self._entries.items()  # (also the form with another pitch of a weight since updated)
                if e[0].expired() or (e[1] != w._version and k[:4] == own[:4] and k[4][::2] == mode[::2])]
        for k in dead:
            self._entries.pop(k, None)
        capture, stream, done = _capture(w), None, None
        if w.is_cuda and not capture:
            stream, done = (w.device.index, ops._stream(w)), torch.cuda.current_stream(w.device).record_event()
        self._entries[own] = (StorageWeakRef(w.untyped_storage()), w._version, capture, stream, done, rows, cols)

    def clear(self):
        self._entries.clear()

    def __len__(self):
        return len(self._entries)


_weight_cache = _WeightCastCache()


def _cast_weight(w: torch.Tensor, mode: str, need_cols: bool, cfg: MXFP8Config, pitch_pad: int = 0,
                 whole_blocks: bool = True):
    """(row-wise, column-wise or None) MXFP8 forms of a weight [N, K] or stacked [G, N, K], MFMA
    scale order.  2-D weights: GEMM operands as `ops.to_operands` makes them (the contraction in whole
    128-deep blocks, `pitch_pad` bytes between the rows); with `whole_blocks` off the dense form
    over exactly N and K.  The column-wise form of a stack or a dense form exists when asked for and
    N is a multiple of 32.  Cached, both forms are made for whoever asks first, but with padded rows: there the
    column-wise one joins the entry when it is first asked for (see `cached_weights`)."""
    cached = cfg.cache_weight_casts
    whole = whole_blocks and w.dim() == 2
    # the cache keeps padded, rounded-up and dense casts apart; where nothing is rounded the last two have the
    # same bytes, and one entry serves both
    key = (mode, pitch_pad, whole and _rounded_up(w))
    if cached:
        hit = _weight_cache.get(w, key)
        if hit is not None and (hit[1] is not None or not need_cols or whole or w.shape[-2] % ops.BLOCK):
            return _as_asked(w, key, hit, need_cols, whole)
        need_cols = need_cols or not pitch_pad  # cast once in full, whoever asks first
    wb = (_castable(w) if whole else w if w.dtype == torch.bfloat16 else w.to(torch.bfloat16)).contiguous()
    both = need_cols and (whole or wb.shape[-2] % ops.BLOCK == 0)
    if wb.dim() == 3:
        q = ops.to_mx_dim0_dim1_batched(wb, mode, MX_SCALES_MFMA) if both else (_cast_w_rows(wb, mode), None)
    elif both:
        q = ops.to_mx_dim0_dim1(wb, mode, MX_SCALES_MFMA, pitch_pad, whole)
    else:
        q = (ops.to_operands(wb, mode, True, False, pitch_pad) if whole
             else (ops.to_mx_dim0(wb, mode, MX_SCALES_MFMA), None))
    if cached:
        _weight_cache.put(w, key, q[0], q[1])
    return q


def cached_weights(ws, mode: str, need_cols, cfg: MXFP8Config, frozen: bool = False):
    """(`_cast_weight` of every matrix as whole-block operands, bytes between the rows of their codes) for an eager forward
    on cached casts: all operands of a product have one pitch, so the forward casts its activations with this one.

    The casts that are there are taken as they lie, whoever made them, so that a weight is cast once and kept in one
    form; column-wise codes that a backward needs join an entry that has none.  Where there are none yet, a forward
    without gradients on `frozen` weights leaves rows apart and casts row-wise only (as `post_optimizer_hook` does on a
    model that takes no gradients at all), anyone else makes the dense form, which traced callers share.
    Rows a whole number of KB long lie on few channels of the L2 and of the memory: 512 tokens 4096 -> 2 x 14336
    59.7 us on dense rows from memory, 52.0 on rows apart; 14336 -> 4096 52.0 and 47.7."""
    dense = False
    for pad in ((ops.CODE_PITCH_PAD, 0) if frozen else (0, ops.CODE_PITCH_PAD)):
        found = []
        for w in ws:
            key = (mode, pad, _rounded_up(w))
            hit = _weight_cache.get(w, key)
            if hit is not None:
                found.append((w, key, hit))
            elif pad:
                break
        if len(found) == len(ws):
            return [_as_asked(*each, need, True) for each, need in zip(found, need_cols)], pad
        dense = dense or (pad == 0 and len(found) > 0)
    pad = ops.CODE_PITCH_PAD if frozen and not dense else 0
    return [_cast_weight(w, mode, need, cfg, pad) for w, need in zip(ws, need_cols)], pad


def rows_apart(w: torch.Tensor, mode: str) -> bool:
    """The cache holds operands of the matrix with rows apart: for traced callers, so that they do not cast what
    `post_optimizer_hook` or a forward without gradients has cast."""
    return (w.dim() == 2 and ops.CODE_PITCH_PAD > 0
            and _weight_cache.get(w, (mode, ops.CODE_PITCH_PAD, _rounded_up(w))) is not None)


def _rounded_up(w: torch.Tensor) -> bool:
    """Whole-block operands of the matrix are larger than dense ones."""
    return bool(w.shape[0] % ops.WHOLE_BLOCK or w.shape[1] % ops.WHOLE_BLOCK)


def _as_asked(w: torch.Tensor, key, hit, need_cols: bool, whole: bool):
    """A cached cast as its caller wants it: in its form, with the column-wise codes.  Those that are cast now join the entry,
    whose row-wise codes stay where they lie (a graph may read them), except under graph capture, where only the replay
    fills them."""
    if (type(hit[0]) is ops.Operand) != whole:
        hit = _in_form(w, key, hit, whole)
    if need_cols and whole and hit[1] is None:
        hit = hit[0], ops.to_operands(_castable(w).contiguous(), key[0], False, True, hit[0].ld - hit[0].k)[1]
        if not (w.is_cuda and torch.cuda.is_current_stream_capturing()):
            _weight_cache.put(w, key, *hit)
    return hit


def _in_form(w: torch.Tensor, key, hit, whole: bool):
    """A cached cast in the other form, which its caller wants: operands, or dense `MXData` (views of an operand's buffer).
    An operand made from a dense entry takes its place, except under graph capture, where it is filled
    by the replay only and the entry may serve others."""
    rows, cols = hit
    if not whole:
        return rows.data(), (None if cols is None else cols.data())
    hit = ops.Operand.of(rows), (None if cols is None else ops.Operand.of(cols))
    if not (w.is_cuda and torch.cuda.is_current_stream_capturing()):
        _weight_cache.put(w, key, *hit)
    return hit


def _one_launch(ws, cfg: MXFP8Config, whole_blocks: bool = True) -> bool:
    """Both forms of all the weights can come from one launch (`ops.CastList`): nothing cached,
    matrices as whole-block operands or stacks of whole tiles, on one GPU."""
    if cfg.cache_weight_casts or len({w.device for w in ws}) != 1 or not ws[0].is_cuda:
        return False
    if all(w.dim() == 2 for w in ws):
        return whole_blocks
    return all(w.dim() == 3 and w.shape[1] % ops.WHOLE_BLOCK == 0 and w.shape[2] % ops.WHOLE_BLOCK == 0 for w in ws)


def _list_weights(casts: ops.CastList, ws, mode: str, pitch_pad: int) -> list:
    wbs = [_castable(w).contiguous() for w in ws]
    return [casts.add_stack(w) if w.dim() == 3
            else ops.to_mx_dim0_dim1(w, mode, MX_SCALES_MFMA, pitch_pad, True, cast_list=casts) for w in wbs]


def _cast_weights(ws, mode: str, need_cols, cfg: MXFP8Config, pitch_pad: int = 0, whole_blocks: bool = True) -> list:
    """`_cast_weight` of every weight, `need_cols[i]` for its column-wise form."""
    if all(need_cols) and _one_launch(ws, cfg, whole_blocks):
        casts = ops.CastList(mode)
        q = _list_weights(casts, ws, mode, pitch_pad)
        casts.launch()
        return q
    return [_cast_weight(w, mode, need, cfg, pitch_pad, whole_blocks) for w, need in zip(ws, need_cols)]


def _cast_activation_and_weights(x2: torch.Tensor, src: torch.Tensor, ws, mode: str, need_dx: bool, need_dw: bool,
                                 cfg: MXFP8Config, pitch_pad: int = 0) -> list:
    """[`_cast_activation` of x2, then `_cast_weight` of every weight] (column-wise forms of the activation
    with need_dw, of the weights with need_dx), in one launch where both forms of all are wanted."""
    if need_dx and need_dw and x2.device == ws[0].device and x2.numel() and _one_launch(ws, cfg):
        key = (mode, pitch_pad)
        hit = _cast_cache.get(src, key)
        if hit is None or hit[1] is None:
            casts = ops.CastList(mode)
            hit = casts.add(x2, pitch_pad)
            rest = _list_weights(casts, ws, mode, pitch_pad)
            casts.launch()
            _cast_cache.put(src, key, hit)
            return [hit, *rest]
    return [_cast_activation(x2, src, mode, need_cols=need_dw, pitch_pad=pitch_pad),
            *_cast_weights(ws, mode, [need_dx] * len(ws), cfg, pitch_pad)]


# ----------------------------------------------------------------------------- dense linear
def _castable(t: torch.Tensor) -> torch.Tensor:
    """`t` in a type the operand casts read: bf16, or float32 which they round to bf16 themselves."""
    return t if t.dtype in (torch.bfloat16, torch.float32) else t.to(torch.bfloat16)


def _linear_apply(x2: torch.Tensor, src: torch.Tensor, weight: torch.Tensor, cfg: MXFP8Config, K: int, N: int, frozen: bool):
    """x2 W^T without gradients.  The activation's cast is shared with sibling linears on `src`, but for few rows, which are
    cast inside their product; the weight is cast once, whichever way the product runs."""
    mode, pad = cfg.scale_mode, ops.CODE_PITCH_PAD
    if cfg.cache_weight_casts:
        for pad in ((pad, 0) if frozen else (0, pad)):  # (what `cached_weights` finds, 1.5 us sooner)
            wq0, _ = _weight_cache.get(weight, (mode, pad, _rounded_up(weight))) or (None, None)
            if type(wq0) is ops.Operand:
                break
        else:
            ((wq0, _),), pad = cached_weights((weight,), mode, (False,), cfg, frozen)
    else:
        wq0, _ = _cast_weight(weight, mode, False, cfg, pitch_pad=pad)
    native = ops.native_block_ok(x2, K, N)
    if native:  # (what else `few_rows_ok` asks for, the native call checks itself)
        few = x2.dtype == torch.bfloat16 and ops.few_rows_size(x2.shape[0], K, N)
        native = few or _cast_cache.get(src, (mode, pad)) is None
    else:
        few = ops.few_rows_ok(x2, N)
    if native and type(wq0) is ops.Operand:
        out = _lib.blocks().linear_apply(x2, wq0.buf, wq0.scales_buf, wq0.layout, ops._mode(mode), few)
        if out is not None:
            y, xr, xr_layout = out
            if xr is not None:
                _cast_cache.put(src, (mode, pad), (ops.Operand(xr, xr_layout), None))
            return y
    if few and ops.few_rows_ok(x2, N):
        return ops.mx_few_rows(x2, wq0, mode)
    xq0, _ = _cast_activation(x2, src, mode, need_cols=False, pitch_pad=pad)
    return ops.mx_gemm_nt(xq0, wq0)


def _linear_forward(x, weight, cfg: MXFP8Config, need_dx: bool, need_dw: bool, frozen: bool = False):
    """(y, column-wise x or None, column-wise W or None) of the converted linear; `frozen`: see `cached_weights`."""
    mode, K, N = cfg.scale_mode, x.shape[-1], weight.shape[0]
    x2 = _castable(x if x.dim() == 2 else x.reshape(-1, K))
    if not (need_dx or need_dw):
        y = _linear_apply(x2, x, weight, cfg, K, N, frozen)
        return (y if x.dim() == 2 else y.view(*x.shape[:-1], N)), None, None
    # rows further apart than they are long, except with cached weight casts, which have a pitch of their own
    cached, pad = cfg.cache_weight_casts, ops.CODE_PITCH_PAD
    if need_dx and need_dw and pad and not cached and ops.native_block_ok(x2, K, N) and _cast_cache.get(x, (mode, pad)) is None:
        out = _lib.blocks().linear_forward(x2, _castable(weight), ops._mode(mode), pad)
        if out is not None:
            y, xr, xr_layout, xc, xc_layout, wc, wc_layout = out
            xq1 = ops.Operand(xc, xc_layout)
            _cast_cache.put(x, (mode, pad), (ops.Operand(xr, xr_layout), xq1))
            return (y if x.dim() == 2 else y.view(*x.shape[:-1], N)), xq1, ops.Operand(wc, wc_layout)
    if cached:
        ((wq0, wq1),), pad = cached_weights((weight,), mode, (need_dx,), cfg)
        xq0, xq1 = _cast_activation(x2, x, mode, need_cols=need_dw, pitch_pad=pad)
    else:
        (xq0, xq1), (wq0, wq1) = _cast_activation_and_weights(x2, x, (weight,), mode, need_dx, need_dw, cfg, pad)
    y = ops.mx_gemm_nt(xq0, wq0)
    return (y if x.dim() == 2 else y.view(*x.shape[:-1], N)), xq1, wq1


class _MXLinear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, cfg: MXFP8Config):
        need_dx, need_dw = ctx.needs_input_grad[:2]
        y, xq1, wq1 = _linear_forward(x, weight, cfg, need_dx, need_dw)
        ctx.cfg = cfg
        ctx.x_shape = x.shape
        ctx.x_dtype = x.dtype
        ctx.w_dtype = weight.dtype
        ctx.x_layout, ctx.w_layout = (xq1.layout if need_dw else None), (wq1.layout if need_dx else None)
        if need_dx or need_dw:  # the backward's casts take the pitch of the operands that they meet
            kept = wq1 if need_dx else xq1
            ctx.pad = kept.ld - kept.k
        ctx.save_for_backward(xq1.buf if need_dw else None, wq1.buf if need_dx else None)
        return y

    @staticmethod
    def backward(ctx, dy):
        _cast_cache.clear()  # the forward whose sibling linears shared a cast is over
        mode = ctx.cfg.scale_mode
        need_dx, need_dw = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        x_buf, w_buf = ctx.saved_tensors
        dy2 = _castable(dy if dy.dim() == 2 else dy.reshape(-1, dy.shape[-1]))
        pad = ctx.pad
        dx = dw = None
        if need_dx and need_dw and pad and ops.native_block_ok(dy2, dy2.shape[1], ctx.x_shape[-1]):
            out = _lib.blocks().linear_backward(dy2, x_buf, ctx.x_layout, w_buf, ctx.w_layout, ops._mode(mode), pad,
                                                ctx.x_dtype == torch.float32, ctx.w_dtype == torch.float32)
            if out is not None:
                dx, dw = out
                dx = dx if len(ctx.x_shape) == 2 else dx.view(ctx.x_shape)
                return (dx if dx.dtype == ctx.x_dtype else dx.to(ctx.x_dtype),
                        dw if dw.dtype == ctx.w_dtype else dw.to(ctx.w_dtype), None)
        dyq0, dyq1 = ops.to_operands(dy2, mode, need_dx, need_dw, pad)
        if need_dx:
            dx = ops.mx_gemm_nt_as(dyq0, ops.saved_operand(w_buf, ctx.w_layout, dy2.device), ctx.x_dtype)
            if len(ctx.x_shape) != 2:
                dx = dx.view(ctx.x_shape)
        if need_dw:
            dw = ops.mx_gemm_nt_as(dyq1, ops.saved_operand(x_buf, ctx.x_layout, dy2.device), ctx.w_dtype)
        return dx, dw, None


def mx_linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, cfg: MXFP8Config, frozen: bool = False):
    """``F.linear`` with the matmul in MXFP8; the bias add stays in high precision.  `frozen`: the weight takes no
    gradients (`weight` itself, an alias made without gradients, does not tell)."""
    if x.shape[-1] % ops.BLOCK:
        raise ValueError(f"MXFP8 linear needs in_features % 32 == 0, got {x.shape[-1]}")
    out_dtype = x.dtype
    if torch._C._is_any_autocast_enabled() and torch.is_autocast_enabled(x.device.type):
        out_dtype = torch.get_autocast_dtype(x.device.type)
    if torch.is_grad_enabled() or ops._transformed():
        y = _MXLinear.apply(x, weight, cfg)
    else:
        y = _linear_forward(x, weight, cfg, False, False, frozen)[0]
    if y.dtype != out_dtype:
        y = y.to(out_dtype)
    if bias is not None:
        y = y + bias.to(y.dtype)
    return y


# ----------------------------------------------------------------------------- grouped GEMM
def _pad_plan(offs: torch.Tensor, T: int, align: int = 32, length_multiple: int = 1, direct: bool = False):
    """Device-side plan that moves rows of variable-size groups into `align`-aligned groups.

    Returns (gather indices into [x; 0-row] for the padded layout, padded inclusive offsets,
    the way back).  The way back is, for every original row, its row in the padded layout or the
    index of an appended zero row (int64 [T]: a gather) -- or, with `direct`, a copy of the
    unpadded group ends (int32 [G]) for a grouped GEMM that writes the unpadded rows itself.
    No host synchronisation: the padded length is the static bound `ops.plan_length`.
    """
    G = offs.numel()
    sizes = torch.diff(offs, prepend=offs.new_zeros(1))
    max_len = ops.plan_length(T, G, align, length_multiple)
    perm, _, m_offsets = ops.group_offsets_pad(sizes, G, 1, max_len, align)
    if direct:
        return perm, m_offsets, offs.to(torch.int32).clone()
    back = torch.full((T + 1,), max_len, dtype=torch.int64, device=offs.device)
    back[perm] = torch.arange(max_len, device=offs.device)  # perm == -1 writes the spare slot T
    return perm, m_offsets, back[:T]


def _cast_into_groups(t: torch.Tensor, perm, mode: str, order: int, want_cols: bool):
    """(row-wise, column-wise or None) casts of `t` moved into its padded group layout: the
    gather by `perm` happens inside the cast kernel (padding slots read as zero rows)."""
    if perm is not None:
        return ops.to_mx_rows_gathered(t, perm, mode, order, want_cols)
    if want_cols:
        return ops.to_mx_dim0_dim1(t, mode, order)
    return ops.to_mx_dim0(t, mode, order), None


def _grouped_2d3d_padded(a: MXData, b: MXData, offs_p: torch.Tensor, back, out_rows: int,
                         a2: MXData | None = None, b2: MXData | None = None):
    """Grouped GEMM (with a2, b2: the sum of two) in the padded layout, result in the original
    row order [out_rows, N]; `back` as `_pad_plan` returns it (None: nothing was padded).  On
    the gather path one spare zero row behind the GEMM's output serves rows that belong to no
    group."""
    Tp, N = a.codes.shape[0], b.codes.shape[1]
    two = a2 is not None
    if back is not None and back.dtype == torch.int32:  # the GEMM leaves the padding out itself
        return ops.mx_grouped_gemm_2d3d_rows_out(a, b, offs_p, back, out_rows, a2, b2)
    if back is None:
        return ops.mx_grouped_gemm_2d3d_pair(a, b, a2, b2, offs_p) if two else ops.mx_grouped_gemm_2d3d(a, b, offs_p)
    if ops._watched() and not two:  # the dispatcher form of the GEMM allocates its own output
        y = ops.mx_grouped_gemm_2d3d(a, b, offs_p)
        return torch.cat((y, y.new_zeros(1, N)))[back]
    buf = torch.empty((Tp + 1, N), dtype=torch.bfloat16, device=a.codes.device)
    buf[Tp].zero_()
    if two:
        ops.mx_grouped_gemm_2d3d_pair(a, b, a2, b2, offs_p, buf[:Tp])
    else:
        ops.mx_grouped_gemm_2d3d(a, b, offs_p, buf[:Tp])
    return buf[back]


class _MXGroupedMM(torch.autograd.Function):
    """out[rows of g] = x[rows of g] @ w[g]^T with w [G, N, K]; offs = inclusive cumsum, int32."""

    @staticmethod
    def forward(ctx, x, weight, offs, cfg: MXFP8Config):
        mode = cfg.scale_mode
        T, K = x.shape
        G, N, _ = weight.shape
        xb = x if x.dtype == torch.bfloat16 else x.to(torch.bfloat16)
        w = weight if weight.dtype == torch.bfloat16 else weight.to(torch.bfloat16)
        w = w.contiguous()
        plan = None
        # Groups are padded to the 32 rows the format needs; the persistent kernel takes them as
        # they are (scales in MFMA order, the token axis rounded up to whole 128-deep blocks).
        fast = K % 128 == 0 and N % 128 == 0 and G <= ops.FAST_MAX_GROUPS
        order = MX_SCALES_MFMA if fast else MX_SCALES_ROWMAJOR
        perm = back = None
        if cfg.pad_token_groups_for_grouped_mm or fast:
            plan = _pad_plan(offs, T, ops.BLOCK, ops.FAST_LENGTH_MULTIPLE if fast else 1, direct=fast)
            perm, offs_p, back = plan
        else:
            offs_p = offs
            if T % ops.BLOCK:
                raise ValueError("without padding the token dimension must be a multiple of 32")
        xb = xb.contiguous()
        need_dx, need_dw = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        xq0, xq1 = _cast_into_groups(xb, perm, mode, order, need_dw)
        wq0, wq1 = _cast_weight(weight, mode, need_dx, cfg)
        y = _grouped_2d3d_padded(xq0, wq0, offs_p, back, T)
        ctx.cfg = cfg
        ctx.dims = (T, K, N, G)
        ctx.dtypes = (x.dtype, weight.dtype)
        ctx.padded = plan is not None
        ctx.order = order
        saved = [offs_p]
        if plan is not None:
            saved += [plan[0], plan[2]]
        if need_dw:
            saved += [xq1.codes, xq1.scales]
        if need_dx:
            ctx.have_wq1 = wq1 is not None
            saved += [wq1.codes, wq1.scales] if wq1 is not None else [w]
        ctx.save_for_backward(*saved)
        return y

    @staticmethod
    def backward(ctx, dy):
        mode = ctx.cfg.scale_mode
        T, K, N, G = ctx.dims
        need_dx, need_dw = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        saved = list(ctx.saved_tensors)
        offs_p = saved.pop(0)
        dyb = (dy if dy.dtype == torch.bfloat16 else dy.to(torch.bfloat16)).contiguous()
        perm = back = None
        if ctx.padded:
            perm, back = saved.pop(0), saved.pop(0)
        dx = dw = None
        if need_dw:
            xq1 = MXData(saved.pop(0), saved.pop(0), ctx.order)
        if ctx.padded or (need_dx and need_dw and N % ops.BLOCK == 0):
            dyq0, dyq1 = _cast_into_groups(dyb, perm, mode, ctx.order, need_dw)
        else:
            dyq0 = ops.to_mx_dim0(dyb, mode, ctx.order) if need_dx else None
            dyq1 = ops.to_mx_dim1(dyb, mode, ctx.order) if need_dw else None
        if need_dx:
            if ctx.have_wq1:
                wq1 = MXData(saved.pop(0), saved.pop(0), MX_SCALES_MFMA)
            else:
                wq1 = ops.to_mx_dim1_batched(saved.pop(0), mode, MX_SCALES_MFMA)
            dx = _grouped_2d3d_padded(dyq0, wq1, offs_p, back, T)
            if dx.dtype != ctx.dtypes[0]:
                dx = dx.to(ctx.dtypes[0])
        if need_dw:
            dw = ops.mx_grouped_gemm_2d2d(dyq1, xq1, offs_p)
            if dw.dtype != ctx.dtypes[1]:
                dw = dw.to(ctx.dtypes[1])
        return dx, dw, None, None


def _cast_w_rows(w: torch.Tensor, mode: str) -> MXData:
    """Row-wise cast of stacked matrices w [G, N, K] with one MFMA-order scale block each."""
    return ops.to_mx_dim0_batched(w, mode, MX_SCALES_MFMA)


def mx_grouped_mm(x: torch.Tensor, w_t: torch.Tensor, offs: torch.Tensor, cfg: MXFP8Config):
    """``torch._grouped_mm(x, w_t, offs=offs)`` for x [T, K], w_t [G, K, N] = weight^T."""
    if x.dim() != 2 or w_t.dim() != 3 or offs is None:
        raise NotImplementedError("MXFP8 grouped_mm supports the 2D x 3D form with offsets only")
    weight = w_t.transpose(-2, -1)  # back to the parameter's [G, N, K] layout
    if x.shape[-1] % ops.BLOCK:
        raise ValueError(f"MXFP8 grouped_mm needs K % 32 == 0, got {x.shape[-1]}")
    return _MXGroupedMM.apply(x, weight, offs.to(torch.int32), cfg)


def grouped_mm(x: torch.Tensor, w_t: torch.Tensor, offs: torch.Tensor):
    """``torch._grouped_mm(x, w_t, offs=offs)`` that reaches a converted weight in a traced graph
    too.  Eagerly the weight's ``__torch_function__`` sees ``torch._grouped_mm``; Dynamo offers it
    only the functions ``torch.overrides.get_overridable_functions()`` lists, which leaves out
    underscore names, so a traced ``torch._grouped_mm`` on a converted weight would run in bf16
    without a word.  Code that may be compiled calls this instead."""
    if (torch.compiler.is_compiling() and isinstance(w_t, MXFP8TrainingWeight)
            and not isinstance(x, MXFP8TrainingWeight)):
        from .compiled import mx_grouped_mm_traced

        cfg = w_t.mx_config
        with torch._C.DisableTorchFunctionSubclass():
            return mx_grouped_mm_traced(x, w_t, offs, cfg.scale_mode, cfg.pad_token_groups_for_grouped_mm)
    return torch._grouped_mm(x, w_t, offs=offs)


# ----------------------------------------------------------------------------- the wrapper
_LINEAR_FUNCS = {F.linear}
_GROUPED_FUNCS = {torch._grouped_mm}


def _unwrap(t):
    return t.as_subclass(torch.Tensor) if isinstance(t, MXFP8TrainingWeight) else t


class MXFP8TrainingWeight(torch.Tensor):
    """A high-precision weight whose GEMMs run in MXFP8.

    Shares storage with the tensor it was made from (like ``nn.Parameter``), so in-place
    initialisation and optimizer updates act on the real weight.  Every op other than
    ``F.linear`` / ``torch._grouped_mm`` behaves as for a plain tensor, and results that are
    views or casts of the weight stay wrapped so that ``w.bfloat16().transpose(-2, -1)`` still
    reaches the grouped kernel.
    """

    mx_config: MXFP8Config = MXFP8Config()

    @staticmethod
    def __new__(cls, data: torch.Tensor, config: MXFP8Config | None = None):
        t = torch.Tensor._make_subclass(cls, data, data.requires_grad)
        t.mx_config = config or MXFP8Config()
        return t

    def __repr__(self):
        return f"MXFP8TrainingWeight({self.as_subclass(torch.Tensor)!r}, config={self.mx_config!r})"

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        kwargs = kwargs or {}
        if func in _LINEAR_FUNCS:
            x = args[0]
            w = args[1] if len(args) > 1 else kwargs["weight"]
            b = args[2] if len(args) > 2 else kwargs.get("bias")
            if isinstance(w, cls) and not isinstance(x, cls):
                if torch.compiler.is_compiling():
                    # a tracer cannot follow the eager path's library calls: the linear enters
                    # the graph as one opaque operator (torchtitan_amd/compiled.py)
                    from .compiled import mx_linear_traced

                    with torch._C.DisableTorchFunctionSubclass():
                        return mx_linear_traced(x, w, b, w.mx_config.scale_mode, w.mx_config.cache_weight_casts)
                cfg = w.mx_config
                if cfg.cache_weight_casts:
                    with torch._C.DisableTorchFunctionSubclass():
                        frozen = not w.requires_grad
                    return mx_linear(x, _unwrap(w), _unwrap(b), cfg, frozen)
                return mx_linear(x, _unwrap(w), _unwrap(b), cfg)
        elif func in _GROUPED_FUNCS:
            a, b = args[0], args[1]
            offs = kwargs.get("offs", args[2] if len(args) > 2 else None)
            if isinstance(b, cls) and not isinstance(a, cls):
                if torch.compiler.is_compiling():  # as for the linear: one opaque operator
                    from .compiled import mx_grouped_mm_traced

                    with torch._C.DisableTorchFunctionSubclass():
                        return mx_grouped_mm_traced(a, b, offs, b.mx_config.scale_mode,
                                                    b.mx_config.pad_token_groups_for_grouped_mm)
                return mx_grouped_mm(a, _unwrap(b), offs, b.mx_config)
        cfg = next((a.mx_config for a in _flatten(args) if isinstance(a, cls)), None)
        with torch._C.DisableTorchFunctionSubclass():
            out = func(*args, **kwargs)
        return _rewrap(out, cls, cfg, func)

    # pickling: the plain tensor plus the config (and whether it was a Parameter)
    def __reduce_ex__(self, proto):
        plain = self.as_subclass(torch.Tensor)
        if getattr(self, "_is_param", False):
            return (_rebuild_parameter, (plain.detach(), self.mx_config, self.requires_grad))
        return (MXFP8TrainingWeight, (plain, self.mx_config))

    def __deepcopy__(self, memo):
        """An independent copy that is still a converted weight (and still a Parameter if this
        one is): what ``copy.deepcopy(model)`` needs, e.g. when a trainer clones a converted model
        per pipeline stage."""
        if id(self) in memo:
            return memo[id(self)]
        data = self.as_subclass(torch.Tensor).detach().clone(memory_format=torch.preserve_format)
        out = MXFP8TrainingWeight(data, self.mx_config)
        if getattr(self, "_is_param", False):
            out = _as_parameter(data, self.mx_config, self.requires_grad)
        else:
            out.requires_grad_(self.requires_grad)
        memo[id(self)] = out
        return out


def _as_parameter(data: torch.Tensor, cfg: MXFP8Config, requires_grad: bool) -> "MXFP8TrainingWeight":
    """A converted weight that is an ``nn.Parameter`` (``isinstance`` holds through the
    ``_is_param`` mark ``nn.Parameter`` itself puts on tensor subclasses), sharing `data`'s
    storage.  Built directly rather than through ``nn.Parameter(wrapper)``: that detaches the
    wrapper, and the result is a view whose base keeps the dtype and device of conversion time
    when ``module.to(...)`` later swaps the parameter's data -- a tracer that checks a tensor's
    base against its fake twin then refuses the parameter."""
    t = torch.Tensor._make_subclass(MXFP8TrainingWeight, data, requires_grad)
    t.mx_config = cfg
    t._is_param = True
    return t


def _rebuild_parameter(data: torch.Tensor, cfg: MXFP8Config, requires_grad: bool):
    return _as_parameter(data, cfg, requires_grad)


# views, casts, detach and clone of a weight are still that weight, and so is the storage that
# `Module.to_empty` gives a meta-device parameter (torch.empty_like); zeros_like and the other
# factory functions (optimizer state) make plain tensors
_KEEP_WRAPPED = {
    torch.Tensor.transpose, torch.Tensor.t, torch.Tensor.bfloat16, torch.Tensor.to,
    torch.Tensor.detach, torch.Tensor.requires_grad_, torch.Tensor.contiguous,
    torch.Tensor.view, torch.Tensor.reshape, torch.Tensor.float, torch.Tensor.half,
    torch.transpose, torch.empty_like, torch.Tensor.clone, torch.clone,
    torch.Tensor.cuda, torch.Tensor.cpu, torch.Tensor.type,
}


def _flatten(args):
    for a in args:
        if isinstance(a, (list, tuple)):
            yield from _flatten(a)
        else:
            yield a


def _rewrap(out, cls, cfg, func):
    """Results of view / cast / clone style ops on a wrapped weight stay wrapped; in-place ops
    return their (already wrapped) input; everything else is a plain tensor."""
    if cfg is None or func not in _KEEP_WRAPPED:
        return out
    if isinstance(out, torch.Tensor) and not isinstance(out, cls):
        wrapped = out.as_subclass(cls)
        wrapped.mx_config = cfg
        return wrapped
    return out


def wrap_parameter(param: torch.nn.Parameter, cfg: MXFP8Config) -> torch.nn.Parameter:
    """A Parameter of type MXFP8TrainingWeight sharing `param`'s storage."""
    if isinstance(param.data, MXFP8TrainingWeight) or isinstance(param, MXFP8TrainingWeight):
        return param
    return _as_parameter(param.data, cfg, param.requires_grad)
