"""Host-side logic of torchtitan_amd.ops that needs no GPU: operand pitches, shape gates."""
import pytest
import torch

from torchtitan_amd import ops
from torchtitan_amd.ops import MXData, MX_SCALES_MFMA, MX_SCALES_ROWMAJOR


def _codes(rows, cols, pad=0):
    return torch.zeros((rows, cols + pad), dtype=torch.uint8)[:, :cols]


def test_common_pitch_keeps_one_pitch_and_copies_when_they_differ():
    a, b = _codes(64, 256, 128), _codes(32, 256, 128)
    (ra, rb), ld = ops._common_pitch(a, b)
    assert ld == 384 and ra.data_ptr() == a.data_ptr() and rb.data_ptr() == b.data_ptr()
    # dense operands stay as they are
    (ra, rb), ld = ops._common_pitch(_codes(64, 256), _codes(32, 256))
    assert ld == 256 and ra.is_contiguous() and rb.is_contiguous()
    # differing pitches: dense copies of both
    (ra, rb), ld = ops._common_pitch(a, _codes(32, 256))
    assert ld == 256 and ra.is_contiguous() and rb.is_contiguous() and ra.data_ptr() != a.data_ptr()
    # a pitch the persistent kernel does not take (not a multiple of 128) unless the caller allows it
    c, d = _codes(64, 256, 16), _codes(32, 256, 16)
    (rc, rd), ld = ops._common_pitch(c, d)
    assert ld == 256 and rc.is_contiguous()
    (rc, rd), ld = ops._common_pitch(c, d, multiple=16)
    assert ld == 272 and rc.data_ptr() == c.data_ptr()
    # a transposed view is not an operand as it stands
    t = torch.zeros((256, 64), dtype=torch.uint8).t()
    (rt, _), ld = ops._common_pitch(t, _codes(32, 256))
    assert rt.is_contiguous() and ld == 256


def test_code_rows_and_pitch_rule():
    c = ops._code_rows(96, 160, 128, "cpu")
    assert c.shape == (96, 160) and c.stride() == (288, 1)
    s = ops._code_rows(96, 160, 128, "cpu", stack=2)
    assert s.shape == (2, 96, 160) and s.stride() == (96 * 288, 288, 1)
    assert ops._code_rows(96, 160, 0, "cpu").is_contiguous()
    assert ops._pitch_ok(128) == 128 and ops._pitch_ok(16) == 16
    assert ops._pitch_ok(0) == 0 and ops._pitch_ok(8) == 0 and ops._pitch_ok(-128) == 0


def test_unpadded_output_gate():
    def data(rows, cols, order, stack=0):
        shape = (stack, rows, cols) if stack else (rows, cols)
        return MXData(torch.zeros(shape, dtype=torch.uint8), torch.zeros(1, dtype=torch.uint8), order)

    a, b = data(256, 256, MX_SCALES_MFMA), data(128, 256, MX_SCALES_MFMA, stack=4)
    assert ops.rows_out_supported(a, b)
    assert ops.rows_out_supported(a, b, a, b)
    assert not ops.rows_out_supported(a, b, a, None)                                  # half a second operand set
    assert not ops.rows_out_supported(data(256, 256, MX_SCALES_ROWMAJOR), b)          # row-major scales
    assert not ops.rows_out_supported(data(256, 160, MX_SCALES_MFMA), data(128, 160, MX_SCALES_MFMA, stack=4))  # K % 128
    assert not ops.rows_out_supported(data(240, 256, MX_SCALES_MFMA), b)              # T % 32
    assert not ops.rows_out_supported(a, data(128, 256, MX_SCALES_MFMA, stack=ops.FAST_MAX_GROUPS + 1))
    with pytest.raises(ValueError):
        ops.mx_grouped_gemm_2d3d_rows_out(data(256, 256, MX_SCALES_ROWMAJOR), b, torch.zeros(4, dtype=torch.int32),
                                          torch.zeros(4, dtype=torch.int32), 200)
    with pytest.raises(ValueError):  # more output rows than padded rows
        ops.mx_grouped_gemm_2d3d_rows_out(a, b, torch.zeros(4, dtype=torch.int32), torch.zeros(4, dtype=torch.int32), 300)
    with pytest.raises(ValueError):  # int64 group ends
        ops.mx_grouped_gemm_2d3d_rows_out(a, b, torch.zeros(4, dtype=torch.int64), torch.zeros(4, dtype=torch.int32), 200)


def test_block_pitch_is_for_training_steps_without_cached_weight_casts():
    from torchtitan_amd.mx_blocks import block_pitch_pad
    from torchtitan_amd.mx_tensor import MXFP8Config

    cfg = MXFP8Config()
    assert block_pitch_pad(cfg, True, True) == ops.CODE_PITCH_PAD
    assert block_pitch_pad(cfg, True, False) == 0 and block_pitch_pad(cfg, False, True) == 0
    cached = MXFP8Config(cache_weight_casts=True)
    assert block_pitch_pad(cached, True, True) == 0


@pytest.fixture
def no_launches(monkeypatch):
    """Everything around the library calls, on the CPU: no call is made and outputs keep what they held."""
    from torchtitan_amd import mx_tensor

    monkeypatch.setattr(ops, "_call", lambda *args: None)
    monkeypatch.setattr(ops, "_stream", lambda t: 0)
    monkeypatch.setattr(ops, "_operand_input", lambda x, f32_ok=False: x)
    monkeypatch.setattr(ops, "_check_hp", lambda x: x)
    monkeypatch.setattr(ops, "_split_workspace", lambda *args: None)
    mx_tensor._weight_cache.clear()
    mx_tensor.clear_cast_cache()
    yield
    mx_tensor._weight_cache.clear()
    mx_tensor.clear_cast_cache()


def _bf16(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


# contractions that round up to the same whole blocks, and the same ones
@pytest.mark.parametrize("wrong,right", [(2016, 2048), (32, 128), (1920, 2016), (2048, 2048)])
def test_products_compare_the_contraction_before_it_is_rounded_up(no_launches, wrong, right):
    operand = lambda rows, depth, pad=128: ops.to_operands(_bf16(rows, depth), "rceil", True, False, pad)[0]
    for M in (16, 200):
        x, x2, w, w2 = operand(M, wrong), operand(M, wrong), operand(256, right), operand(256, right)
        calls = [lambda: ops.mx_gemm_nt(x, w), lambda: ops.mx_gemm_nt(x, w, _bf16(M, 256)),
                 lambda: ops.mx_gemm_nt(x, operand(256, right, 0)), lambda: ops.mx_gemm_nt_pair(x, w, x2, w2),
                 lambda: ops.mx_gemm_nt_pair(w, w2, w, operand(256, wrong)),
                 lambda: ops.mx_gemm_nt_shared_a(x, w, w2), lambda: ops.mx_gemm_nt_shared_a(x, operand(256, wrong), w),
                 lambda: ops.mx_gemm_nt_shared_b(x, x2, w), lambda: ops.mx_gemm_nt_shared_b(w, operand(256, wrong), w2),
                 lambda: ops.mx_few_rows(_bf16(16, wrong), w),
                 lambda: ops.mx_few_rows(_bf16(16, right), w, "floor", operand(256, wrong))]
        for call in calls:
            if wrong == right:
                call()
            else:
                with pytest.raises(ValueError):
                    call()


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("tokens", [16, 200])
def test_mismatched_modules_raise(no_launches, monkeypatch, grad, tokens):
    from torchtitan_amd import mx_blocks, mx_tensor

    cfg = mx_tensor.MXFP8Config()
    x = _bf16(tokens, 2016)
    monkeypatch.setattr(ops, "few_rows_ok", lambda t, columns: t.shape[0] <= ops.FEW_ROWS)
    weight = lambda *shape: mx_tensor.MXFP8TrainingWeight(_bf16(*shape).requires_grad_(grad), cfg)
    mismatched = (lambda: mx_tensor.mx_linear(x, weight(512, 2048).as_subclass(torch.Tensor), None, cfg),
                  lambda: mx_blocks.mx_feed_forward(x, weight(2048, 2048), weight(2016, 2048), weight(2048, 2048)),
                  lambda: mx_blocks.mx_feed_forward(x, weight(2016, 2016), weight(2016, 2048), weight(2016, 2016)),
                  lambda: mx_blocks.mx_swiglu_linear(x, x, weight(512, 2048)))
    with torch.set_grad_enabled(grad):
        for call in mismatched:
            with pytest.raises(ValueError, match="contraction|same shape"):
                call()
        mx_blocks.mx_feed_forward(x, weight(2048, 2016), weight(2016, 2048), weight(2048, 2016))


def test_a_cached_cast_is_given_in_the_form_its_caller_wants(no_launches):
    from torchtitan_amd import mx_tensor

    cfg = mx_tensor.MXFP8Config(cache_weight_casts=True)
    w = _bf16(128, 384)
    cast = lambda whole: mx_tensor._cast_weight(w, "rceil", True, cfg, whole_blocks=whole)
    dense = cast(False)
    for q in dense:
        q.codes.random_(0, 255), q.scales.random_(0, 255)
    whole = cast(True)  # a copy, which takes the dense entry's place
    for q, d in zip(whole, dense):
        assert type(q) is ops.Operand and type(d) is MXData and q.depth == d.codes.shape[1]
        assert torch.equal(q.codes, d.codes) and torch.equal(q.scales, d.scales) and q.codes.is_contiguous()
    assert cast(True)[0] is whole[0] and len(mx_tensor._weight_cache) == 1
    for q, d in zip(cast(False), dense):  # and serves both
        assert type(q) is MXData and torch.equal(q.codes, d.codes) and torch.equal(q.scales, d.scales)
    with pytest.raises(ValueError):
        ops.Operand.of(MXData(_codes(128, 160), torch.zeros(1280, dtype=torch.uint8), MX_SCALES_MFMA))


@pytest.mark.parametrize("tokens,dim,hidden,norm", [(64, 128, 256, False), (96, 160, 224, False), (160, 256, 416, True)])
@pytest.mark.parametrize("need_dx,need_dw", [(True, True), (True, False), (False, True)])
def test_traced_block_has_the_shapes_that_its_fake_kernel_gives(no_launches, monkeypatch, tokens, dim, hidden, norm, need_dx,
                                                               need_dw):
    """The operators' bodies with the launches left out against their fake kernels, forward and backward."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from torchtitan_amd import compiled, mx_blocks

    monkeypatch.setattr(mx_blocks, "_rms_norm_backward",  # (torch's own is for the GPU)
                        lambda dx, x, rstd, w, need_x, need_w: (dx if need_x else None, w.clone() if need_w else None))

    def run(fwd, bwd):
        x, w1, w2, w3 = _bf16(tokens, dim), _bf16(hidden, dim), _bf16(dim, hidden), _bf16(hidden, dim)
        n = torch.ones(dim, dtype=torch.bfloat16) if norm else None
        out = fwd(x, w1, w2, w3, n, 1e-5, 1, False, need_dx, need_dw)
        return *out, *bwd(_bf16(tokens, dim), list(out[1:]), x if norm else None, n, 1, need_dx, need_dw, need_dw, need_dw,
                          norm and need_dx)

    real = run(compiled.mx_ffn_fwd._init_fn, compiled.mx_ffn_bwd._init_fn)
    with FakeTensorMode():
        fake = run(torch.ops.torchtitan_amd.mx_ffn_fwd, torch.ops.torchtitan_amd.mx_ffn_bwd)
    assert [t.shape for t in real] == [t.shape for t in fake] and [t.dtype for t in real] == [t.dtype for t in fake]
    storages = [t.untyped_storage().data_ptr() for t in real[1:15] if t.numel()]
    assert len(set(storages)) == len(storages)


@pytest.mark.parametrize("T,rows", [(192, 512), (704, 1664), (705, 1664), (1984, 4096), (4032, 8192), (6080, 12416)])
def test_traced_experts_have_the_padded_length_of_the_plan(T, rows):
    """The fake kernels' layouts at bounds of whole 512s: an additional block, but for powers of two."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    A, D, H, G, k = torch.ops.torchtitan_amd, 128, 256, 4, 2
    with FakeTensorMode():
        x, e1, e2 = _bf16(T, D), torch.empty(G, H, D), torch.empty(G, D, H)
        scores, order, counts = torch.empty(T, k), torch.empty(T * k, dtype=torch.int64), torch.empty(G, dtype=torch.int64)
        out = A.mx_routed_experts_fwd(x, scores, e1, e2, e1, order, counts, True, 1, False, True, True, True)
        assert out[6].shape == (2, rows, H)
        offs, pairs = torch.empty(G, dtype=torch.int32), _bf16(T * k, D)
        assert A.mx_grouped_ffn_fwd(pairs, e1, e2, e1, offs, 1, True, False, True, True)[4].shape == (2, rows, H)
        assert A.mx_grouped_mm_fwd(pairs, e1, offs, 1, True)[4].shape == (D, rows)


@pytest.mark.parametrize("need_dx,need_dw", [(True, True), (True, False), (False, True)])
def test_traced_linear_has_the_shapes_that_its_fake_kernel_gives(no_launches, need_dx, need_dw):
    """... also where the weight is frozen, or the input takes no gradient: what is not kept comes to the backward empty."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from torchtitan_amd import compiled

    def run(fwd, bwd):
        out = fwd(_bf16(2, 96, 160), _bf16(224, 160), 1, need_dx, need_dw, False)
        return *out, *bwd(_bf16(2, 96, 224), *out[1:], 1, need_dx, need_dw)

    real = run(compiled.mx_linear_fwd._init_fn, compiled.mx_linear_bwd._init_fn)
    with FakeTensorMode():
        fake = run(torch.ops.torchtitan_amd.mx_linear_fwd, torch.ops.torchtitan_amd.mx_linear_bwd)
    assert [t.shape for t in real] == [t.shape for t in fake] and [t.dtype for t in real] == [t.dtype for t in fake]
    assert real[5].shape == ((192, 160) if need_dx else (0,)) and real[6].shape == ((224, 160) if need_dw else (0,))


def test_remembered_activation_cast_stays_on_its_stream(no_launches, monkeypatch):
    """A sibling on the stream that cast the activation takes the codes; one on another stream, whose work is not
    ordered behind that launch, or in another graph capture casts again."""
    from torchtitan_amd import mx_tensor

    place = (0x10, 0)
    monkeypatch.setattr(mx_tensor, "_place", lambda t: place, raising=False)
    x = _bf16(200, 256)
    cast = lambda: mx_tensor._cast_activation(x, x, "rceil", True)
    first = cast()
    assert cast() is first
    for place in ((0x20, 0), (0x20, 1), (0x20, 2), (0x10, 2), (0x10, 0)):
        again = cast()
        assert again is not first and cast() is again
        first = again
    x.add_(1)
    assert cast() is not first


def test_remembered_activation_cast_is_read_and_dropped_as_a_whole(no_launches):
    """Threads that remember, look up and drop entries: a lookup gives the cast of its own tensor or nothing."""
    import sys
    import threading

    from torchtitan_amd import mx_tensor

    cache, wrong = mx_tensor._ActivationCastCache(), []

    def work(i):
        xs = [_bf16(1, 32) for _ in range(4)]
        try:
            for n in range(20000):
                x = xs[n % 4]
                cache.put(x, i, (i, n % 4))
                got = cache.get(x, i)
                if got not in (None, (i, n % 4)):
                    wrong.append(got)
                if n % 3 == 0:
                    cache.clear()
        except Exception as ex:  # (a thread's own exception would pass unnoticed)
            wrong.append(ex)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)  # between any two steps of a lookup
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not wrong


@pytest.mark.parametrize("cached", [False, True])
def test_a_forward_without_gradients_casts_each_operand_once(no_launches, monkeypatch, cached):
    """... also where the native call hands its input back, and where a sibling linear has cast the activation."""
    from torchtitan_amd import _lib, mx_tensor

    class Blocks:
        handed_back = 0

        def linear_apply(self, *args):
            self.handed_back += 1

    blocks, casts = Blocks(), []
    monkeypatch.setattr(_lib, "blocks", lambda: blocks)
    monkeypatch.setattr(ops, "native_block_ok", lambda *args: True)
    monkeypatch.setattr(ops, "_call", lambda name, tag, device, *args: casts.append((name, args[0])))
    cfg = mx_tensor.MXFP8Config(cache_weight_casts=cached)
    x, weights = _bf16(200, 256), [_bf16(384, 256), _bf16(160, 256)]
    for w in weights:
        mx_tensor._linear_forward(x, w, cfg, False, False)
    casts = [pointer for name, pointer in casts if name == "mx_cast_pad" or name.startswith("mx_cast_dim")]
    assert blocks.handed_back == 1  # (the second linear takes the activation's cast as it is)
    assert sorted(casts) == sorted(t.data_ptr() for t in (x, *weights))


@pytest.mark.parametrize("pairs", [0, 1, 96, 127, 128, 129, 352, 383, 384, 385, 480, 481, 131072, 12983 * 8])
@pytest.mark.parametrize("experts", [1, 8, 128])
def test_padded_layouts_of_whole_blocks_are_no_whole_512s(pairs, experts):
    """A bound of the aligned groups, at most two blocks beyond it, whose rows of column-wise codes do not lie 4 KB apart,
    unless they are a power of two below 65536 (where the additional block costs more than it gives)."""
    need, got = pairs + 32 * experts, ops.plan_length(pairs, experts, 32, 128)
    power = got in (512, 1024, 2048, 4096, 8192, 16384, 32768)
    assert got % 128 == 0 and (got % 512 or power) and need <= got < need + 256
    assert got < need + 128 or (got - 128) % 512 == 0
    assert ops.plan_length(pairs, experts, 32) == need + -need % 32


@pytest.mark.parametrize("need,rows", [(384, 384), (385, 512), (512, 512), (1536, 1664), (4000, 4096), (8192, 8192),
                                       (12288, 12416), (32768, 32768), (65536, 65664), (135168, 135296)])
def test_padded_lengths_by_the_bound_of_their_groups(need, rows):
    assert ops.plan_length(need - 32 * 4, 4, 32, 128) == rows


def _frozen_readers(path, weights, norm):
    """The ways in which a program reads the frozen weights of a linear, of a SwiGLU block or of linears behind a norm:
    calls that take whether gradients flow through the weights."""
    from torchtitan_amd import compiled, mx_blocks, mx_tensor

    w1, w2, w3 = weights
    (H, D), mode = w1.shape, ops.SCALE_MODES["rceil"]
    plain = [w.as_subclass(torch.Tensor) for w in weights]

    def x(grad, cols=D):
        return _bf16(160, cols).requires_grad_(grad)

    def block_of_norm(grad):
        return mx_blocks.mx_norm_feed_forward(x(grad), norm, 1e-5, w1, w2, w3)

    return {
        "linear": ((w1,), lambda grad: mx_tensor.mx_linear(x(grad), plain[0], None, w1.mx_config, True),
                   lambda grad: compiled.mx_linear_fwd._init_fn(x(False), plain[0], mode, grad, False, True)),
        "block": (weights, lambda grad: mx_blocks.mx_feed_forward(x(grad), w1, w2, w3), block_of_norm,
                  lambda grad: compiled.mx_ffn_fwd._init_fn(x(False), *plain, None, 1e-5, mode, True, grad, False),
                  lambda grad: compiled.mx_ffn_fwd._init_fn(x(False), *plain, norm, 1e-5, mode, True, grad, False)),
        "norm and linears": ((w1, w3), lambda grad: mx_blocks.mx_norm_linears(x(grad), norm, 1e-5, (w1, w3)),
                             lambda grad: mx_tensor.mx_linear(x(grad), plain[0], None, w1.mx_config, True)),
        "gate and linear": ((w2,), lambda grad: mx_blocks.mx_swiglu_linear(x(grad, H), x(grad, H), w2)),
    }[path]


@pytest.mark.parametrize("path,reader", [("linear", 0), ("linear", 1), ("block", 0), ("block", 1), ("block", 2), ("block", 3),
                                         ("norm and linears", 0), ("gate and linear", 0)])
@pytest.mark.parametrize("grad", [False, True])
def test_a_frozen_weight_is_cast_once_whoever_reads_it(no_launches, monkeypatch, path, reader, grad):
    """Every forward on cached casts of frozen weights takes the entry that another one has made, with gradients through
    it or without: each form of a weight is cast once, and no weight has two entries."""
    from torchtitan_amd import mx_tensor

    cfg = mx_tensor.MXFP8Config(cache_weight_casts=True)
    weights = [mx_tensor.MXFP8TrainingWeight(_bf16(*shape), cfg) for shape in ((256, 384), (384, 256), (256, 384))]
    used, *readers = _frozen_readers(path, weights, torch.ones(384, dtype=torch.bfloat16))
    casts = []

    def call(name, tag, device, *args):
        if name == "mx_cast_pad":
            casts.extend((args[0], form) for form, at in (("rows", 5), ("columns", 8)) if args[at] is not None)
        elif name in ("mx_cast_dim0", "mx_cast_dim0_dim1", "mx_cast_dim0_dim1_ld"):
            casts.extend((args[0], form) for form in ("rows", "columns")[:1 if name == "mx_cast_dim0" else 2])

    def read(i, grad):
        with torch.set_grad_enabled(grad):
            return readers[i](grad)

    monkeypatch.setattr(ops, "_call", call)
    read(reader, grad)
    for again in (False, True, False):
        for i in range(len(readers)):
            read(i, again)
    own = {w.data_ptr() for w in used}
    assert sorted(c for c in casts if c[0] in own) == sorted((p, form) for p in own for form in ("rows", "columns"))
    assert len(mx_tensor._weight_cache) == len(used)
    with torch.no_grad():  # (an update leaves no entry of the old values behind)
        for w in used:
            w.add_(1)
    read(0, True), read(0, False)
    assert len(mx_tensor._weight_cache) == len(used)


def test_operands_of_a_frozen_weight_agree_on_their_pitch(no_launches):
    """... so that no product makes copies of them: forward and backward through an entry with rows apart."""
    from torchtitan_amd import mx_blocks, mx_tensor

    cfg, seen = mx_tensor.MXFP8Config(cache_weight_casts=True), []
    weights = [mx_tensor.MXFP8TrainingWeight(_bf16(*shape), cfg) for shape in ((256, 384), (384, 256), (256, 384))]
    product = ops._operands
    try:
        ops._operands = lambda *qs: seen.append(product(*qs)) or seen[-1]
        with torch.no_grad():  # (makes the entries)
            mx_blocks.mx_feed_forward(_bf16(160, 384), *weights)
        h = torch.zeros(160, 256, dtype=torch.bfloat16, requires_grad=True)
        for run in (lambda x: mx_blocks.mx_feed_forward(x, *weights),
                    lambda x: mx_tensor.mx_linear(x, weights[0].as_subclass(torch.Tensor), None, cfg, True),
                    lambda x: mx_blocks.mx_swiglu_linear(h, h, weights[1])):
            x = torch.zeros(160, 384, dtype=torch.bfloat16, requires_grad=True)
            y = run(x)
            y.backward(torch.zeros_like(y))
    finally:
        ops._operands = product
    assert seen and all(seen)
    assert all(e[5].ld == e[5].k + ops.CODE_PITCH_PAD and e[6].ld == e[6].k + ops.CODE_PITCH_PAD
               for e in mx_tensor._weight_cache._entries.values())
