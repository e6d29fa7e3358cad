"""Linears, SwiGLU blocks and routed experts whose launches come from one native call (csrc/host/blocks.cpp) against
the general path over the forms that the call accepts, and those that it hands back: bit for bit, results and gradients."""
import pytest
import torch
import torch.nn as nn

from tests.test_converter_gpu import _convert
from torchtitan_amd import _lib, mx_tensor, ops
from torchtitan_amd.modules import FeedForward, Linear
from torchtitan_amd.modules.moe import MoE

pytestmark = pytest.mark.gpu


class _Counted:
    """The native module with the calls that it took, by name."""

    def __init__(self, module):
        self._module, self.taken = module, []

    def __getattr__(self, name):
        fn = getattr(self._module, name)

        def call(*args):
            out = fn(*args)
            if out is not None:
                self.taken.append(name)
            return out
        return call


def _both(monkeypatch, fn):
    """(fn() on native calls, fn() on the general path, names of the native calls taken)."""
    counted = _Counted(_lib.blocks())
    mx_tensor.clear_cast_cache()
    with monkeypatch.context() as m:
        m.setattr(_lib, "blocks", lambda: counted)
        native = fn()
    mx_tensor.clear_cast_cache()
    with monkeypatch.context() as m:
        m.setattr(ops, "native_block_ok", lambda *a: False)
        general = fn()
    return native, general, counted.taken


def _same(a, b):
    for i, (x, y) in enumerate(zip(a, b, strict=True)):
        assert x.dtype == y.dtype and x.shape == y.shape, i
        assert torch.equal(x, y), i


def _step(block, params, x, dy, autocast=False, hooks=None):
    x = x.detach().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast), hooks() if hooks else torch.enable_grad():
        y = block(x)
    return [y.detach(), *torch.autograd.grad(y, [x, *params], dy)]


def _holder(module, device, dtype=torch.bfloat16, **kw):
    holder = nn.Module()
    holder.block = module
    holder.to(device).to(dtype)
    for p in module.parameters():
        nn.init.normal_(p, 0.0, 0.02)
    _convert(holder, ["block"], **kw)
    return module


FORMS = {  # from randn(*shape), which has the device and the type: a copy to either would lay the rows out anew
    "plain": lambda randn, t, w: randn(t, w),
    "rows of a wider matrix": lambda randn, t, w: randn(t, w + 64)[:, :w],
    "rows that are not aligned": lambda randn, t, w: randn(t, w + 3)[:, 3:],
    "columns first": lambda randn, t, w: randn(w, t).t(),
    "one row for all": lambda randn, t, w: randn(1, w).expand(t, w),
    "three dimensions": lambda randn, t, w: randn(1, t, w),
}


def _form(form, device, dtype, tokens, width):
    return FORMS[form](lambda *shape: torch.randn(shape, device=device, dtype=dtype), tokens, width)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("tokens,inner,outer", [(1, 160, 256), (33, 256, 160), (129, 512, 384), (300, 160, 144), (700, 384, 1056)])
@pytest.mark.parametrize("params", ["bfloat16", "float32"])
def test_linear(device, monkeypatch, form, tokens, inner, outer, params):
    torch.manual_seed(tokens + inner)
    dtype = getattr(torch, params)
    lin = _holder(Linear.Config().build(in_features=inner, out_features=outer), device, dtype)
    x, dy = _form(form, device, dtype, tokens, inner), _form(form, device, torch.bfloat16, tokens, outer)
    run = lambda: _step(lin, [lin.weight], x, dy, autocast=params == "float32")
    native, general, taken = _both(monkeypatch, run)
    _same(native, general)
    if form in ("plain", "rows of a wider matrix", "three dimensions"):
        assert "linear_forward" in taken and ("linear_backward" in taken) == (outer % 32 == 0)
    with torch.no_grad():
        native, general, taken = _both(monkeypatch, lambda: [lin(x) if params == "bfloat16" else lin(x.bfloat16())])
    _same(native, general)


@pytest.mark.parametrize("tokens", [1, 32, 33, 64, 65, 300])
@pytest.mark.parametrize("cached", [True, False])
def test_linear_without_gradients(device, monkeypatch, tokens, cached):
    lin = _holder(Linear.Config().build(in_features=2176, out_features=288), device, cache=cached)
    x = torch.randn(tokens, 2176, device=device, dtype=torch.bfloat16)
    with torch.no_grad():
        native, general, taken = _both(monkeypatch, lambda: [lin(x), lin(x)])
    _same(native, general)
    assert "linear_apply" in taken


@pytest.mark.parametrize("tokens,dtype", [(16, torch.float32), (16, torch.bfloat16), (200, torch.bfloat16)])
@pytest.mark.parametrize("form", ["plain", "rows that are not aligned"])
def test_siblings_without_gradients(device, monkeypatch, tokens, dtype, form):
    """Linears on one activation cast it once, but for the few bf16 rows that are cast inside their products, and their
    weights once each."""
    lins = [_holder(Linear.Config().build(in_features=256, out_features=n), device) for n in (384, 160, 160)]
    x, weights = _form(form, device, dtype, tokens, 256), []
    cast = mx_tensor._cast_weight
    monkeypatch.setattr(mx_tensor, "_cast_weight", lambda w, *args, **kw: weights.append(w.shape[0]) or cast(w, *args, **kw))
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == torch.float32):
        native, general, taken = _both(monkeypatch, lambda: [lin(x) for lin in lins])
    _same(native, general)
    assert weights == 2 * [384, 160, 160]
    few = tokens <= ops.FEW_ROWS and dtype == torch.bfloat16
    assert taken == (["linear_apply"] * (3 if few else 1) if form == "plain" else [])


def test_siblings_and_frozen_weights(device, monkeypatch):
    """Linears on one activation share its cast whichever path made it; a frozen weight leaves the native call out."""
    a = _holder(Linear.Config().build(in_features=256, out_features=384), device)
    b = _holder(Linear.Config().build(in_features=256, out_features=160), device)
    x0 = torch.randn(130, 256, device=device, dtype=torch.bfloat16)

    def both():
        x = x0.detach().requires_grad_(True)
        ya, yb = a(x), b(x)
        grads = torch.autograd.grad(ya.sum() + yb.sum(), [x, a.weight, b.weight])
        return [ya.detach(), yb.detach(), *grads]
    native, general, taken = _both(monkeypatch, both)
    _same(native, general)
    assert taken.count("linear_forward") == 1
    b.weight.requires_grad_(False)

    def frozen():
        x = x0.detach().requires_grad_(True)
        y = b(x)
        return [y.detach(), *torch.autograd.grad(y.float().sum(), [x])]
    native, general, taken = _both(monkeypatch, frozen)
    _same(native, general)
    assert taken == []


@pytest.mark.parametrize("form", ["plain", "rows of a wider matrix", "columns first", "three dimensions"])
@pytest.mark.parametrize("tokens,dim,hidden", [(33, 160, 256), (129, 256, 160), (300, 384, 544)])
def test_feed_forward(device, monkeypatch, form, tokens, dim, hidden):
    torch.manual_seed(tokens)
    ff = _holder(FeedForward.Config(hidden_dim=hidden).build(dim=dim), device)
    x, dy = (_form(form, device, torch.bfloat16, tokens, dim) for _ in range(2))
    run = lambda: _step(ff, list(ff.parameters()), x, dy)
    native, general, taken = _both(monkeypatch, run)
    _same(native, general)
    if form != "columns first":
        assert taken == ["ffn_forward", "ffn_backward"]
    # saved tensors that come back as other tensors
    native, general, taken = _both(monkeypatch, lambda: _step(ff, list(ff.parameters()), x, dy, hooks=lambda: torch.autograd.graph.save_on_cpu()))
    _same(native, general)


@pytest.mark.parametrize("before", [True, False])
@pytest.mark.parametrize("experts,top_k,shared,tokens", [(1, 1, 0, 40), (8, 2, 1, 200), (16, 4, 0, 37)])
def test_routed_experts(device, monkeypatch, experts, top_k, shared, tokens, before):
    torch.manual_seed(tokens)
    moe = MoE(MoE.Config(num_experts=experts, num_shared_experts=shared, hidden_dim=256, top_k=top_k, score_func="softmax",
                         score_before_experts=before, route_norm=True), dim=384).to(device).to(torch.bfloat16)
    moe.init_weights(init_std=0.02, buffer_device=device)
    holder = nn.Module()
    holder.moe = moe
    _convert(holder, ["experts"])
    x, dy = (torch.randn(1, tokens, 384, device=device, dtype=torch.bfloat16) for _ in range(2))

    def run():
        moe.tokens_per_expert.zero_()
        return [*_step(moe, list(moe.parameters()), x, dy), moe.tokens_per_expert.clone()]
    native, general, taken = _both(monkeypatch, run)
    _same(native, general)
    if experts % 8 == 0:  # (the gate's and the router's own kernels, whose choices the call takes)
        assert "routed_forward" in taken and "routed_backward" in taken


@pytest.mark.parametrize("tokens,rows", [(127, 512), (128, 512), (640, 1664), (641, 1664), (896, 2048)])
def test_routed_experts_lay_out_the_planned_rows(device, monkeypatch, tokens, rows):
    """The padded layout of the native call has the rows of the general one, also where its bound is a whole number of 512."""
    torch.manual_seed(tokens)
    moe = _block("experts", device)
    x, dy = (torch.randn(1, tokens, 256, device=device, dtype=torch.bfloat16) for _ in range(2))

    def run():
        sizes = []
        pack = lambda t: sizes.append(torch.tensor(t.shape)) or t
        out = _step(moe, list(moe.parameters()), x, dy, hooks=lambda: torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t))
        return [*out, torch.tensor(sorted(int(n) for s in sizes for n in s))]
    native, general, taken = _both(monkeypatch, run)
    _same(native, general)
    assert "routed_forward" in taken and rows in native[-1].tolist() and rows == ops.plan_length(2 * tokens, 8, 32, 128)


def _block(kind, device):
    if kind == "linear":
        return _holder(Linear.Config().build(in_features=256, out_features=384), device)
    if kind == "feed forward":
        return _holder(FeedForward.Config(hidden_dim=384).build(dim=256), device)
    moe = MoE(MoE.Config(num_experts=8, num_shared_experts=0, hidden_dim=256, top_k=2, score_func="softmax"),
              dim=256).to(device).to(torch.bfloat16)
    moe.init_weights(init_std=0.02, buffer_device=device)
    holder = nn.Module()
    holder.moe = moe
    _convert(holder, ["experts"])
    return moe


@pytest.mark.parametrize("kind", ["linear", "feed forward", "experts"])
def test_saved_tensors_that_hooks_return_as_others(device, monkeypatch, kind):
    """Hooks may give a backward its saved tensors with other strides; on another device, or with less in them, is an
    error on either path."""
    torch.manual_seed(1)
    block = _block(kind, device)
    x, dy = (torch.randn(1, 200, n, device=device, dtype=torch.bfloat16) for n in (256, 384 if kind == "linear" else 256))
    pack = lambda t: t
    strided = lambda t: torch.stack((t, t), -1)[..., 0]
    moved = lambda t: t.cpu()
    short = lambda t: t.view(-1)[:t.numel() // 2].clone() if t.dtype == torch.uint8 and t.dim() == 1 else t
    step = lambda unpack: _step(block, list(block.parameters()), x, dy,
                                hooks=lambda: torch.autograd.graph.saved_tensors_hooks(pack, unpack))
    want = step(lambda t: t)
    native, general, taken = _both(monkeypatch, lambda: step(strided))
    assert any(name.endswith("_forward") for name in taken) and not any(name.endswith("_backward") for name in taken)
    _same(native, want)
    _same(general, want)
    with pytest.raises((RuntimeError, TypeError)):
        step(moved)
    if kind != "experts":  # (whose codes and scales are tensors with shapes of their own)
        with pytest.raises(RuntimeError, match="saved MXFP8 operand"):
            step(short)


def test_capture(device):
    """A captured step of native calls replays on new inputs."""
    lin = _holder(Linear.Config().build(in_features=256, out_features=384), device)
    x = torch.randn(200, 256, device=device, dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn(200, 384, device=device, dtype=torch.bfloat16)
    step = lambda: torch.autograd.grad(lin(x), [x, lin.weight], dy)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for seed in range(3):
        torch.manual_seed(seed)
        with torch.no_grad():
            x.copy_(torch.randn(200, 256, device=device))
        graph.replay()
        torch.cuda.synchronize()
        _same(out, step())


def test_other_threads_run_during_native_calls(device, monkeypatch):
    """The library is called with the interpreter lock released: every entry point is replaced by a function that says
    whether its caller holds it (1: an error status), and launches nothing."""
    import ctypes

    blocks = [_block(kind, device) for kind in ("linear", "feed forward", "experts")]
    counted, called = _Counted(_lib.blocks()), []

    def held(status, name):
        called.append(name)
        raise AssertionError(f"{name} was called with the interpreter lock held")

    address = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    _lib.blocks().bind({name: address for name in _lib.SIGNATURES}, held)
    try:
        with monkeypatch.context() as m:
            m.setattr(_lib, "blocks", lambda: counted)
            for block, outer in zip(blocks, (384, 256, 256)):
                x, dy = (torch.zeros(1, 200, n, device=device, dtype=torch.bfloat16) for n in (256, outer))
                _step(block, list(block.parameters()), x, dy)
            with torch.no_grad():
                for tokens in (16, 200):
                    blocks[0](torch.zeros(tokens, 256, device=device, dtype=torch.bfloat16))
    finally:
        _lib._blocks = None
        _lib.blocks()  # bound to the library again
    assert not called
    assert {"linear_forward", "linear_backward", "linear_apply", "ffn_forward", "ffn_backward", "routed_forward",
            "routed_backward"} <= set(counted.taken)


def test_threads_on_streams_of_their_own(device):
    """Two threads take the same linears over the same activation, which changes from pass to pass: each orders its
    stream behind what wrote the activation and no more, so a cast taken over from the other's stream, or memory that it
    gave back, would show.  Every pass of every thread is compared."""
    import threading

    a = _holder(Linear.Config().build(in_features=256, out_features=384), device)
    b = _holder(Linear.Config().build(in_features=256, out_features=160), device)
    passes, shape = 12, (1000, 256)
    xs = [torch.randn(shape, device=device, dtype=torch.bfloat16) for _ in range(passes)]

    def step(x):
        x = x.detach().requires_grad_(True)
        ya, yb = a(x), b(x)
        return [ya.detach(), yb.detach(), *torch.autograd.grad((ya, yb), [x, a.weight, b.weight], (ya.detach(), yb.detach()))]

    def forward(x):
        with torch.no_grad():  # (nothing drops the remembered cast between the threads)
            return [a(x), b(x)]

    want = [[*step(x), *forward(x)] for x in xs]
    x, got, failed = torch.empty(shape, device=device, dtype=torch.bfloat16), {}, []
    written, barrier = torch.cuda.Event(), threading.Barrier(3, timeout=60)

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for n in range(passes):
                    barrier.wait()  # x of this pass is on its way
                    stream.wait_event(written)
                    got[n, i] = [*step(x), *forward(x)]
                    stream.synchronize()
                    barrier.wait()
        except Exception as ex:
            failed.append(ex)
            barrier.abort()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    try:
        for n in range(passes):
            x.copy_(xs[n])
            written.record()
            barrier.wait()
            barrier.wait()
    except threading.BrokenBarrierError:
        pass
    for t in threads:
        t.join()
    assert not failed, failed
    for n in range(passes):
        for i in range(2):
            _same(got[n, i], want[n])


def test_remembered_cast_serves_its_own_stream(device):
    """A linear on another stream than the one that cast its activation casts again; what was cast there is there."""
    lin = _holder(Linear.Config().build(in_features=256, out_features=384), device)
    x, side = torch.randn(200, 256, device=device, dtype=torch.bfloat16), torch.cuda.Stream()
    key = ("rceil", ops.CODE_PITCH_PAD)
    with torch.no_grad():
        mx_tensor.clear_cast_cache()
        want = lin(x)
        assert mx_tensor._cast_cache.get(x, key) is not None
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            assert mx_tensor._cast_cache.get(x, key) is None
            got = lin(x)
            assert mx_tensor._cast_cache.get(x, key) is not None
        assert mx_tensor._cast_cache.get(x, key) is None
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want)


def test_cached_weight_cast_on_another_stream(device):
    """A cached weight cast that is still queued when another stream asks for it: that stream waits for it."""
    plain = _holder(Linear.Config().build(in_features=2176, out_features=288), device)
    lin = _holder(Linear.Config().build(in_features=2176, out_features=288), device, cache=True)
    x, side = torch.randn(300, 2176, device=device, dtype=torch.bfloat16), torch.cuda.Stream()
    with torch.no_grad():
        for p, q in zip(lin.parameters(), plain.parameters()):
            p.copy_(q)
        want = plain(x)
        torch.cuda.synchronize()
        torch.cuda._sleep(100_000_000)  # some 50 ms in front of the cast
        first = lin(x)
        with torch.cuda.stream(side):
            got = lin(x)
            side.synchronize()
        for p in lin.parameters():
            p.mul_(1)  # (a new version: the entry is replaced)
        again = lin(x)
    torch.cuda.synchronize()
    for y in (first, got, again):
        assert torch.equal(y, want)


def test_errors_keep_their_types(device, monkeypatch):
    """Memory that runs out is torch's error on either path; a status of the library is the package's."""
    lin = _holder(Linear.Config().build(in_features=4096, out_features=4096), device)
    x = torch.randn(8192, 4096, device=device, dtype=torch.bfloat16, requires_grad=True)
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(device) + (1 << 20)) / total, device)
    held = []  # what earlier tests left in the allocator's cache would serve the linear
    for size in (1 << 30, 1 << 28, 1 << 26, 1 << 24, 1 << 22, 1 << 20):
        try:
            while len(held) < 10000:
                held.append(torch.empty(size, dtype=torch.uint8, device=device))
        except torch.OutOfMemoryError:
            pass
    try:
        for native in (True, False):
            with monkeypatch.context() as m:
                if not native:
                    m.setattr(ops, "native_block_ok", lambda *a: False)
                with pytest.raises(torch.OutOfMemoryError):
                    lin(x)
    finally:
        held.clear()
        torch.cuda.set_per_process_memory_fraction(1.0, device)
    blocks, w = _lib.blocks(), lin.weight.detach().as_subclass(torch.Tensor)
    with pytest.raises(_lib.MXLibraryError, match="mx_cast_pad_many"):
        blocks.linear_forward(x.detach(), w, 7, 128)  # no such scale mode
    assert torch.isfinite(lin(x)).all()


@pytest.mark.parametrize("form", ["plain", "rows of a wider matrix", "rows that are not aligned", "columns first"])
def test_single_launches(device, monkeypatch, form):
    """The gate, the routing, the log-probabilities and the hand-over's lists through the native module and step by step:
    the same outputs for operands that it takes and for those that it hands back."""
    torch.manual_seed(3)
    T, D, E, k, V = 33, 256, 16, 4, 1003
    bf, f32 = torch.bfloat16, torch.float32
    x, w, base = (_form(form, device, bf, rows, D) for rows in (T, E, T))
    dlogits, logits = _form(form, device, f32, T, E), _form(form, device, f32, T, E)
    bias, dtop = torch.randn(E, device=device), _form(form, device, f32, T, k)
    vocab, grad = _form(form, device, bf, T, V), torch.randn(2 * T, device=device)[::2]
    target = torch.randint(0, V, (T,), device=device)
    listed = [_form(form, device, t, 7, 96) for t in (bf, f32)] + [torch.randn(2, 5, 64, device=device)]

    def run():
        out = [ops.gate_logits(x, w), ops.gate_dx(dlogits, w), ops.gate_dx(dlogits, w, base), ops.gate_dw(dlogits, x)]
        for softmax in (True, False):
            top, selected, counts, blocks = ops.route_topk(logits, bias if softmax else None, k, softmax, True, 2.5)
            out += [top, selected, counts, blocks, ops.route_topk_bwd(logits, selected, dtop, softmax, True, 2.5)]
        lp, lse = ops.token_logprob_fwd(vocab, target)
        out += [lp, lse, ops.token_logprob_bwd(vocab, target, lse, grad), ops.token_logprob_bwd(vocab, target, lse, lp)]
        sent = ops.to_mx_rows_many(listed, "rceil")
        return out + [t for q in sent for t in (q.codes, q.scales)] + ops.mx_dequant_many(sent)

    counted = _Counted(_lib.blocks())
    with monkeypatch.context() as m:
        m.setattr(_lib, "blocks", lambda: counted)
        native = run()
    with monkeypatch.context() as m:
        m.setattr(ops, "_single", lambda x: False)
        general = run()
    _same(native, general)
    if form == "plain":
        assert {"gate_logits", "gate_dx", "gate_dw", "route_topk", "route_topk_bwd", "token_logprob_fwd", "token_logprob_bwd",
                "rows_many", "dequant_many"} <= set(counted.taken)
