"""The smaller tiles of the persistent GEMM (192 and 128 rows or columns), their splits along K and their float32
results: at the edges of tiles, 128-row scale groups and 128-deep blocks, against the products of the same codes in
float64 and against 256 x 256 tiles, whose sums every unsplit tile forms in the same order."""
import numpy as np
import pytest
import torch

from tests.helpers import bf16_from_bits, randn_bits
from torchtitan_amd import _lib, ops

pytestmark = pytest.mark.gpu

TILES = [(4, 4), (3, 4), (4, 3), (2, 4), (4, 2)]


@pytest.fixture
def hooks():
    lib = _lib.load()
    yield lib
    lib.mx_debug_set_tile(0, 0, 0)
    lib.mx_debug_set_grid(0)
    lib.mx_debug_force_kernel(0)


def _operand(device, rng, rows, K, std=1.0):
    """(pitched operand, what its codes and scales stand for, in float64)"""
    x = bf16_from_bits(randn_bits(rng, (rows, K), std=std, outliers=1e-3), device)
    q = ops.to_operands(x, "rceil", cols=False, pitch_pad=128)[0]
    scales = torch.exp2(ops.scale_unlayout(q.scales.contiguous(), rows, q.k // 32).double() - 127)
    return q, (q.codes.view(torch.float8_e4m3fn).double().view(rows, -1, 32) * scales[..., None]).view(rows, q.k)


def _float32(a, b, ld, ws=None):
    """The product's float32 form, rows `ld` apart."""
    M, N = a.rows, b.rows
    out = torch.full((M, ld), 7.0, dtype=torch.float32, device=a.buf.device)
    ops._call("mx_gemm_nt_f32_ld", "gemm_nt", out.device, a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr,
              out.data_ptr(), M, N, a.k, a.ld, ld, None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(),
              ops._stream(out))
    assert bool((out[:, N:] == 7.0).all())
    return out[:, :N]


def _check(got, want):
    """`got` is no further from `want` (float64) than its rounding to bf16 by more than 1 %: float32 sums of up to
    a few thousand terms are off by less than 2^-18 of the terms' norm, a hundredth of the rounding's 2^-9 / sqrt(3) and
    less, and errors of that size add in squares."""
    err = lambda t: float((t.double() - want).norm() / want.norm())
    assert err(got) <= 1.01 * err(want.bfloat16())


@pytest.mark.parametrize("M,N,K", [(65, 136, 128),      # less than any tile, one block
                                   (128, 384, 256), (129, 392, 384),
                                   (192, 192, 384), (193, 200, 512), (191, 576, 128),
                                   (385, 1160, 640), (577, 776, 896)])
def test_every_tile_forms_the_same_sums(device, hooks, M, N, K):
    rng = np.random.default_rng(M + N + K)
    (a, ha), (a2, ha2) = _operand(device, rng, M, K), _operand(device, rng, M, K, 0.3)
    (b, hb), (b2, hb2) = _operand(device, rng, N, K, 0.02), _operand(device, rng, N, K, 0.05)
    runs = {}
    for grid in (0, 8):  # 8 workgroups: several tiles each, the ring runs on from one into the next
        for tile in TILES:
            hooks.mx_debug_set_grid(grid)
            hooks.mx_debug_set_tile(*tile, 0)
            out = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device=device)
            ops._gemm_operands(a, b, out[:, :N])
            assert bool((out[:, N:] == 7.0).all())
            got = [out[:, :N].contiguous()]
            assert torch.equal(_float32(a, b, N + 24), got[0].float())
            if M > 128:
                got += [ops.mx_gemm_nt_shared_a(a, b, b2), ops.mx_gemm_nt_shared_b(a, a2, b), ops.mx_gemm_nt_pair(a, b, a2, b2)]
            runs[grid, tile] = got
    want = runs[0, (4, 4)]
    _check(want[0], ha @ hb.T)
    if M > 128:
        _check(want[1][1], ha @ hb2.T)
        _check(want[2][1], ha2 @ hb.T)
        _check(want[3], ha @ hb.T + ha2 @ hb2.T)
    for key, got in runs.items():
        for i, (g, w) in enumerate(zip(got, want, strict=True)):
            assert torch.equal(g, w), (key, i)


@pytest.mark.parametrize("slices", [2, 3, 6])
@pytest.mark.parametrize("tile", [(4, 4), (2, 4), (4, 2)])
@pytest.mark.parametrize("M,N,K", [(65, 136, 4096), (200, 392, 4224), (513, 264, 4352)])
def test_splits_along_k(device, hooks, M, N, K, tile, slices):
    rng = np.random.default_rng(M + slices)
    (a, ha), (b, hb) = _operand(device, rng, M, K), _operand(device, rng, N, K, 0.02)
    hooks.mx_debug_set_tile(*tile, slices)
    need = int(hooks.mx_gemm_nt_workspace_bytes(M, N, K))
    assert need == slices * M * N * 4
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=device)  # (NaN)
    out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=device)
    for grid in (0, 8):
        hooks.mx_debug_set_grid(grid)
        ops._call("mx_gemm_nt_ld", "gemm_nt_splitk", device, a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr,
                  out.data_ptr(), M, N, a.k, a.ld, N, ws.data_ptr(), need, ops._stream(out))
        _check(out, ha @ hb.T)
        assert torch.equal(_float32(a, b, N, ws), out.float())


@pytest.mark.parametrize("slices", [2, 6])
@pytest.mark.parametrize("tile", [(4, 4), (2, 4), (4, 2)])
@pytest.mark.parametrize("M,N,K", [(129, 136, 2176), (200, 392, 4224), (513, 264, 1664)])
def test_splits_of_a_sum_of_two_products(device, hooks, M, N, K, tile, slices):
    rng = np.random.default_rng(M + slices)
    (a, ha), (a2, ha2) = _operand(device, rng, M, K), _operand(device, rng, M, K, 0.3)
    (b, hb), (b2, hb2) = _operand(device, rng, N, K, 0.02), _operand(device, rng, N, K, 0.05)
    hooks.mx_debug_set_tile(*tile, slices)
    need = int(hooks.mx_gemm_nt_pair_workspace_bytes(M, N, K))
    assert need == slices * M * N * 4
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=device)  # (NaN)

    def run(lent):
        out = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device=device)
        ops._call("mx_gemm_nt_pair_ws", "gemm_nt_pair", device, a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr,
                  a2.codes_ptr, a2.scales_ptr, b2.codes_ptr, b2.scales_ptr, out.data_ptr(), M, N, K, a.ld, N + 24,
                  ws.data_ptr(), lent, ops._stream(out))
        assert bool((out[:, N:] == 7.0).all())
        return out[:, :N]

    for grid in (0, 8):
        hooks.mx_debug_set_grid(grid)
        _check(run(need), ha @ hb.T + ha2 @ hb2.T)
    hooks.mx_debug_set_tile(0, 0, 0)
    hooks.mx_debug_set_grid(0)
    ws.fill_(0xFF)
    _check(run(0), ha @ hb.T + ha2 @ hb2.T)  # too little memory lent: one chain, nothing written there
    assert bool((ws == 0xFF).all())


@pytest.mark.parametrize("M,N,K", [(65, 136, 128), (256, 1024, 256), (300, 264, 1024)])
def test_float32_results_of_short_contractions(device, M, N, K):
    """(these run on the kernel of one 128 x 128 tile per workgroup)"""
    rng = np.random.default_rng(M)
    a, b = _operand(device, rng, M, K)[0], _operand(device, rng, N, K, 0.02)[0]
    want = ops.mx_gemm_nt(a, b)
    assert torch.equal(_float32(a, b, N + 8), want.float())
    got = ops.mx_gemm_nt_as(a, b, torch.float32)
    assert got.dtype == torch.float32 and torch.equal(got, want.float())
    few = a.first_rows(64)  # no float32 form: the bf16 result, converted
    assert torch.equal(ops.mx_gemm_nt_as(few, b, torch.float32), ops.mx_gemm_nt(few, b).float())


def test_shapes_that_are_split(device, hooks):
    """Which way a shape runs: few rows on their own kernel as long as that is ahead, slices where tiles are few
    and the contraction is long, and never more partial sums than one 256 x 256 tile per CU but for shapes of
    more tiles than half of the CUs."""
    need = lambda M, N, K: int(hooks.mx_gemm_nt_workspace_bytes(M, N, K))
    with torch.cuda.device(device):
        assert need(16, 4096, 8192) == 0 and need(64, 4096, 4096) == 0 and need(64, 4096, 8192) > 0
        assert need(256, 4096, 8192) > 0 and need(2048, 2048, 2048) == 0 and need(4096, 4096, 4096) == 0
        for M in (65, 200, 1000, 2048):
            for N in (1024, 4096, 6144):
                for K in (1024, 4096, 16384, 147456):
                    assert need(M, N, K) <= 64 << 20 or -(-M // 256) * -(-N // 256) > 128
        pair = lambda M, N, K: int(hooks.mx_gemm_nt_pair_workspace_bytes(M, N, K))
        assert pair(256, 4096, 14336) == 8 * 256 * 4096 * 4 and pair(128, 4096, 14336) == pair(300, 1000, 14300) == 0
        assert pair(256, 4096, 2048) == pair(4096, 2048, 6144) == pair(16384, 4096, 14336) == 0
        for M in (129, 200, 1000, 2048, 5003):
            for N in (1024, 4096, 6144):
                for K in (2176, 6144, 14336, 147456):
                    assert pair(M, N, K) <= 64 << 20 and pair(M, N, K) % (2 * M * N * 4) == 0


def test_one_product_prepares_all_others_for_capture(device, hooks):
    """The first dense product on tiles raises the LDS limits of every tile and form, so that a graph may capture others
    than the one that the program warmed up on: nothing is left to raise, and captured products replay as eager ones."""
    rng = np.random.default_rng(5)
    M, N, K = 200, 264, 4352
    (a, a2), (b, b2) = [[_operand(device, rng, rows, K, std)[0] for _ in range(2)] for rows, std in ((M, 1.0), (N, 0.02))]
    ops.mx_gemm_nt(a, b)
    raised = hooks.mx_debug_lds_limits_raised()
    assert raised >= 3 * len(TILES) + 3 + 3  # plain, float32 and sum of two; slices of K; one tile a workgroup

    def products():
        out = []
        for tile in TILES:
            for slices in (0, 2) if tile[0] * tile[1] != 12 else (0,):
                hooks.mx_debug_set_tile(*tile, slices)
                ops._gemm_workspace.clear()
                out += [ops.mx_gemm_nt(a, b), ops.mx_gemm_nt_as(a, b, torch.float32), ops.mx_gemm_nt_pair(a, b, a2, b2),
                        ops.mx_gemm_nt_shared_a(a, b, b2), ops.mx_gemm_nt_shared_b(a, a2, b)]
        hooks.mx_debug_set_tile(0, 0, 0)
        ops._gemm_workspace.clear()
        return out
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = products()
    assert hooks.mx_debug_lds_limits_raised() == raised
    for std in (1.0, 3.0):
        a.buf.copy_(_operand(device, rng, M, K, std)[0].buf)
        graph.replay()
        torch.cuda.synchronize()
        for i, (x, y) in enumerate(zip(got, products(), strict=True)):
            assert torch.equal(x, y), i


@pytest.mark.parametrize("kernel", [1, 2, 3])
def test_float32_results_on_a_forced_kernel(device, hooks, kernel):
    """A forced kernel is not split, whatever is lent, and gives the bf16 product's values on that kernel."""
    rng = np.random.default_rng(kernel)
    M, N, K = 200, 392, 8192
    (a, _), (b, _) = _operand(device, rng, M, K), _operand(device, rng, N, K, 0.02)
    need = int(hooks.mx_gemm_nt_workspace_bytes(M, N, K))
    assert need > 0
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=device)
    hooks.mx_debug_force_kernel(kernel)
    assert torch.equal(_float32(a, b, N, ws), ops.mx_gemm_nt(a, b).float())
    assert bool((ws == 0xFF).all())


@pytest.mark.parametrize("slices", [2, 6])
@pytest.mark.parametrize("tile", [(4, 4), (2, 4), (4, 2)])
@pytest.mark.parametrize("M,N,K", [(1, 136, 16896), (16, 264, 16896), (33, 392, 5760), (64, 136, 4352)])
def test_splits_of_few_rows(device, hooks, M, N, K, tile, slices):
    """Up to 64 rows, of contractions behind the line up to which their own kernel runs."""
    rng = np.random.default_rng(M + slices)
    (a, ha), (b, hb) = _operand(device, rng, M, K), _operand(device, rng, N, K, 0.02)
    hooks.mx_debug_set_tile(*tile, slices)
    need = int(hooks.mx_gemm_nt_workspace_bytes(M, N, K))
    assert need == slices * M * N * 4
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=device)  # (NaN)
    out = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device=device)
    for grid in (0, 8):
        hooks.mx_debug_set_grid(grid)
        ops._call("mx_gemm_nt_ld", "gemm_nt_splitk", device, a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr,
                  out.data_ptr(), M, N, a.k, a.ld, N + 24, ws.data_ptr(), need, ops._stream(out))
        _check(out[:, :N], ha @ hb.T)
        assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(64, 4096, 8192), (33, 1024, 14336), (16, 4096, 17408)])
def test_few_rows_that_are_split_by_shape(device, M, N, K):
    rng = np.random.default_rng(M)
    (a, ha), (b, hb) = _operand(device, rng, M, K), _operand(device, rng, N, K, 0.02)
    with torch.cuda.device(device):
        assert int(_lib.load().mx_gemm_nt_workspace_bytes(M, N, K)) > 0
    _check(ops.mx_gemm_nt(a, b), ha @ hb.T)


@pytest.mark.parametrize("N,K", [(1024, 2048), (4096, 4096), (392, 384)])
def test_rows_do_not_depend_on_how_many_there_are(device, N, K):
    """More than 64 rows of a contraction of up to 4096: one chain of sums in one order on every kernel and tile."""
    rng = np.random.default_rng(N)
    a, b = _operand(device, rng, 3001, K)[0], _operand(device, rng, N, K, 0.02)[0]
    want = ops.mx_gemm_nt(a, b)
    for M in (65, 128, 129, 200, 1000, 2048):
        assert torch.equal(ops.mx_gemm_nt(a.first_rows(M), b), want[:M]), M


@pytest.mark.parametrize("M,N,K", [(65, 136, 128), (64, 200, 640), (128, 384, 256), (129, 392, 768), (192, 136, 896),
                                   (321, 200, 1024), (200, 328, 2176), (577, 776, 1152)])
@pytest.mark.parametrize("pad", [0, 128])
def test_tiles_of_the_few_tiles_kernel_form_the_same_sums(device, hooks, M, N, K, pad):
    """64 x 64 and 128 x 64 tiles against 256 x 256 ones: rows and columns that end inside a tile or a half of a scale
    group, contractions shorter, as long and longer than the ring, and the sum of two whose second one begins inside it."""
    rng = np.random.default_rng(M + N + K)
    (a, ha), (a2, _) = _operand(device, rng, M, K), _operand(device, rng, M, K, 0.3)
    (b, hb), (b2, _) = _operand(device, rng, N, K, 0.02), _operand(device, rng, N, K, 0.05)
    if pad == 0:
        a, a2, b, b2 = (ops.Operand.of(q.data()._replace(codes=q.codes.contiguous())) for q in (a, a2, b, b2))

    def run(tile):
        hooks.mx_debug_set_tile(*tile, 0)
        out = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device=device)
        ops._call("mx_gemm_nt_ld", "gemm_nt", device, a.codes_ptr, a.scales_ptr, b.codes_ptr, b.scales_ptr, out.data_ptr(), M, N,
                  a.k, a.ld, N + 24, None, 0, ops._stream(out))
        assert bool((out[:, N:] == 7.0).all())
        got = [out[:, :N].contiguous()]
        if M > 64:
            got.append(_float32(a, b, N + 24))
        if M > 128:
            got += [ops.mx_gemm_nt_shared_a(a, b, b2), ops.mx_gemm_nt_shared_b(a, a2, b), ops.mx_gemm_nt_pair(a, b, a2, b2)]
        return got

    hooks.mx_debug_force_kernel(3)
    want = run((4, 4))
    hooks.mx_debug_force_kernel(0)
    _check(want[0], ha @ hb.T)
    for tile in ((1, 1), (2, 1)):
        for i, (g, w) in enumerate(zip(run(tile), want, strict=True)):
            if M > 64 or i:  # (up to 64 rows have a kernel of their own, with sums in another order)
                assert torch.equal(g, w), (tile, i)


@pytest.mark.parametrize("M,N,K", [(129, 136, 128), (256, 256, 384), (300, 392, 640), (385, 200, 2016), (512, 1000, 4096)])
@pytest.mark.parametrize("mode", ["floor", "rceil"])
@pytest.mark.parametrize("pad", [0, 128])
def test_gate_in_the_product_gives_the_bits_of_the_gate_behind_it(device, M, N, K, mode, pad):
    """Rows and columns that end inside a tile, a scale group and a 32-column block; sizes of the factors from where
    the gate is linear to where it overflows, blocks of zeros, infinities and NaN."""
    rng = np.random.default_rng(M + N + K)
    x = bf16_from_bits(randn_bits(rng, (M, K), std=1.0, outliers=1e-3), device)
    x[1:60:7] = 0
    x[2], x[67], x[3, 5], x[70, 9] = 1e30, -1e30, float("nan"), float("inf")
    w, w2 = (bf16_from_bits(randn_bits(rng, (N, K), std=s, outliers=1e-3), device) for s in (0.05, 2.0))
    w[:64], w2[64:96] = w[:64] * 1e-12, 0
    a, b, b2 = (ops.to_operands(t, mode, cols=False, pitch_pad=pad)[0] for t in (x, w, w2))
    h = ops.mx_gemm_nt_shared_a(a, b, b2)
    want = ops.swiglu_to_operands(h[0], h[1], mode, False, pad)[0]
    got = ops.mx_gemm_nt_swiglu(a, b, b2, mode, planned=True)
    assert (got.k, got.ld, got.depth) == (want.k, want.ld, want.depth)
    wrong = (got.codes != want.codes).nonzero().tolist()
    assert not wrong, (len(wrong), wrong[:8])
    assert torch.equal(*(ops.scale_unlayout(q.scales.contiguous(), M, q.k // 32) for q in (got, want)))


@pytest.mark.parametrize("M,N,K", [(700, 1000, 128), (1025, 520, 256), (700, 1000, 640), (2048, 776, 384), (520, 2056, 2016)])
@pytest.mark.parametrize("mode", ["floor", "rceil"])
def test_gate_in_the_product_over_several_tiles_a_workgroup(device, hooks, M, N, K, mode):
    """Eight workgroups take three tiles and more each, the last rows and columns ragged, over one, two and an odd number of
    blocks: the next tile's copies are in flight while a tile is gated, and the waves change between both weights."""
    rng = np.random.default_rng(M + N + K)
    x, w, w2 = (bf16_from_bits(randn_bits(rng, (rows, K), std=s, outliers=1e-3), device)
                for rows, s in ((M, 1.0), (N, 0.05), (N, 0.5)))
    a, b, b2 = (ops.to_operands(t, mode, cols=False, pitch_pad=128)[0] for t in (x, w, w2))
    h = ops.mx_gemm_nt_shared_a(a, b, b2)
    want = ops.swiglu_to_operands(h[0], h[1], mode, False, 128)[0]
    for grid in (8, 16):
        hooks.mx_debug_set_grid(grid)
        assert -(-M // 256) * -(-N // 128) > grid
        got = ops.mx_gemm_nt_swiglu(a, b, b2, mode, planned=True)
        wrong = (got.codes != want.codes).nonzero().tolist()
        assert not wrong, (grid, len(wrong), wrong[:8])
        assert torch.equal(*(ops.scale_unlayout(q.scales.contiguous(), M, q.k // 32) for q in (got, want))), grid


@pytest.mark.parametrize("M,N,K,gated", [(4096, 6144, 2048, 1), (3001, 8192, 1024, 1), (512, 14336, 4096, 1), (1500, 4992, 2048, 1),
                                         (2270, 4096, 1536, 0), (1409, 6080, 768, 0), (3533, 4736, 1920, 0),
                                         (2048, 5632, 2048, 0), (512, 8192, 3072, 0)])
def test_gate_in_the_product_is_chosen_where_it_is_ahead(device, M, N, K, gated):
    """Full rounds of tiles, not a last round of few (measured: 7 to 15 % behind the two launches) nor half of the CUs."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the line is for 256 CUs")
    assert _lib.load().mx_gemm_nt_swiglu_planned(M, N, K) == gated


@pytest.mark.parametrize("norm", [False, True])
def test_feed_forward_without_gradients_gates_in_the_product(device, monkeypatch, norm):
    """A block of two rounds of tiles takes the gated launch by itself, behind a norm or not, and gives the bits of the
    two launches."""
    from torchtitan_amd import mx_blocks
    from torchtitan_amd.mx_tensor import MXFP8Config, MXFP8TrainingWeight

    M, D, H = 4096, 2048, 6144
    g = torch.Generator(device=device).manual_seed(3)
    rn = lambda *shape, std=1.0: (torch.randn(shape, generator=g, device=device) * std).to(torch.bfloat16)
    cfg = MXFP8Config(fuse_rmsnorm_cast=norm)
    x, n = rn(M, D), (rn(D) * 0.1 + 1).to(torch.bfloat16)
    w1, w2, w3 = (MXFP8TrainingWeight(rn(*shape, std=0.02), cfg) for shape in ((H, D), (D, H), (H, D)))
    run = (lambda: mx_blocks.mx_norm_feed_forward(x, n, 1e-5, w1, w2, w3)) if norm else (
        lambda: mx_blocks.mx_feed_forward(x, w1, w2, w3))
    calls, call = [], ops._call
    assert _lib.load().mx_gemm_nt_swiglu_planned(M, H, D)
    with torch.no_grad():
        with monkeypatch.context() as m:
            m.setattr(ops, "_call", lambda name, *args: calls.append(name) or call(name, *args))
            got = run()
        assert calls.count("mx_gemm_nt_swiglu_ld") == 1 and "mx_gemm_nt_shared_a_ld" not in calls
        with monkeypatch.context() as m:
            m.setattr(ops, "mx_gemm_nt_swiglu", lambda *args: None)
            want = run()
    assert torch.equal(got, want) and bool(torch.isfinite(got).all())
