"""Products of a few tokens that finish the residual stream and leave its norm's root to the reader.

``ops.gemm(..., next_norm=...)`` against float64: the stream, what is left of the norm, and the products that take it,
at the edges of the kernel's sizes: one token to sixteen (one matrix instruction to 8, two beyond), blocks of 8 and of 16
weight rows, k shares that are empty, partial and of more steps than are in flight, bfloat16 and float32 norm weights.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F32, BF16 = "cuda", torch.float32, torch.bfloat16
# bfloat16 has 8 significant bits: one rounding to it is off by 2^-8 of the value at most (half of the last place of a value
# just above a power of two); float32 sums of some thousand terms add some 1e-6 of the terms' sum, which is left out
ROUND = 2.0 ** -8


def gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


@pytest.fixture(scope="module")
def ops():
    from photon_infer_amd import ops as o
    o.ensure_loaded(BF16)
    return o


def made(ops, M, N, K, w_dtype=BF16, eps=1e-5, pad=0):
    g = gen(M * 7 + N + K)
    a = (torch.randn(M, K + pad, generator=g, device=DEV)).to(BF16)[:, :K]
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF16)
    x0 = torch.randn(M, N, generator=g, device=DEV)
    weight = (torch.rand(N, generator=g, device=DEV) + 0.5).to(w_dtype)
    ws = ops.KernelWorkspace(DEV)
    assert ws.add_stream_copy(w)
    x = x0.clone()
    ops.gemm(x, a, w, accumulate=True, may_defer=True, ws=ws, next_norm=(weight, eps))
    return ws, x, x0.double() + a.double() @ w.double().t(), weight


@pytest.mark.parametrize("M", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("N,K,w_dtype", [(64, 512, BF16), (64, 1088, F32), (192, 3136, BF16), (2048, 2048, BF16), (2048, 4160, F32),
                                         (3072, 576, BF16), (3136, 4544, F32), (4096, 2112, BF16)])
def test_finished_stream_and_left_norm_against_float64(ops, M, N, K, w_dtype):
    from photon_infer_amd.ops import fast
    if not fast._finish_blocks(M, N, K) or fast._skinny_splits(M, N, K) < 2:
        pytest.skip("a size that the pieces keep")
    ws, x, want, weight = made(ops, M, N, K, w_dtype, pad=8)
    assert ws.counts["norms_left"] == 1 and ws.pending is None
    left = ws.take_left_norm(x, weight, 1e-5)
    assert isinstance(left, ops.LeftNorm) and ws.left_norm is None
    assert ((x.double() - want).abs() <= 2e-6 * (want.abs() + 1.0) * max(1.0, (K / 64) ** 0.5)).all()
    assert torch.equal(left.h, (x * weight.float()).to(BF16))
    sums = (x.double() ** 2).sum(1)
    assert (left.sums.double().sum(1) - sums).abs().max() <= 1e-5 * sums.max()
    # its readers: a product in pieces of k and whole, float32 and bfloat16, and the gated unit
    norm = (x.double() / torch.sqrt(sums[:, None] / N + 1e-5)) * weight.double()
    g = gen(5)
    for rows in (96, 8224):              # 16 rows to a block, and 32
        w2 = (torch.randn(rows, N, generator=g, device=DEV) * N ** -0.5).to(BF16)
        assert ws.add_stream_copy(w2)
        ws.counts["left_norms_read"] = 0
        want2 = norm @ w2.double().t()
        size = (norm.abs() @ w2.double().abs().t())               # what the rounding of the activations may sum up to
        got = ops.qkv_projection(left, w2, F32, ws)
        if isinstance(got, ops.Partials):
            got = got.part.view(-1)[:got.splits * M * rows].view(got.splits, M, rows).sum(0)
        assert ((got.double() - want2).abs() <= ROUND * size).all()
        out = torch.empty(M, rows, dtype=BF16, device=DEV)
        ops.gemm(out, left, w2, ws=ws)
        assert ((out.double() - want2).abs() <= ROUND * (size + want2.abs())).all()
        if rows % 32 == 0:
            unit = torch.empty(M, rows // 2, dtype=BF16, device=DEV)
            ops.gemm_swiglu(unit, left, w2, 16, ws=ws)
            z = want2.view(M, rows // 32, 2, 16)
            s = size.view(M, rows // 32, 2, 16)
            wanted = (torch.nn.functional.silu(z[:, :, 0]) * z[:, :, 1]).reshape(M, -1)
            slack = (1.1 * s[:, :, 0] * z[:, :, 1].abs() + s[:, :, 1] * z[:, :, 0].abs()).reshape(M, -1)
            assert ((unit.double() - wanted).abs() <= ROUND * (1.1 * slack + wanted.abs() + 1e-3)).all()
        assert ws.counts["left_norms_read"] == 3, ws.counts


@pytest.mark.parametrize("M", [1, 8, 16])
@pytest.mark.parametrize("N,K,scale,eps", [(256, 512, 1e-3, 1e-5), (2048, 2048, 0.1, 0.5), (192, 1024, 1.0, 0.0)])
def test_readers_apply_the_root_with_its_eps(ops, M, N, K, scale, eps):
    """Streams whose mean square is small beside eps, of its size, and with no eps at all: a root without it, with another
    one or of a mean over the pieces would be far off."""
    g = gen(M + N)
    a = (torch.randn(M, K, generator=g, device=DEV) * scale).to(BF16)
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF16)
    weight, ws = (torch.rand(N, generator=g, device=DEV) + 0.5).to(BF16), ops.KernelWorkspace(DEV)
    w2 = (torch.randn(96, N, generator=g, device=DEV) * N ** -0.5).to(BF16)
    assert ws.add_stream_copy(w) and ws.add_stream_copy(w2)
    x = torch.randn(M, N, generator=g, device=DEV) * scale
    ops.gemm(x, a, w, accumulate=True, may_defer=True, ws=ws, next_norm=(weight, eps))
    left = ws.take_left_norm(x, weight, eps)
    norm = x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + eps) * weight.double()
    out = torch.empty(M, 96, device=DEV)
    ops.gemm(out, left, w2, ws=ws)
    assert ws.counts["left_norms_read"] == 1
    assert ((out.double() - norm @ w2.double().t()).abs() <= ROUND * (norm.abs() @ w2.double().abs().t())).all()


@pytest.mark.parametrize("M", [1, 9, 16])
@pytest.mark.parametrize("N,K", [(16, 512), (64, 4096), (4112, 512), (8224, 576), (1024, 2048)])
def test_all_of_k_in_a_block_where_the_caller_says_so(ops, M, N, K):
    """In the place of pieces: stored in float32 and bfloat16, and added; 16 rows to a block and 32."""
    from photon_infer_amd.ops import fast
    g = gen(M + N + K)
    a, w = torch.randn(M, K + 8, generator=g, device=DEV).to(BF16)[:, :K], (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF16)
    ws = ops.KernelWorkspace(DEV)
    assert ws.add_stream_copy(w) and fast._skinny_splits(M, N, K) > 1
    want, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    slack = 2.0 ** -24 * (K / 64 + 8) * size              # float32 sums: a chain of K / 64 steps a wave at most, the waves' sums
    x0 = torch.randn(M, N, generator=g, device=DEV)
    f32, b16, x = torch.empty(M, N, device=DEV), torch.empty(M, N, dtype=BF16, device=DEV), x0.clone()
    ops.gemm(f32, a, w, ws=ws, whole=True)
    ops.gemm(b16, a, w, ws=ws, whole=True)
    ops.gemm(x, a, w, accumulate=True, ws=ws, whole=True)
    assert ws.counts["split_products"] == 0
    assert ((f32.double() - want).abs() <= slack).all() and torch.equal(b16, f32.to(BF16))
    assert ((x.double() - x0.double() - want).abs() <= slack + 2.0 ** -23 * (x0.double().abs() + want.abs())).all()


@pytest.mark.parametrize("copies", [(True, True), (True, False), (False, True), (False, False)])
def test_mixers_side_by_side_read_one_norm_of_the_stream_before(ops, copies):
    """The second mixer reads its activations when the first has written the stream already: whichever of them can apply the
    root, both see the norm of the stream before."""
    from photon_infer_amd.parts import StepContext
    from photon_infer_amd.parts.base import Mixer
    from photon_infer_amd.parts.block import SideBySide
    M, D, I = 5, 256, 512
    g = gen(4)
    rnd = lambda n, k: (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)

    class Product(Mixer):
        takes_left_norm = True

        def __init__(self):
            self.w_in, self.w_o = rnd(I, D), rnd(D, I) * 8           # a large update

        def streamed_weights(self):
            return [self.w_in, self.w_o]

        def forward(self, h, x, ctx, cache):
            y = torch.empty(M, I, dtype=BF16, device=DEV)
            ops.gemm(y, h, self.w_in, ws=ctx.workspace)
            ops.gemm(x, y, self.w_o, accumulate=True, may_defer=ctx.may_defer, ws=ctx.workspace, next_norm=ctx.next_norm)

    ws, x, _, weight = made(ops, M, D, 512)
    mixers = [Product(), Product()]
    for m, copy in zip(mixers, copies):
        ws.add_stream_copy(m.w_o)
        if copy:
            ws.add_stream_copy(m.w_in)
    x0 = x.double()
    norm = x0 / torch.sqrt((x0 ** 2).mean(1, keepdim=True) + 1e-5) * weight.double()
    left = ws.take_left_norm(x, weight, 1e-5)
    after = torch.ones(D, dtype=BF16, device=DEV)
    i32 = torch.zeros(M, dtype=torch.int32, device=DEV)
    ctx = StepContext(T=M, R=M, dtype=BF16, token_ids=i32, positions=i32, req_of_token=i32, q_start=i32, kv_len=i32, slots=i32, block_tables={}, logit_rows=i32,
                      may_defer=True, next_norm=(after, 1e-5), workspace=ws)
    SideBySide([("a.", mixers[0]), ("b.", mixers[1])]).forward(left, x, ctx, [None, None])
    assert ws.counts["left_norms_read"] == (2 if all(copies) else 0) and ws.pending is None
    ys = [norm @ m.w_in.double().t() for m in mixers]
    want = x0 + sum(y @ m.w_o.double().t() for y, m in zip(ys, mixers))
    # the activations are rounded twice on the way, each by ROUND of the terms that reach the next sum
    sizes = [(norm.abs() @ m.w_in.double().abs().t() + y.abs()) @ m.w_o.double().abs().t() for y, m in zip(ys, mixers)]
    assert ((x.double() - want).abs() <= ROUND * sum(sizes) + 1e-5 * want.abs()).all()
    assert (sum(y @ m.w_o.double().t() for y, m in zip(ys, mixers))).norm() > 4 * x0.norm()
    final = ws.take_left_norm(x, after, 1e-5)
    assert torch.equal(final.h, x.to(BF16))


@pytest.mark.parametrize("M,heads,head_dim,count,inside", [(1, 8, 64, 2, True), (1, 32, 64, 3, True), (1, 32, 64, 8, True), (1, 32, 64, 16, True), (1, 32, 64, 40, False), (1, 8, 80, 9, True),
                                                          (1, 24, 128, 5, True), (1, 5, 128, 13, True), (1, 24, 128, 12, False), (1, 8, 64, 17, False), (3, 5, 128, 13, False), (2, 8, 80, 9, False),
                                                          (2, 8, 64, 2, False), (7, 24, 128, 3, False), (8, 32, 64, 4, False), (9, 32, 64, 3, False), (16, 32, 64, 2, False),
                                                          (16, 24, 128, 2, False), (16, 32, 64, 8, False)])
def test_key_ranges_into_a_finished_stream(ops, M, heads, head_dim, count, inside):
    """Attention's key ranges as activations: merged by the finishing product where they are few, by the merging kernel
    before it elsewhere; empty ranges, ranges of unlike maxima."""
    N, K = 512, heads * head_dim
    g = gen(count + K)
    part = torch.randn(M, heads, count, head_dim + 4, generator=g, device=DEV)
    part[..., head_dim] *= 3
    part[..., head_dim + 1] = part[..., head_dim + 1].abs() + 0.5
    if count > 2:
        part[:, :, 1, head_dim], part[:, :, 1, :head_dim], part[:, :, 1, head_dim + 1] = float("-inf"), 0.0, 0.0
    rows = torch.arange(M, dtype=torch.int32, device=DEV)
    ranges = ops.KeyRanges(part, count, M, heads, head_dim, rows)
    weights = torch.exp2(part[..., head_dim].double() - part[..., head_dim].double().amax(-1, keepdim=True))
    merged = (part[..., :head_dim].double() * weights[..., None]).sum(2) / (part[..., head_dim + 1].double() * weights).sum(2)[..., None]
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF16)
    weight = (torch.rand(N, generator=g, device=DEV) + 0.5).to(BF16)
    ws = ops.KernelWorkspace(DEV)
    ws.add_stream_copy(w)
    x0 = torch.randn(M, N, generator=g, device=DEV)
    x = x0.clone()
    ops.gemm(x, ranges, w, accumulate=True, may_defer=True, ws=ws, next_norm=(weight, 1e-5))
    assert ws.counts["norms_left"] == 1 and ws.counts["ranges_merged_by_product"] == int(inside)
    a = merged.reshape(M, K)
    want = x0.double() + a @ w.double().t()
    assert ((x.double() - want).abs() <= ROUND * (a.abs() @ w.double().abs().t()) + 1e-5).all()
    left = ws.take_left_norm(x, weight, 1e-5)
    assert torch.equal(left.h, (x * weight.float()).to(BF16))
    assert (left.sums.double().sum(1) - (x.double() ** 2).sum(1)).abs().max() <= 1e-5 * (x.double() ** 2).sum(1).max()


def test_rows_that_are_not_finite_stay_by_themselves_and_zero_rows_keep_their_eps(ops):
    M, N, K = 8, 256, 512
    g = gen(3)
    a = torch.randn(M, K, generator=g, device=DEV).to(BF16)
    a[2, 5], a[6, 100] = float("inf"), float("nan")
    a[4] = 0
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).to(BF16)
    weight = torch.ones(N, dtype=BF16, device=DEV)
    ws = ops.KernelWorkspace(DEV)
    ws.add_stream_copy(w)
    x = torch.zeros(M, N, device=DEV)
    ops.gemm(x, a, w, accumulate=True, may_defer=True, ws=ws, next_norm=(weight, 1e-5))
    left = ws.take_left_norm(x, weight, 1e-5)
    out = torch.empty(M, 64, dtype=F32, device=DEV)
    reader = (torch.randn(64, N, generator=g, device=DEV) * 0.05).to(BF16)
    ws.add_stream_copy(reader)
    ops.gemm(out, left, reader, ws=ws)
    assert ws.counts["left_norms_read"] == 1
    good = [0, 1, 3, 4, 5, 7]
    assert torch.isfinite(x[good]).all() and torch.isfinite(out[good]).all() and (out[4] == 0).all()
    assert not torch.isfinite(x[2]).any() and torch.isnan(x[6]).all() and torch.isnan(out[2]).all() and torch.isnan(out[6]).all()


@pytest.mark.parametrize("T,D,table_dtype,w_dtype,h_dtype", [(1, 64, BF16, BF16, BF16), (3, 1000, BF16, F32, BF16), (8, 2048, BF16, BF16, BF16), (5, 8192, F32, F32, F32),
                                                           (300, 2052, F32, BF16, BF16)])
def test_embedding_and_its_norm_in_one_kernel(ops, T, D, table_dtype, w_dtype, h_dtype):
    g = gen(D)
    table = torch.randn(50, D, generator=g, device=DEV).to(table_dtype)
    weight = (torch.rand(D, generator=g, device=DEV) + 0.5).to(w_dtype)
    ids = torch.randint(0, 50, (T,), generator=g, device=DEV).to(torch.int32)
    if T > 2:
        ids[1] = 50                                     # not in the table: a row that is not a number, and no fault
    for scale in (1.0, 3.5):
        x, plain, ws = torch.empty(T, D, device=DEV), torch.empty(T, D, device=DEV), ops.KernelWorkspace(DEV)
        assert ops.embedding_norm(x, table, ids, scale, weight, 1e-5, h_dtype, ws)
        ops.embedding(plain, table, ids, scale)
        assert torch.equal(x.view(torch.int32), plain.view(torch.int32))
        left = ws.take_left_norm(x, weight, 1e-5)
        assert left.count == 0 and left.h.dtype == h_dtype
        good = [t for t in range(T) if ids[t] < 50]
        want = plain[good].double() / torch.sqrt((plain[good].double() ** 2).mean(1, keepdim=True) + 1e-5) * weight.double()
        slack = want.abs() * (ROUND if h_dtype == BF16 else 1e-6)
        assert ((left.h[good].double() - want).abs() <= slack * 1.001).all()
        assert torch.isnan(left.h[[t for t in range(T) if t not in good]].float()).all()
    assert not ops.embedding_norm(torch.empty(1, 30, device=DEV), torch.zeros(4, 30, device=DEV), ids[:1] * 0, 1.0, torch.ones(30, device=DEV), 1e-5, F32, ws)


@pytest.mark.parametrize("T,D,table_dtype,w_dtype,h_dtype", [(1, 64, BF16, BF16, BF16), (3, 1000, BF16, F32, BF16), (5, 1024, F32, F32, F32), (8, 3072, BF16, BF16, BF16),
                                                           (17, 8192, BF16, BF16, BF16), (256, 4096, BF16, BF16, BF16), (257, 4096, F32, F32, F32),
                                                           (257, 2048, BF16, BF16, BF16), (300, 2052, F32, BF16, BF16), (257, 8192, BF16, F32, F32)])
def test_embedding_and_its_norm_have_the_bits_of_the_two_kernels(ops, T, D, table_dtype, w_dtype, h_dtype):
    """At both sides of every change in the norm's threads: a step's results do not hang on which kernels made its first norm."""
    g = gen(T + D)
    table = torch.randn(50, D, generator=g, device=DEV).to(table_dtype)
    weight = (torch.rand(D, generator=g, device=DEV) + 0.5).to(w_dtype)
    ids = torch.randint(0, 50, (T,), generator=g, device=DEV).to(torch.int32)
    for scale in (1.0, 3.7):
        x, plain, ws, want = torch.empty(T, D, device=DEV), torch.empty(T, D, device=DEV), ops.KernelWorkspace(DEV), torch.empty(T, D, dtype=h_dtype, device=DEV)
        assert ops.embedding_norm(x, table, ids, scale, weight, 1e-5, h_dtype, ws)
        ops.embedding(plain, table, ids, scale)
        ops.rmsnorm(want, plain, weight, 1e-5)
        assert torch.equal(x, plain) and torch.equal(ws.take_left_norm(x, weight, 1e-5).h, want)


@pytest.mark.parametrize("M,D,I", [(1, 128, 512), (8, 2048, 1024), (9, 256, 1024), (16, 3072, 576)])
def test_a_clamped_feed_forward_in_two_kernels(ops, M, D, I):
    g = gen(D + I)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    wg, wu, w_down = ((rnd(I, D) * 2 * D ** -0.5).to(BF16), (rnd(I, D) * 2 * D ** -0.5).to(BF16), (rnd(D, I) * I ** -0.5).to(BF16))
    bg, bu, bd, weight = rnd(I), rnd(I), rnd(D), (torch.rand(D, generator=g, device=DEV) + 0.5).to(BF16)
    pair = lambda a, b: torch.stack([a.view(I // 16, 16, -1), b.view(I // 16, 16, -1)], 1).reshape(2 * I, -1).contiguous()
    w, bias = pair(wg, wu), pair(bg[:, None], bu[:, None]).view(-1)
    x0, h = rnd(M, D), rnd(M, D).to(BF16)
    ws = ops.KernelWorkspace(DEV)
    ws.add_stream_copy(w), ws.add_stream_copy(w_down)
    x, act = x0.clone(), torch.empty(M, I, dtype=BF16, device=DEV)
    assert ops.clamped_mlp(x, act, h, w, bias, 1.5, 1.702, 16, w_down, bd, (weight, 1e-5), ws)
    # the unit has slopes of at most 1.2 (limit + 1) in the gate and limit in the up value; float32 sums of some 1e-6 of their terms
    gd, ud = h.double() @ wg.double().t() + bg, h.double() @ wu.double().t() + bu
    terms = h.double().abs() @ torch.maximum(wg, wu).double().abs().t()
    gd, ud = gd.clamp(max=1.5), ud.clamp(-1.5, 1.5)
    unit = gd * torch.sigmoid(1.702 * gd) * (ud + 1)
    assert ((act.double() - unit).abs() <= ROUND * unit.abs() + 1e-5 * (1 + terms)).all()
    want = x0.double() + bd + act.double() @ w_down.double().t()
    assert ((x.double() - want).abs() <= 1e-5 * (1 + want.abs())).all()
    left = ws.take_left_norm(x, weight, 1e-5)
    assert torch.equal(left.h, (x * weight.float()).to(BF16)) and ws.counts["norms_left"] == 1
    # after a norm whose root is left: the same as after the whole norm, but for where it is rounded
    left2 = ops.LeftNorm(x, weight, 1e-5, left.h, left.sums, left.count)
    again, act2 = x.clone(), torch.empty_like(act)
    assert ops.clamped_mlp(again, act2, left2, w, bias, 1.5, 1.702, 16, w_down, bd, (weight, 1e-5), ws)
    n = x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * weight.double()
    gd, ud = n @ wg.double().t() + bg, n @ wu.double().t() + bu
    off = ROUND * (n.abs() @ torch.maximum(wg.abs(), wu.abs()).double().t())
    gd, ud = gd.clamp(max=1.5), ud.clamp(-1.5, 1.5)
    unit = gd * torch.sigmoid(1.702 * gd) * (ud + 1)
    assert ((act2.double() - unit).abs() <= ROUND * unit.abs() + (1.2 * 2.5 + 1.5) * off + 1e-5).all()
    # no streaming copy of the one or the other: nothing is touched
    bare, before = ops.KernelWorkspace(DEV), x.clone()
    assert not ops.clamped_mlp(x, act, h, w, bias, 1.5, 1.702, 16, w_down, bd, (weight, 1e-5), bare) and torch.equal(x, before)


def test_whoever_else_reads_or_changes_the_stream_finds_it_finished(ops):
    """Another norm, another update of the stream and a reader that takes no left norm."""
    ws, x, want, weight = made(ops, 3, 256, 512)
    other = torch.ones(256, dtype=BF16, device=DEV)
    assert ws.take_left_norm(x, other, 1e-5) is None and ws.left_norm is None          # another norm's: dropped, not handed on
    ws, x, want, weight = made(ops, 3, 256, 512)
    a, w = torch.ones(3, 64, dtype=BF16, device=DEV), torch.ones(256, 64, dtype=BF16, device=DEV)
    ops.gemm(x, a, w, accumulate=True, ws=ws)
    assert ws.left_norm is None and (x.double() - want - 64).abs().max() < 1e-4
    ws, x, want, weight = made(ops, 3, 256, 512)
    left = ws.take_left_norm(x, weight, 1e-5)
    whole = torch.empty(3, 256, dtype=BF16, device=DEV)
    ops.rmsnorm(whole, x, weight, 1e-5)
    assert torch.equal(ops.whole_norm(left), whole)
    wide = torch.randn(40, 256, generator=gen(1), device=DEV)                          # float32 weights: no product here takes it
    got, same = torch.empty(3, 40, device=DEV), torch.empty(3, 40, device=DEV)
    ops.gemm(got, left, wide, ws=ws)
    ops.gemm(same, whole, wide, ws=ws)
    assert torch.equal(got, same)
    # without a streaming copy, or without the caller's word that the norm is next, the update stays in pieces
    for copies, norm in ((False, True), (True, False)):
        ws = ops.KernelWorkspace(DEV)
        w = torch.ones(2048, 512, dtype=BF16, device=DEV)
        if copies:
            ws.add_stream_copy(w)
        x = torch.zeros(2, 2048, device=DEV)
        ops.gemm(x, torch.ones(2, 512, dtype=BF16, device=DEV), w, accumulate=True, may_defer=True, ws=ws,
                 next_norm=(torch.ones(2048, device=DEV), 1e-5) if norm else None)
        assert ws.left_norm is None and ws.pending is not None and ws.counts["norms_left"] == 0


@pytest.mark.parametrize("batch", [1, 5, 12])
def test_a_models_decode_steps_leave_their_norms(tmp_path, batch):
    """A model whose matrices have streaming copies: decode steps leave the norms of whole layers to the next projection,
    with and without graphs, to the same tokens, and their logits are those of the steps that make every norm."""
    from photon_infer_amd import EngineOptions, ModelRunner, StepEntry
    from photon_infer_amd.config import LlamaConfig

    cfg = LlamaConfig.from_dict(dict(architectures=["LlamaForCausalLM"], hidden_size=512, intermediate_size=1024, num_attention_heads=8,
                                     num_key_value_heads=2, head_dim=64, num_hidden_layers=3, vocab_size=1024, max_position_embeddings=512,
                                     rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=True))
    from photon_infer_amd.registry import build_model_spec
    g = gen(9)
    tensors = {s.name: (torch.rand(s.shape, generator=g, device=DEV) + 0.5 if s.role == "norm" else torch.randn(s.shape, generator=g, device=DEV) * 0.04).to(BF16)
               for s in build_model_spec(cfg).tensor_specs()}

    def run(graphs, leave):
        runner = ModelRunner(None, EngineOptions(max_batch=batch, max_cache_tokens=batch * 64, max_model_len=128, use_graphs=graphs, keep_logits=True),
                             config=cfg, tensors=dict(tensors))
        if not leave:
            runner.model.final_norm.leaves_root = False
            for b in runner.model.blocks:
                b.norm1.leaves_root = b.norm2.leaves_root = False
        for i in range(batch):
            runner.admit(i)
            runner.step([StepEntry(i, list(range(3 + i, 12 + 2 * i)))])
        rows = []
        for t in range(4):
            runner.decode_step([StepEntry(i, [17 * t + i], [0]) for i in range(batch)], [0.0] * batch, [0.0] * batch)
            rows.append(runner.decode_logits.clone())
        return torch.stack(rows).double(), runner.workspace.counts

    eager, counts = run(False, True)
    assert counts["norms_left"] > 0, counts
    graphed, _ = run(True, True)
    assert torch.equal(eager, graphed)
    whole, counts = run(False, False)
    assert counts["norms_left"] == 0
    # three layers of bfloat16 activations: their roundings, not their sizes, differ
    assert (eager - whole).norm() <= 0.02 * whole.norm()


def test_every_kernel_that_writes_a_stream_takes_its_norm_back(ops):
    """Behind an update that left its norm, whatever else changes the stream in place, with the workspace or without."""
    D, I = 256, 64
    vec, res = torch.ones(D, device=DEV), lambda: torch.randn(3, D, device=DEV)
    experts = ops.group_entries(torch.tensor([[0, 1], [1, 0], [0, 1]], dtype=torch.int32, device=DEV), 2)
    a, w = torch.ones(3, 64, dtype=BF16, device=DEV), torch.ones(D, 64, dtype=BF16, device=DEV)
    writers = {
        "row bias": lambda x: ops.add_row_bias(x, vec),
        "bias on the way": lambda x: ops.clamped_glu(torch.empty(3, I, dtype=BF16, device=DEV), torch.zeros(3, 2 * I, device=DEV), torch.zeros(I, device=DEV),
                                                     torch.zeros(I, device=DEV), 7.0, 1.7, x, vec),
        "product without the workspace": lambda x: ops.gemm(x, a, w, accumulate=True),
        "branch": lambda x: ops.branch_norm_add(x, res(), vec, 1e-5, 1.0),
        "sandwich": lambda x: ops.sandwich_norm_add(x, res(), (vec, vec), 1e-5),
        "join": lambda x: ops.rms_join(x, res(), vec, 1e-5),
        "experts": lambda x: ops.combine_choices(x, torch.randn(experts.rows, D, device=DEV), None, experts, accumulate=True),
        "torch": lambda x: x.add_(1),
    }
    for name, write in writers.items():
        ws, x, _, weight = made(ops, 3, D, 512)
        assert ws.left_norm is not None, name
        write(x)
        assert ws.take_left_norm(x, weight, 1e-5) is None, name


@pytest.mark.parametrize("M", [1, 16])
@pytest.mark.parametrize("rows", [96, 40, 2056])
def test_readers_without_a_streaming_copy_take_their_ordinary_way(ops, M, rows):
    """A matrix whose rows are no multiple of 16 has no copy, one that nobody named neither: the norm is made whole, and the
    product is, to the bit and in pieces where it is cut, that of the whole norm."""
    N = 512
    ws, x, _, weight = made(ops, M, N, 1024)
    left = ws.take_left_norm(x, weight, 1e-5)
    whole = torch.empty(M, N, dtype=BF16, device=DEV)
    ops.rmsnorm(whole, x, weight, 1e-5)
    w2 = (torch.randn(rows, N, generator=gen(rows), device=DEV) * N ** -0.5).to(BF16)
    for dtype in (F32, BF16):
        made_, want = torch.empty(M, rows, dtype=dtype, device=DEV), torch.empty(M, rows, dtype=dtype, device=DEV)
        ops.gemm(made_, left, w2, ws=ws)
        cut = ws.counts["split_products"]
        ops.gemm(want, whole, w2, ws=ws)
        assert torch.equal(made_, want) and cut > 0 and ws.counts["split_products"] == 2 * cut
        ws.counts["split_products"] = 0
        pieces = [ops.qkv_projection(h, w2, dtype, ws) for h in (left, whole)]
        assert all(isinstance(p, ops.Partials) and p.splits > 1 for p in pieces)
        ws.counts["split_products"] = 0
    if rows % 32 == 0:
        unit, want = torch.empty(M, rows // 2, dtype=BF16, device=DEV), torch.empty(M, rows // 2, dtype=BF16, device=DEV)
        ops.gemm_swiglu(unit, left, w2, 16, ws=ws)
        ops.gemm_swiglu(want, whole, w2, 16, ws=ws)
        assert torch.equal(unit, want)
    assert ws.counts["left_norms_read"] == 0
