"""Decode attention of the float32 path from the q|k|v projection: against the separate kernels (the same cache, bit for bit) and
against float64 attention over the pages, at the edges of its tiles of 16 keys, four waves and key ranges."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F32 = "cuda", torch.float32


@pytest.fixture(scope="module")
def ops():
    from photon_infer_amd import ops as o
    o.ensure_loaded(F32)
    return o


def step(ops, lens, hd, nh, nkv, page, pieces, seed, extra=0):
    from photon_infer_amd.parts import StepContext
    g = torch.Generator(device=DEV).manual_seed(seed)
    R = len(lens)
    pages = [-(-n // page) for n in lens]
    total, width = sum(pages), max(pages)
    order = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    table = torch.full((R, width), -1, dtype=torch.int32)
    at = 0
    for r, n in enumerate(pages):
        table[r, :n] = order[at:at + n]
        at += n
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ctx = StepContext(T=R, R=R, dtype=F32, token_ids=i32([0] * R), positions=i32([n - 1 for n in lens]), req_of_token=i32(list(range(R))),
                      q_start=i32(list(range(R + 1))), kv_len=i32(lens), slots=i32(list(range(R))), block_tables={0: table.to(DEV)}, logit_rows=i32([]),
                      q_lens=[1] * R, kv_lens=list(lens), max_q_len=1, max_kv_len=max(lens), all_decode=True)
    k = torch.randn(total, nkv, page, hd, generator=g, device=DEV)
    v = torch.randn(total, nkv, hd, page, generator=g, device=DEV)
    for r, n in enumerate(lens):                     # slots behind a request's last token hold what a later one left: not finite here
        if n % page:
            k[table[r, pages[r] - 1], :, n % page:] = float("nan")
            v[table[r, pages[r] - 1], :, :, n % page:] = float("inf")
    cols = (nh + 2 * nkv) * hd + extra
    proj = torch.randn(pieces, R, cols, generator=g, device=DEV) / pieces ** 0.5
    rot = torch.rand(R, hd // 2, generator=g, device=DEV) * 6.28
    return ctx, table.to(DEV), k, v, proj, torch.cat([rot.cos(), rot.sin()], 1).contiguous()


@pytest.mark.parametrize("hd,nh,nkv,page,window,pieces", [(64, 32, 8, 16, 0, 5), (64, 4, 4, 16, 0, 1), (64, 6, 2, 32, 40, 2), (128, 8, 4, 16, 0, 3), (128, 16, 2, 48, 100, 1),
                                                          (64, 8, 1, 16, 0, 1)])
@pytest.mark.parametrize("lens", [[1], [16, 17, 1, 64, 65], [70, 63, 49, 31, 15, 128, 129, 2], [1030, 511, 512, 513]])
def test_against_the_separate_kernels_and_float64(ops, hd, nh, nkv, page, window, pieces, lens):
    ctx, table, k, v, proj, rot = step(ops, lens, hd, nh, nkv, page, pieces, hd + nh + len(lens), extra=12)
    R, scale = len(lens), hd ** -0.5
    qkv = ops.Partials(proj, pieces, R, proj.shape[2]) if pieces > 1 else proj[0]
    rotary = (rot, hd, False)
    # rotation and cache write by the kernel of their own
    k1, v1, q = k.clone(), v.clone(), torch.empty(R, nh * hd, device=DEV)
    parts = qkv if pieces > 1 else ops.Partials(proj, 1, R, proj.shape[2])
    ops.rope_kv_write(q, None, None, ctx.positions, ctx.req_of_token, rotary, nh, nkv, hd, k1, v1, table, page, pieces=parts, write_kv=True)
    apart = torch.empty(R, nh * hd, device=DEV)
    ops.paged_attention(apart, q, k1, v1, table, ctx, nh, nkv, hd, page, scale, window)
    k2, v2, got = k.clone(), v.clone(), torch.full((R, nh * hd), 7.0, device=DEV)
    assert ops.decode_attention_from_projection(got, qkv, ctx, rotary, nh, nkv, hd, k2, v2, table, page, scale, window, True) is True
    bits = lambda t: t.view(torch.int32)
    assert torch.equal(bits(k2), bits(k1)) and torch.equal(bits(v2), bits(v1))
    for r, n in enumerate(lens):
        lo = max(0, n - window) if window else 0
        pages = table[r, :-(-n // page)].long()
        keys = k1[pages].transpose(0, 1).reshape(nkv, -1, hd)[:, lo:n].double()
        values = v1[pages].permute(1, 0, 3, 2).reshape(nkv, -1, hd)[:, lo:n].double()
        qq = q[r].view(nkv, nh // nkv, hd).double()
        w = torch.softmax(qq @ keys.transpose(1, 2) * scale, -1)
        want, size = (w @ values).reshape(-1), (w @ values.abs()).reshape(-1)
        # scores of hd products, off by hd 2^-24 of their terms' sum; weights by as much of themselves; sums of the keys in chains
        # of 16 per wave
        slack = 2.0 ** -24 * (2 * scale * (qq.abs() @ keys.abs().transpose(1, 2)).amax() * hd ** 0.5 + 40) * size
        for name, t in (("from the projection", got), ("apart", apart)):
            assert ((t[r].double() - want).abs() <= slack).all(), (name, r, n, ((t[r].double() - want).abs() / slack).max())
    # a layer that reads another's cache: queries only, nothing written
    k3, v3, again = k2.clone(), v2.clone(), torch.empty(R, nh * hd, device=DEV)
    assert ops.decode_attention_from_projection(again, qkv, ctx, rotary, nh, nkv, hd, k3, v3, table, page, scale, window, False) is True
    assert torch.equal(again, got) and torch.equal(bits(k3), bits(k2))


def test_what_it_leaves_to_the_separate_kernels(ops):
    for hd, nh, nkv in ((48, 4, 2), (64, 10, 2), (96, 3, 3)):
        ctx, table, k, v, proj, rot = step(ops, [20, 3], hd, nh, nkv, 16, 1, 1)
        assert ops.decode_attention_from_projection(torch.empty(2, nh * hd, device=DEV), proj[0], ctx, (rot, hd, False), nh, nkv, hd, k, v, table, 16, 0.1, 0, True) is False
