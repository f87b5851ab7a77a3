"""Key ranges of the bfloat16 decode attention that two waves share, and ranges of one wave: against float64 over the pages, at
contexts that leave ranges and second waves without keys, and with the product's own merge of them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F32, BF16 = "cuda", torch.float32, torch.bfloat16
ROUND = 2.0 ** -8


@pytest.fixture(scope="module")
def ops():
    from photon_infer_amd import ops as o
    o.ensure_loaded(BF16)
    return o


@pytest.mark.parametrize("hd,nh,nkv,page,window", [(64, 32, 8, 16, 0), (64, 4, 4, 32, 0), (64, 16, 1, 16, 40), (128, 8, 2, 16, 0), (128, 16, 8, 48, 300)])
@pytest.mark.parametrize("lens", [[1], [129], [300, 1, 33, 64], [1030, 5, 512, 513, 32, 31, 97], [2100, 1]])
def test_ranges_of_two_waves_and_of_one(ops, monkeypatch, hd, nh, nkv, page, window, lens):
    from photon_infer_amd.ops import fast
    from photon_infer_amd.parts import StepContext
    g = torch.Generator(device=DEV).manual_seed(hd + nh + len(lens))
    R, scale, pages = len(lens), hd ** -0.5, [-(-n // page) for n in lens]
    total, width, at = sum(pages), max(pages), 0
    order = torch.randperm(total, generator=torch.Generator().manual_seed(3)).to(torch.int32)
    table = torch.full((R, width), -1, dtype=torch.int32)
    for r, n in enumerate(pages):
        table[r, :n] = order[at:at + n]
        at += n
    table = table.to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ctx = StepContext(T=R, R=R, dtype=BF16, token_ids=i32([0] * R), positions=i32([n - 1 for n in lens]), req_of_token=i32(list(range(R))),
                      q_start=i32(list(range(R + 1))), kv_len=i32(lens), slots=i32(list(range(R))), block_tables={0: table}, logit_rows=i32([]),
                      q_lens=[1] * R, kv_lens=list(lens), max_q_len=1, max_kv_len=max(lens), all_decode=True)
    k, v = torch.randn(total, nkv, page, hd, generator=g, device=DEV).to(BF16), torch.randn(total, nkv, hd, page, generator=g, device=DEV).to(BF16)
    proj = torch.randn(2, R, (nh + 2 * nkv) * hd, generator=g, device=DEV)
    qkv = ops.Partials(proj, 2, R, proj.shape[2])
    angle = torch.rand(R, hd // 2, generator=g, device=DEV) * 6.28
    rotary = (torch.cat([angle.cos(), angle.sin()], 1).contiguous(), hd, False)
    ws = ops.KernelWorkspace(DEV)
    splits = fast.decode_splits(R, nkv, max(lens))
    results, shared = {}, False
    monkeypatch.setattr(fast, "RANGES_SHARED_UP_TO", 16)
    for name, share in (("two waves", 2), ("one wave", 1 << 30)):
        monkeypatch.setattr(fast, "RANGES_TO_SHARE", share)
        k1, v1, q = k.clone(), v.clone(), torch.empty(R, nh * hd, dtype=BF16, device=DEV)
        fused, apart, merged = (torch.full((R, nh * hd), 7.0, dtype=BF16, device=DEV) for _ in range(3))
        assert ops.decode_attention_from_projection(fused, qkv, ctx, rotary, nh, nkv, hd, k1, v1, table, page, scale, window, True, ws) is True
        ops.rope_kv_write(q, None, None, ctx.positions, ctx.req_of_token, rotary, nh, nkv, hd, k1, v1, table, page, pieces=qkv, write_kv=True)
        ops.paged_attention(apart, q, k1, v1, table, ctx, nh, nkv, hd, page, scale, window, ws)
        assert torch.equal(fused, apart), name
        left = ops.decode_attention_from_projection(merged, qkv, ctx, rotary, nh, nkv, hd, k1, v1, table, page, scale, window, True, ws, leave_ranges=1 << 20)
        ranges, waves = fast.decode_range_waves(splits, R, nkv)
        fits = R * -(-splits // 2) * nkv <= fast.compute_units()
        assert (ranges, waves) == ((-(-splits // 2), 2) if share == 2 and splits > 1 and fits else (splits, 1))
        shared |= waves == 2
        if ranges > 1:
            assert isinstance(left, ops.KeyRanges) and left.count == ranges
            fast.merge_ranges(merged, left)
        else:
            assert left is True
        assert torch.equal(merged, fused), name
        results[name] = fused
    assert shared or splits == 1 or R * -(-splits // 2) * nkv > fast.compute_units()
    for r, n in enumerate(lens):
        lo = max(0, n - window) if window else 0
        mine = table[r, :pages[r]].long()
        keys = k1[mine].transpose(0, 1).reshape(nkv, -1, hd)[:, lo:n].double()
        values = v1[mine].permute(1, 0, 3, 2).reshape(nkv, -1, hd)[:, lo:n].double()
        w = torch.softmax(q[r].view(nkv, nh // nkv, hd).double() @ keys.transpose(1, 2) * scale, -1)
        want, size = (w @ values).reshape(-1), (w @ values.abs()).reshape(-1)
        # weights are rounded to bfloat16 for the matrix instruction and so is the result
        for name, got in results.items():
            assert ((got[r].double() - want).abs() <= ROUND * (1.05 * size + want.abs()) + 1e-5).all(), (name, r, n)
