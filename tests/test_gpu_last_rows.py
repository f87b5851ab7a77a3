"""The last block of a step takes in only the tokens whose logits are wanted: the same logits, the same caches and states."""
import pytest
import torch

import tiny_dokanex
import tiny_models
import tiny_rorevik
from gpu_tools import DEV, attention_ctx, paged, randn
from tiny_models import random_tokens

pytestmark = pytest.mark.gpu

# single tokens in a step: enough that it is cut where less than half of them are wanted (ops.STREAMED_TOKENS)
SINGLES = {"float32": 36, "bfloat16": 130}


def logits_of_steps(folder, dtype, monkeypatch, cuts=True):
    """Logits of steps that want one token of many, none, some; then of steps of single tokens, which want every one; and which of
    the steps ended in rows.  ``cuts`` False: the last block's mixer says nothing of rows, and what follows it alone is cut."""
    from photon_infer_amd import EngineOptions, ModelRunner, StepEntry
    from photon_infer_amd.parts import PreNormBlock

    n = SINGLES[dtype]
    runner = ModelRunner(folder, EngineOptions(dtype=dtype, max_batch=n + 6, max_cache_tokens=32 * (n + 40), max_model_len=256, use_graphs=False))
    long, other, short = random_tokens(150, 200, 1), random_tokens(140, 200, 3), random_tokens(41, 200, 2)
    few = [f"few {i}" for i in range(n)]
    for rid in ["a", "b", "c"] + few:
        runner.admit(rid)
    ended, forward_last = [], PreNormBlock.forward_last

    def seen(self, x, ctx, cache):
        if not cuts:
            monkeypatch.setattr(type(self.mixer), "cuts_rows", False)
        ended.append((ctx.T, ctx.logit_rows.shape[0]))
        return forward_last(self, x, ctx, cache)

    with monkeypatch.context() as m:
        m.setattr(PreNormBlock, "forward_last", seen)
        m.setattr(torch.Tensor, "index_select", None)      # a library's kernel: loading its module took the first prompt 70 to 140 ms
        cut = [runner.step([StepEntry("a", long, [149])]),
               runner.step([StepEntry("b", short, [])]),
               runner.step([StepEntry("c", other, [139, 5]), StepEntry("b", [7], []), StepEntry("a", [9], [0])]),
               runner.step([StepEntry(rid, short[i % 39:i % 39 + 2], []) for i, rid in enumerate(few)]),
               runner.step([StepEntry(rid, [3 + i], [0] if i % 7 == 2 else []) for i, rid in enumerate(few)])]
        whole = [runner.step([StepEntry("b", [11], [0]), StepEntry("c", [12], [0]), StepEntry("a", [13], [0])]),
                 runner.step([StepEntry(rid, [20 + i], [0]) for i, rid in enumerate(few[:24])])]
    assert cut[1] is None and cut[3] is None
    wanted = [(150, 1), (41, 0), (142, 3), (2 * n, 0), (n, len(range(2, n, 7)))]
    return [t.clone() for t in cut if t is not None], [t.clone() for t in whole], ended, wanted


@pytest.mark.parametrize("cuts", [True, False], ids=["mixer and rest", "rest"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("tiny,name", [(tiny_models, "D"), (tiny_models, "F"), (tiny_models, "G"), (tiny_rorevik, "B"), (tiny_rorevik, "C"),
                                       (tiny_dokanex, "B"), (tiny_dokanex, "C")],
                         ids=lambda v: getattr(v, "__name__", v))
def test_rows_that_nobody_reads_change_nothing(tmp_path, monkeypatch, tiny, name, dtype, cuts):
    from photon_infer_amd.parts.model import DecoderModel

    folder = tiny.make_model_dir(tmp_path, name)
    cut, whole, ended, wanted = logits_of_steps(folder, dtype, monkeypatch, cuts)
    assert ended == wanted
    monkeypatch.setattr(DecoderModel, "_ends_in_rows", staticmethod(lambda block, ctx: False))
    cut_ref, whole_ref, ended, _ = logits_of_steps(folder, dtype, monkeypatch)
    assert ended == []
    # what later steps read was written before anything was cut: the same bits
    assert all(torch.equal(a, b) for a, b in zip(whole, whole_ref))
    for got, ref in zip(cut, cut_ref):
        assert got.shape == ref.shape and torch.isfinite(got).all()
        # products of fewer rows add in another order: float32 rounding, and in bfloat16 now and then an activation of the last
        # block by one place (2^-8 of it), of which a logit adds up many with either sign
        bound = 3e-5 if dtype == "float32" else 2.0 ** -6
        assert (got - ref).abs().max() <= bound * max(1.0, ref.abs().max().item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,D,M", [(1, 1, 1), (40, 2048, 1), (40, 7, 5), (300, 1030, 150), (9, 4100, 3), (33, 64, 0)])
def test_copies_of_rows(T, D, M, dtype):
    """Widths and addresses for units of 16, 4 and 2 bytes, strides, one, two and three tensors, rows that are not there."""
    from photon_infer_amd import ops
    from photon_infer_amd.errors import KernelError
    wide, x = randn(T, D + 9, seed=1).to(dtype).to(DEV), randn(T, D + 3, seed=2).float().to(DEV)
    rows = torch.randperm(T, generator=torch.Generator().manual_seed(3))[:M].to(torch.int32).to(DEV)
    for tensors in ([x], [x, wide], [wide[:, 8:8 + D], x], [wide[:, 1:1 + D], x[:, 1:], wide]):
        made = ops.copy_rows(rows, *tensors)
        assert len(made) == len(tensors)
        assert all(torch.equal(m, t[rows.long()]) and m.is_contiguous() for m, t in zip(made, tensors))
    if M:
        rows[0], rows[-1] = T, -1 if M > 1 else T
        made = ops.copy_rows(rows, x, wide)
        for m, t in zip(made, (x, wide)):
            assert m[0].isnan().all() and m[-1].isnan().all() and torch.equal(m[1:-1], t[rows[1:-1].long()])
    with pytest.raises(KernelError, match="columns side by side"):
        ops.copy_rows(rows, x[:, :2 * (D // 2):2] if D > 1 else x.double())


# mixers that say that they cut rows and that no design above has in such a block: (kind, parameters)
MIXERS_ALONE = [
    ("attention", dict(num_heads=4, num_kv_heads=2, head_dim=32, names=("q", "k", "v", "o"), any_head_size=True, qkv_bias=True, values_are_keys=True,
                       head_norm_eps=1e-5, feature_gate="g")),
    ("gated_delta_rule", dict(num_heads=4, num_kv_heads=2, key_dim=64, value_dim=32, conv_taps=4, eps=1e-5)),
]


@pytest.mark.parametrize("cuts", [True, False], ids=["mixer and rest", "rest"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["float32", "bfloat16"])
@pytest.mark.parametrize("kind,params", MIXERS_ALONE, ids=[k for k, _ in MIXERS_ALONE])
def test_a_block_that_ends_in_rows_is_the_block(monkeypatch, kind, params, dtype, cuts):
    """The wanted rows of the whole block's stream, and the same bits in what the mixer keeps."""
    from photon_infer_amd import ops
    from photon_infer_amd.parts import MIXERS, LayerCache, PreNormBlock, RMSNorm, SwiGLU

    D, lens, page = 128, [70, 90], 16
    mixer = MIXERS.make(kind, hidden_size=D, **params)
    block = PreNormBlock(("n1.", RMSNorm(D, 1e-5)), ("m.", mixer), ("n2.", RMSNorm(D, 1e-5)), ("f.", SwiGLU(D, 192)))
    tensors = {s.name: randn(*s.shape, seed=i, scale=0.5 if len(s.shape) == 1 else s.shape[-1] ** -0.5) for i, s in enumerate(block.tensor_specs())}
    block.load({n: t.to(dtype if t.dim() == 2 else torch.float32).to(DEV) for n, t in tensors.items()}, dtype, torch.device(DEV))
    assert block.ends_in_rows and mixer.cuts_rows
    monkeypatch.setattr(type(mixer), "cuts_rows", cuts)
    table, pages = paged(lens, page, seed=2)
    spec, x = mixer.cache_spec(), randn(sum(lens), D, seed=99).float().to(DEV)

    def run(rows, last):
        if hasattr(spec, "tensors"):
            kept = {t.name: torch.zeros((pages, *t.page_shape(page)), dtype=dtype, device=DEV) for t in spec.tensors}
            cache = LayerCache(group=0, k=kept["k"], v=kept["v"], page_size=page, writes=True, tensors=kept)
        elif hasattr(spec, "shape"):
            kept = {"state": torch.zeros((3, *spec.shape), dtype=torch.float32, device=DEV)}
            cache = LayerCache(state=kept["state"])
        else:
            G, d = params["num_kv_heads"], params["head_dim"]
            kept = {"k": torch.zeros((pages, G, page, d), dtype=dtype, device=DEV), "v": torch.zeros((pages, G, d, page), dtype=dtype, device=DEV)}
            cache = LayerCache(group=0, k=kept["k"], v=kept["v"], page_size=page, writes=True, tensors=kept)
        ctx = attention_ctx(lens, lens, dtype)
        ctx.block_tables, ctx.workspace, ctx.slots = {0: table}, ops.KernelWorkspace(DEV), torch.tensor([2, 0], dtype=torch.int32, device=DEV)
        ctx.logit_rows = torch.tensor(rows, dtype=torch.int32, device=DEV)
        ctx.may_defer = ctx.after_block_consumes = False
        ctx.next_norm = ctx.after_block_norm = ctx.read_rows = None
        stream = x.clone()
        if last:
            stream = block.forward_last(stream, ctx, cache)
        else:
            block.forward(stream, ctx, cache)
            stream = stream[rows]
        assert not ctx.may_defer and ctx.read_rows is None and ctx.workspace.take_pending(stream) is None
        return stream, kept

    for rows in ([159], [], [69, 3, 100], list(range(0, 160, 2))):
        (got, kept), (ref, kept_ref) = run(rows, True), run(rows, False)
        assert got.shape == (len(rows), D) and all(torch.equal(kept[n], kept_ref[n]) for n in kept)
        if rows:
            bound = 3e-5 if dtype == torch.float32 else 2.0 ** -6          # as above
            assert (got - ref).abs().max() <= bound * max(1.0, ref.abs().max().item())
