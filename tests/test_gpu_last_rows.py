"""The last block of a step takes in only the tokens whose logits are wanted: the same logits, the same caches and states."""
import pytest
import torch

import tiny_dokanex
import tiny_models
import tiny_rorevik
import tiny_semezen
from tiny_models import random_tokens

pytestmark = pytest.mark.gpu


def logits_of_steps(folder, dtype):
    """Logits of steps that want one token of many, none, some; then of steps of single tokens, which want every one."""
    from photon_infer_amd import EngineOptions, ModelRunner, StepEntry

    runner = ModelRunner(folder, EngineOptions(dtype=dtype, max_batch=24, max_cache_tokens=2048, max_model_len=256, use_graphs=False))
    long, other, short = random_tokens(150, 200, 1), random_tokens(140, 200, 3), random_tokens(41, 200, 2)
    few = [f"few {i}" for i in range(18)]
    for rid in ["a", "b", "c"] + few:
        runner.admit(rid)
    cut = [runner.step([StepEntry("a", long, [149])]),
           runner.step([StepEntry("b", short, [])]),
           runner.step([StepEntry("c", other, [139, 5]), StepEntry("b", [7], []), StepEntry("a", [9], [0])]),
           runner.step([StepEntry(rid, short[i:i + 2], []) for i, rid in enumerate(few)]),
           runner.step([StepEntry(rid, [3 + i], [0] if i % 7 == 2 else []) for i, rid in enumerate(few)])]
    whole = [runner.step([StepEntry("b", [11], [0]), StepEntry("c", [12], [0]), StepEntry("a", [13], [0])]),
             runner.step([StepEntry(rid, [20 + i], [0]) for i, rid in enumerate(few)])]
    assert cut[1] is None and cut[3] is None
    return [t.clone() for t in cut if t is not None], [t.clone() for t in whole]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("tiny,name", [(tiny_models, "D"), (tiny_models, "F"), (tiny_models, "G"), (tiny_rorevik, "B"), (tiny_rorevik, "C"),
                                       (tiny_dokanex, "B"), (tiny_dokanex, "D"), (tiny_semezen, "B")],
                         ids=lambda v: getattr(v, "__name__", v))
def test_rows_that_nobody_reads_change_nothing(tmp_path, monkeypatch, tiny, name, dtype):
    from photon_infer_amd.parts.model import DecoderModel

    folder = tiny.make_model_dir(tmp_path, name)
    cut, whole = logits_of_steps(folder, dtype)
    monkeypatch.setattr(DecoderModel, "_ends_in_rows", staticmethod(lambda block, ctx: False))
    cut_ref, whole_ref = logits_of_steps(folder, dtype)
    # what later steps read was written before anything was cut: the same bits
    assert all(torch.equal(a, b) for a, b in zip(whole, whole_ref))
    for got, ref in zip(cut, cut_ref):
        assert got.shape == ref.shape and torch.isfinite(got).all()
        # products of fewer rows add in another order: float32 rounding, and in bfloat16 now and then an activation of the last
        # block by one place (2^-8 of it), of which a logit adds up many with either sign
        bound = 3e-5 if dtype == "float32" else 2.0 ** -6
        assert (got - ref).abs().max() <= bound * max(1.0, ref.abs().max().item())
