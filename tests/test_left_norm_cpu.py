"""Norms whose root is left to their reader: when what was left still counts (CPU)."""
import pytest
import torch

from photon_infer_amd import ops
from photon_infer_amd.errors import KernelError
from photon_infer_amd.ops.workspace import LeftNorm

F32, BF16 = torch.float32, torch.bfloat16


def left_in(ws, x, weight):
    ws.left_norm = LeftNorm(x, weight, 1e-5, (x * weight).to(BF16), (x ** 2).sum(1, keepdim=True), 1)
    return ws.left_norm


def test_a_stream_that_somebody_wrote_has_no_norm_left():
    ws, weight = ops.KernelWorkspace("cpu"), torch.ones(8)
    for write in (lambda x: x.add_(1), lambda x: x[1].mul_(2), lambda x: x.view(-1)[:3].zero_(), lambda x: x.copy_(torch.ones(2, 8)), ops._changes):
        x = torch.randn(2, 8)
        left = left_in(ws, x, weight)
        assert ws.take_left_norm(x, weight, 1e-5) is left and ws.left_norm is None
        left = left_in(ws, x, weight)
        write(x)
        assert ws.take_left_norm(x, weight, 1e-5) is None and ws.left_norm is None
        with pytest.raises(KernelError, match="written since"):
            ops.whole_norm(left)


def test_tensors_that_count_no_versions_keep_their_norms():
    with torch.inference_mode():
        ws, weight, x = ops.KernelWorkspace("cpu"), torch.ones(8), torch.randn(2, 8)
        left = left_in(ws, x, weight)
        ops._changes(x)                                  # not an error
        assert ws.take_left_norm(x, weight, 1e-5) is left
