"""The V4 slot-index kernel equals the torch construction, entry by entry."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,win_left,win_right,ratio,n_cmp,K", [
    (1, 1, 0, 0, 1, 0, 0),          # the smallest: the token itself
    (2, 130, 127, 0, 4, 32, 20),    # selected rows
    (1, 300, 15, 3, 128, 2, None),  # every causal block, a window ahead
    (1, 257, 400, 0, 4, 64, 1),     # a window longer than the sequence
])
def test_v4_indices_kernel(B, S, win_left, win_right, ratio, n_cmp, K):
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    cmp = None
    if K:
        cmp = torch.randint(-1, S + n_cmp, (B, S, K), generator=torch.Generator().manual_seed(S), dtype=torch.int32)
    kw = dict(win_left=win_left, win_right=win_right, cmp_ratio=ratio, n_cmp=n_cmp)
    ref = ops.v4_attention_indices(B, S, "cpu", cmp_indices=cmp, **kw)
    got = ops.v4_attention_indices(B, S, torch.device("cuda"), cmp_indices=None if cmp is None else cmp.cuda(), **kw)
    assert got.dtype == torch.int32 and torch.equal(got.cpu(), ref)


def test_v4_indices_left_to_torch(monkeypatch):
    """More batch elements than a grid takes, and indices on another GPU (here: another one is made
    to look current), do not reach the kernel."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    cmp = torch.randint(0, 8, (65536, 1, 2), dtype=torch.int32)
    kw = dict(win_left=0, cmp_ratio=4, n_cmp=4)
    ref = ops.v4_attention_indices(65536, 1, "cpu", cmp_indices=cmp, **kw)
    assert torch.equal(ops.v4_attention_indices(65536, 1, "cuda", cmp_indices=cmp.cuda(), **kw).cpu(), ref)

    def no_kernel():
        raise AssertionError("the kernel was asked for")

    small = cmp[:3].cuda()
    monkeypatch.setattr(ops, "load_library", no_kernel)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    got = ops.v4_attention_indices(3, 1, "cuda", cmp_indices=small, **kw)
    assert torch.equal(got.cpu(), ref[:3])
