"""The absorb weight-gradient kernel at the edges of its token tiles and splits, against fp64.

Tolerance: fp32 sums of exact bf16 products, relative error near sqrt(tokens) 2^-24 (1e-5 with
room); a bf16 result adds its rounding, 2^-9 at most and half of that in the 2-norm."""

from __future__ import annotations

import pytest
import torch

from tests.dsa_cases import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,H,wide_rows,dtype,strided", [
    (1, 1, False, torch.float32, False),
    (31, 3, True, torch.float32, True),
    (33, 2, False, torch.float32, True),
    (64, 128, True, torch.bfloat16, False),
    (1000, 1, False, torch.float32, False),   # three splits, the last one short
    (2100, 16, True, torch.bfloat16, False),  # eight splits
])
def test_absorb_weight_gradient(tokens, H, wide_rows, dtype, strided):
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    g = torch.Generator().manual_seed(tokens)
    a = torch.randn(tokens, H, 128, generator=g).bfloat16()
    b = torch.randn(tokens, H, 576 if strided else 512, generator=g).bfloat16()
    got = ops._absorb_wgrad(a.cuda(), b.cuda()[..., :512], dtype, wide_rows=wide_rows)
    ref = torch.einsum("thi,thj->hij", a.double(), b[..., :512].double())
    ref = ref.transpose(1, 2) if wide_rows else ref
    assert got.dtype == dtype and got.shape == ref.shape
    assert rel_err(got, ref) <= (1e-5 if dtype == torch.float32 else 2.0 ** -9)
