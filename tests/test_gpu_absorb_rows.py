"""The absorb products on the weight as stored, [H, K, N], against the transposed-weight form.

The same products are added in the same order, so the outputs are the same bit for bit; sizes
are one token, the edges of a wave's 64-token tiles and several chunks per workgroup."""

import pytest
import torch

from tests.dsa_cases import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N", [(128, 512), (512, 128)])
@pytest.mark.parametrize("tokens,H,append", [(1, 1, 64), (63, 3, 0), (65, 128, 64), (513, 2, 0), (700, 300, 8)])
def test_absorb_rows_equals_transposed_weight(tokens, H, append, K, N):
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    g = torch.Generator(device="cuda").manual_seed(tokens + K)
    a = torch.randn(tokens, H, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(H, K, N, generator=g, device="cuda").bfloat16()
    e = torch.randn(tokens, H, append, generator=g, device="cuda").bfloat16() if append else None
    got = ops._absorb(a, w, e, k_rows=True)
    assert torch.equal(got, ops.mla_absorb(a, w.transpose(1, 2).contiguous(), append=e))
    ref = torch.bmm(a[:, :2].transpose(0, 1).double(), w[:2].double()).transpose(0, 1)
    assert rel_err(got[:, :2, :N].cpu(), ref.cpu()) <= 2.0 ** -8  # (fp32 sums, one bf16 rounding)


def test_absorb_rows_takes_an_unaligned_weight():
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    buf = torch.randn(2 * 128 * 512 + 1, device="cuda").bfloat16()
    w = buf[1:].view(2, 128, 512)
    a = torch.randn(5, 2, 128, device="cuda").bfloat16()
    pe = torch.randn(5, 2, 64, device="cuda").bfloat16()
    assert torch.equal(ops.mla_absorb_q(a, pe, w), ops.mla_absorb_q(a, pe, w.clone()))
