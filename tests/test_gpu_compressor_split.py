"""Block compressor with a block's slots shared by several lanes.

Sizes: every split of lanes and parts (rows inside one wave, of one wave, of several), part
lengths that do not divide the ratio, several blocks in one wave and one in a workgroup, TND
starts with and without a previous block.

fp32 error: a feature is a weighted mean of n slots whose weights are off by a few ulp each
(expf, at most log2(n) + n / 4 rescalings) and whose sum adds n roundings, all relative to
max |x|: below (2 n) 2^-24 = 1.6e-5 at n = 128, and 1e-5 of the largest pooled value is
asked.  With the norm the pooled row is rounded to bf16 first, and so is the output: a value
at a rounding boundary may move by one bf16 step in each, 2 * 2^-8."""

import pytest
import torch

from oracle import dsa_oracle as O
from tests.dsa_cases import rel_err

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _ops():
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    return ops


def _inputs(rows, width, r, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*rows, width, generator=g), torch.randn(*rows, width, generator=g),
            0.02 * torch.randn(r, width, generator=g), torch.rand(width, generator=g) + 0.5)


@pytest.mark.parametrize("B,nb,D,r,overlap", [
    (1, 1, 512, 128, False), (1, 3, 128, 128, False), (2, 33, 64, 128, False), (1, 65, 128, 128, False),
    (1, 65, 512, 16, False), (1, 70, 1024, 19, False), (1, 2, 1024, 8, True), (1, 5, 4, 128, False),
    (2, 40, 32, 8, True), (1, 3, 256, 130, True), (1, 80, 16, 9, False)])
@pytest.mark.parametrize("norm", [False, True])
def test_split_block(B, nb, D, r, overlap, norm):
    kv, sc, ape, w = _inputs((B, nb * r), D * (2 if overlap else 1), r, nb + D + r)
    w = w[:D] if norm else None
    # whole parts without weight, the first slot among them
    sc[:, 0:r // 2, min(3, D - 1)] = -float("inf")
    rd = min(D, 64)
    ang = torch.outer(torch.arange(nb * r).float(), 0.01 ** (torch.arange(rd // 2).float() / rd))
    fc = torch.polar(torch.ones_like(ang), ang)
    got = _ops().compressor_pool(kv.to(DEV), sc.to(DEV), ape.to(DEV), r, overlap=overlap,
                                 norm_weight=None if w is None else w.to(DEV), freqs_cis=fc.to(DEV), rope_dim=rd).cpu()
    if norm:
        ref = O.compressor_pool(kv, sc, ape, r, overlap=overlap, norm_weight=w, out_dtype=torch.bfloat16,
                                freqs_cis=fc, rope_dim=rd)
        assert got.dtype == torch.bfloat16
    else:
        ref = O.compressor_pool(kv.double(), sc.double(), ape.double(), r, overlap=overlap, freqs_cis=fc, rope_dim=rd)
    assert rel_err(got.float(), ref) <= (2 * 2.0 ** -8 if norm else 1e-5)


@pytest.mark.parametrize("D,r,overlap", [(512, 128, False), (128, 16, True), (256, 24, True)])
def test_split_block_tnd(D, r, overlap):
    from torchtitan_npu_simulator_amd import tnd

    pos = torch.cat([torch.arange(5, 5 + 3 * r), torch.arange(0, r + 3), torch.arange(0, 3), torch.arange(0, 4 * r)])
    kv, sc, ape, w = _inputs((pos.numel(),), D * (2 if overlap else 1), r, D + r)
    w = w[:D]
    bs = tnd.compressed_block_starts(pos, r)
    args = [t.to(DEV) for t in (kv, sc, ape)]
    got = _ops().compressor_pool_tnd(*args, r, bs.to(DEV), pos.to(DEV), overlap=overlap).cpu()
    ref = O.compressor_pool_tnd(kv.double(), sc.double(), ape.double(), r, bs, pos, overlap=overlap)
    assert rel_err(got, ref) <= 1e-5
    got = _ops().compressor_pool_tnd(*args, r, bs.to(DEV), pos.to(DEV), overlap=overlap, norm_weight=w.to(DEV)).cpu()
    ref = O.compressor_pool_tnd(kv, sc, ape, r, bs, pos, overlap=overlap, norm_weight=w, out_dtype=torch.bfloat16)
    assert rel_err(got.float(), ref) <= 2 * 2.0 ** -8
