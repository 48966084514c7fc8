"""Attention with fewer heads than a workgroup's rows: several tokens share one workgroup
(csrc/attn_pack.h), forward, backward and mass against the fp64 oracle and the one-token
kernels, at group tails, odd head counts, holes, repeats and both row widths."""

from __future__ import annotations

import math

import pytest
import torch

from oracle import dsa_oracle as O
from tests.dsa_cases import rand_indices, rel_err

TOL = 2e-2  # bf16 attention and its gradients


def test_packed_workspace_rule():
    """The packed path takes bf16 calls of at most 64 heads whose tokens fill the chip."""
    from torchtitan_npu_simulator_amd import _lib

    size = _lib.load_library().dsa_sparse_mla_fwd_workspace_size
    assert size(_lib.DSA_BF16, 1, 512, 512, 16, 64, 0) > 0
    assert size(_lib.DSA_BF16, 1, 1024, 512, 16, 64, 1 << 40) > 0
    for dt, b, s, s_kv, h, off in ((_lib.DSA_BF16, 1, 512, 512, 65, 0), (_lib.DSA_BF16, 1, 511, 511, 16, 0),
                                   (_lib.DSA_F32, 1, 512, 512, 16, 0), (_lib.DSA_BF16, 1, 512, (1 << 17) + 1, 16, 0),
                                   (_lib.DSA_BF16, 1, 1023, 512, 16, 1 << 40)):
        assert size(dt, b, s, s_kv, h, 64, off) == 0


def _unpacked(ops, q, kv, idx, scale, q_offset):
    """The same forward through the entry point without a workspace (one token per workgroup)."""
    from torchtitan_npu_simulator_amd import _lib

    B, S, H, D = q.shape
    out = torch.empty(B, S, H, 512, dtype=q.dtype, device=q.device)
    smax, ssum = (torch.empty(B, S, H, device=q.device) for _ in range(2))
    _lib.check(_lib.load_library().dsa_sparse_mla_fwd(
        _lib.ptr(q), _lib.ptr(kv), _lib.ptr(idx), _lib.ptr(out), _lib.ptr(smax), _lib.ptr(ssum), _lib.DSA_BF16, B, S,
        kv.shape[1], H, D, 512, idx.shape[-1], scale, q_offset, _lib.stream_of(q.device)), "dsa_sparse_mla_fwd")
    return out, smax, ssum


def _unpacked_mass(q, kv, idx, smax, ssum, scale, q_offset):
    """The mass through the entry point without a workspace."""
    from torchtitan_npu_simulator_amd import _lib

    B, S, H, D = q.shape
    mass = torch.empty(B, S, idx.shape[-1], device=q.device)
    _lib.check(_lib.load_library().dsa_attn_mass(
        _lib.ptr(q), _lib.ptr(kv), _lib.ptr(idx), _lib.ptr(smax), _lib.ptr(ssum), _lib.ptr(mass), _lib.DSA_BF16, B, S,
        kv.shape[1], H, D, idx.shape[-1], scale, q_offset, _lib.stream_of(q.device)), "dsa_attn_mass")
    return mass


@pytest.mark.gpu
@pytest.mark.parametrize("H,S,K,B,q_offset,width,repeat", [
    (16, 517, 64, 1, 0, 576, False),   # three tokens per group, a tail of one
    (8, 1031, 33, 1, 0, 576, False),   # heads padded to 16 rows, odd slot count
    (24, 300, 96, 2, 37, 576, False),  # heads padded to 32 rows, two batch elements, a key prefix
    (64, 601, 128, 1, 0, 576, False),  # two tokens per group, every row used, an odd tail
    (40, 530, 40, 1, 0, 512, False),   # 48 rows per token: a wave's rows belong to two tokens
    (16, 600, 48, 1, 0, 576, True),    # a key twice in one token's list counts twice
])
def test_packed_attention(H, S, K, B, q_offset, width, repeat):
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    s_kv = S + q_offset
    g = torch.Generator().manual_seed(H + S)
    q = torch.randn(B, S, H, width, generator=g).bfloat16()
    kv = torch.randn(B, s_kv, width, generator=g).bfloat16()
    dout = torch.randn(B, S, H, 512, generator=g).bfloat16()
    idx = torch.cat([rand_indices(S, K, q_offset=q_offset, seed=b, shuffle=True, holes=0.2) for b in range(B)])
    if repeat:
        idx[:, 100:400, 5] = idx[:, 100:400, 9]
        idx[:, 100:400, 11] = idx[:, 100:400, 9]
    scale = 1.0 / math.sqrt(width)
    qd, kvd, idd, dod = q.cuda(), kv.cuda(), idx.cuda(), dout.cuda()
    assert _lib.load_library().dsa_sparse_mla_fwd_workspace_size(_lib.DSA_BF16, B, S, s_kv, H, K, q_offset) > 0
    out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, scale, q_offset=q_offset)
    dq, dkv, mass = ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, scale, q_offset=q_offset, return_mass=True)
    again = ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, scale, q_offset=q_offset, return_mass=True)
    for a, b in zip((dq, dkv, mass), again):  # a fixed summation order
        assert torch.equal(a, b)
    # the one-token kernels on the same inputs
    out1, smax1, ssum1 = _unpacked(ops, qd, kvd, idd, scale, q_offset)
    assert torch.equal(smax, smax1)
    assert torch.allclose(ssum, ssum1, rtol=1e-5)
    assert rel_err(out, out1) <= 1e-2
    mass1 = _unpacked_mass(qd, kvd, idd, smax, ssum, scale, q_offset)
    assert torch.allclose(mass, mass1, rtol=1e-5, atol=1e-6)
    # the oracle
    ref, lse = O.sparse_mla_fwd(q, kv, idx, scale, q_offset=q_offset)
    assert rel_err(out, ref) <= TOL
    assert rel_err(mass, O.attn_mass(q, kv, idx, lse, scale, q_offset=q_offset)) <= TOL
    rdq, rdkv = O.sparse_mla_bwd(q, kv, idx, dout, scale, q_offset=q_offset)
    assert rel_err(dq, rdq) <= TOL and rel_err(dkv, rdkv) <= TOL


@pytest.mark.gpu
def test_packed_sink_and_chunks():
    """The sink's gradient over packed tokens, and chunks of groups under a small workspace."""
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    S, H, K, W = 700, 16, 64, 512
    g = torch.Generator().manual_seed(3)
    q, dout = (torch.randn(1, S, H, W, generator=g).bfloat16().cuda() for _ in range(2))
    kv, sink = torch.randn(1, S, W, generator=g).bfloat16().cuda(), torch.randn(H, generator=g).cuda()
    idx = rand_indices(S, K, seed=4, holes=0.3).cuda()
    scale = W ** -0.5
    out, m2, s2 = ops.sparse_mla_fwd(q, kv, idx, scale, sinks=sink)
    ref = O.sparse_attn_sink(q.cpu(), kv.cpu(), sink.cpu(), idx.cpu(), scale)
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert rel_err(out, ref) <= TOL
    full = ops.sparse_mla_bwd(q, kv, idx, out, dout, m2, s2, scale, sinks=sink)
    lib = _lib.load_library()
    most = int(lib.dsa_sparse_mla_bwd_workspace_size(1, S, S, H, W, K))
    for ws in (most, most // 3):
        assert lib.dsa_sparse_mla_bwd_packed(1, S, S, H, W, K, 0, ws) == 1
    part = ops.sparse_mla_bwd(q, kv, idx, out, dout, m2, s2, scale, sinks=sink, workspace_bytes=most // 3)
    one = ops.sparse_mla_bwd(q, kv, idx, out, dout, m2, s2, scale, sinks=sink, workspace_bytes=1 << 18)  # unpacked
    assert lib.dsa_sparse_mla_bwd_packed(1, S, S, H, W, K, 0, 1 << 18) == 0
    assert torch.equal(full[0], part[0])
    for a, b in zip(full[1:], part[1:]):
        assert rel_err(a, b) <= 1e-5
    for a, b in zip(full, one):
        assert rel_err(a, b) <= 1e-2


def test_packed_needs_room():
    """A workspace that holds only a few groups at a time runs one token per workgroup."""
    from torchtitan_npu_simulator_amd import _lib

    lib = _lib.load_library()
    packed, rows = lib.dsa_sparse_mla_bwd_packed, lib.dsa_sparse_mla_bwd_chunk_rows
    for S, H, K in [(4096, 16, 2048), (4096, 64, 2048), (2048, 64, 512), (700, 16, 64)]:
        most = int(lib.dsa_sparse_mla_bwd_workspace_size(1, S, S, H, 576, K))
        assert packed(1, S, S, H, 576, K, 0, most) == 1
        few = most * 100 // S  # (about a hundred tokens' share)
        assert packed(1, S, S, H, 576, K, 0, few) == 0 and rows(1, S, S, 576, K, few) >= 1


@pytest.mark.gpu
def test_packed_capped_workspace_results():
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    S, H, K = 600, 32, 64
    g = torch.Generator().manual_seed(9)
    q, dout = torch.randn(1, S, H, 576, generator=g).bfloat16().cuda(), torch.randn(1, S, H, 512, generator=g).bfloat16().cuda()
    kv = torch.randn(1, S, 576, generator=g).bfloat16().cuda()
    idx = rand_indices(S, K, seed=9).cuda()
    out, smax, ssum = ops.sparse_mla_fwd(q, kv, idx, 576 ** -0.5)
    most = int(_lib.load_library().dsa_sparse_mla_bwd_workspace_size(1, S, S, H, 576, K))
    runs = [ops.sparse_mla_bwd(q, kv, idx, out, dout, smax, ssum, 576 ** -0.5, workspace_bytes=b)
            for b in (most, most // 2, most // 8)]
    for r in runs[1:]:
        for a, b in zip(r, runs[0]):
            assert rel_err(a, b) <= 1e-2


def test_packed_where_lists_overlap():
    """With the causal test, lists that share few keys run one token per workgroup; without it
    (sequences of a batch, V4 windows) the number of keys says nothing."""
    from torchtitan_npu_simulator_amd import _lib

    lib = _lib.load_library()

    def tokens(mass, S, s_kv, H, K, off=None):
        return lib.dsa_attn_packed_tokens(mass, _lib.DSA_BF16, 1, S, s_kv, H, K, s_kv - S if off is None else off)

    def back(S, s_kv, H, K, off=None):
        return lib.dsa_sparse_mla_bwd_packed(1, S, s_kv, H, 576, K, s_kv - S if off is None else off, 32 << 30)

    assert tokens(0, 4096, 16384, 64, 1024) == 2 and tokens(0, 4096, 32768, 64, 1024) == 1
    assert tokens(0, 4096, 131072, 16, 1024) == 8 and tokens(0, 4096, 131072, 64, 1024, off=1 << 40) == 2
    assert back(4096, 16384, 64, 256) == 1 and back(4096, 32768, 64, 256) == 0 and back(1024, 32768, 64, 256) == 1
    assert back(4096, 65536, 16, 256) == 1 and back(4096, 131072, 16, 256) == 0
    assert back(4096, 65536, 64, 256, off=1 << 40) == 1
    assert tokens(1, 1024, 1024, 16, 256) == 1 and tokens(1, 1024, 1024, 16, 512) == 4
    assert tokens(1, 4096, 4096, 16, 64) == 8 and tokens(1, 4096, 32768, 64, 1024) == 1
    # a workspace serves the call with and without the causal test
    for S, s_kv, H, K in [(4096, 32768, 64, 256), (4096, 4096, 16, 512)]:
        most = int(lib.dsa_sparse_mla_bwd_workspace_size(1, S, s_kv, H, 576, K))
        assert lib.dsa_sparse_mla_bwd_packed(1, S, s_kv, H, 576, K, s_kv, most) == 1
        assert lib.dsa_sparse_mla_bwd_chunk_rows(1, S, s_kv, 576, K, most) >= 1
