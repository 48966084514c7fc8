"""Few query tokens against many keys (generation): the forward splits a token's keys over
several workgroups and merges them, against the oracle and the one-workgroup kernel."""

from __future__ import annotations

import math

import pytest
import torch

from oracle import dsa_oracle as O
from tests.dsa_cases import rand_indices, rel_err

TOL = 2e-2  # bf16 attention


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,H,K,s_kv,width,sink", [
    (1, 1, 128, 2048, 3000, 576, False),  # the most splits
    (3, 1, 16, 300, 700, 576, False),     # a head tail, blocks that do not divide by the splits
    (2, 2, 100, 256, 512, 576, False),    # the fewest blocks that split
    (1, 5, 64, 1000, 1500, 512, True),    # the sink joins in the merge
])
def test_split_forward(B, S, H, K, s_kv, width, sink):
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    lib = _lib.load_library()
    off = s_kv - S
    assert lib.dsa_sparse_mla_fwd_workspace_size(_lib.DSA_BF16, B, S, s_kv, H, K, off) > 0
    g = torch.Generator().manual_seed(K)
    q = torch.randn(B, S, H, width, generator=g).bfloat16()
    kv = torch.randn(B, s_kv, width, generator=g).bfloat16()
    idx = torch.cat([rand_indices(S, K, q_offset=off, seed=b, shuffle=True, holes=0.1) for b in range(B)])
    idx[0, 0, : K // 2] = -1  # splits without a key
    if B > 1:
        idx[1] = -1  # rows without a key
    scale = 1.0 / math.sqrt(width)
    sinks = torch.randn(H, generator=g).cuda() if sink else None
    qd, kvd, idd = q.cuda(), kv.cuda(), idx.cuda()
    out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, scale, q_offset=off, sinks=sinks)
    # the same call without a workspace
    o1, m1, s1 = torch.empty_like(out), torch.empty_like(smax), torch.empty_like(ssum)
    _lib.check(lib.dsa_sparse_mla_fwd_ws(
        _lib.ptr(qd), _lib.ptr(kvd), _lib.ptr(idd), _lib.ptr(sinks), _lib.ptr(o1), _lib.ptr(m1), _lib.ptr(s1),
        _lib.DSA_BF16, B, S, s_kv, H, width, 512, K, scale, off, None, 0, _lib.stream_of(qd.device)), "fwd")
    assert torch.equal(smax, m1)
    assert torch.allclose(ssum, s1, rtol=1e-5)
    assert rel_err(out, o1) <= 1e-2
    if sink:
        assert rel_err(out, O.sparse_attn_sink(q, kv, sinks.cpu(), idx, scale)[0]) <= TOL
    else:
        assert rel_err(out, O.sparse_mla_fwd(q, kv, idx, scale, q_offset=off)[0]) <= TOL


@pytest.mark.gpu
def test_split_forward_outgrown_headroom():
    """Logits that outgrow a split's reference by more than the headroom are redone exactly."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    S, H, K, s_kv = 1, 16, 512, 600
    q, kv = torch.zeros(1, S, H, 576), torch.zeros(1, s_kv, 576)
    q[..., 0] = 1.0
    kv[0, :, 0] = torch.linspace(0, 400.0, s_kv)  # every split ends far above its first block
    kv[0, :, 1:512] = torch.randn(s_kv, 511, generator=torch.Generator().manual_seed(1))
    idx = torch.arange(s_kv - K, s_kv, dtype=torch.int32).view(1, 1, K)
    q, kv = q.bfloat16(), kv.bfloat16()
    out, _, _ = ops.sparse_mla_fwd(q.cuda(), kv.cuda(), idx.cuda(), 1.0, q_offset=s_kv)
    assert rel_err(out, O.sparse_mla_fwd(q, kv, idx, 1.0, q_offset=s_kv)[0]) <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["query nan", "query inf", "query -inf", "key nan", "keys of the first half nan",
                                   "keys of the first half -inf", "last key inf"])
@pytest.mark.parametrize("sink", [False, True])
def test_split_forward_not_finite(where, sink):
    """Rows that are not finite come out of the merge as out of the one-workgroup kernel."""
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    H, K, s_kv, inf = 20, 512, 600, float("inf")
    g = torch.Generator().manual_seed(5)
    q = torch.randn(1, 2, H, 576, generator=g).bfloat16()
    kv = torch.randn(1, s_kv, 576, generator=g).bfloat16()
    idx = rand_indices(2, K, q_offset=s_kv - 2, seed=5)
    first = idx[0, 0, : K // 2].long()
    if where == "query nan":
        q[0, 0, 3, 7] = float("nan")
    elif where == "query inf":
        q[0, 0, 3, 7] = inf
    elif where == "query -inf":  # (every logit the same infinity)
        kv[..., 9] = 1.0
        q[0, 0, 3, 9], q[0, 0, 4, 9] = -inf, inf
    elif where == "key nan":
        kv[0, idx[0, 0, 300].long()] = float("nan")
    elif where == "keys of the first half nan":
        kv[0, first] = float("nan")
    elif where == "keys of the first half -inf":
        q[..., 9] = q[..., 9].abs() + 0.1
        kv[0, first, 9] = -inf
    else:
        kv[0, idx[0, 0, K - 1].long(), 9] = inf
    sinks = torch.randn(H, generator=g).cuda() if sink else None
    qd, kvd, idd = q.cuda(), kv.cuda(), idx.cuda()
    lib = _lib.load_library()
    assert lib.dsa_sparse_mla_fwd_workspace_size(_lib.DSA_BF16, 1, 2, s_kv, H, K, s_kv - 2) > 0
    got = ops.sparse_mla_fwd(qd, kvd, idd, 576 ** -0.5, q_offset=s_kv - 2, sinks=sinks)
    one = [torch.empty_like(t) for t in got]
    _lib.check(lib.dsa_sparse_mla_fwd_ws(
        _lib.ptr(qd), _lib.ptr(kvd), _lib.ptr(idd), _lib.ptr(sinks), *(_lib.ptr(t) for t in one), _lib.DSA_BF16, 1, 2,
        s_kv, H, 576, 512, K, 576 ** -0.5, s_kv - 2, None, 0, _lib.stream_of(qd.device)), "fwd")
    for a, b in zip(got, one):
        a, b = a.float(), b.float()
        ok = torch.isfinite(b)
        assert torch.equal(a[~ok].nan_to_num(2.0, 1.0, -1.0), b[~ok].nan_to_num(2.0, 1.0, -1.0))
        # (where O is a NaN the sum holds the NaN logits' weights, which depend on the reference)
        ok &= ~torch.isnan(one[0].float()).any(-1).reshape(ok.shape[:3] + (1,) * (ok.dim() - 3))
        assert torch.allclose(a[ok], b[ok], rtol=2e-2, atol=2e-2)
