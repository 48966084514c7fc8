"""fp32 attention on the matrix units (csrc/attn_f32.hip) at the edges of its tiles: widths,
heads, blocks of keys, rows without keys, the sink; against the fp64 oracle.

Tolerance: every result is a chain of fp32 sums of at most 576 (columns) or K (keys) products,
whose relative error in the 2-norm stays near sqrt(n) 2^-24 < 2e-6; 1e-5 leaves room for exp."""

from __future__ import annotations

import pytest
import torch

from oracle import dsa_oracle as O
from tests.dsa_cases import rand_indices, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("S,H,K,d_qk,d_v,q_offset", [
    (40, 16, 64, 576, 512, 0),
    (33, 20, 33, 576, 512, 7),   # a tail of heads and of keys
    # the smallest (K = 1 has dS = P (dP - delta) = 0 exactly, so dq has no relative error: with
    # three keys the rows that hold one add rounding of 2^-24 of the others' dq)
    (5, 1, 3, 16, 16, 0),
    (70, 4, 100, 80, 48, 0),     # widths that leave waves without a tile
    (9, 3, 2048, 512, 512, 2500),
])
def test_f32_attention(S, H, K, d_qk, d_v, q_offset):
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    s_kv = S + q_offset
    g = torch.Generator().manual_seed(S + K)
    q, kv = torch.randn(2, S, H, d_qk, generator=g), torch.randn(2, s_kv, d_qk, generator=g)
    dout = torch.randn(2, S, H, d_v, generator=g)
    idx = torch.cat([rand_indices(S, K, q_offset=q_offset, seed=b, shuffle=True, holes=0.2) for b in range(2)])
    idx[0, S // 2] = -1  # a row without keys
    if K > 64:
        idx[1, :, 32:64] = -1  # a block without keys
    scale = d_qk ** -0.5
    qd, kvd, idd, dod = q.cuda(), kv.cuda(), idx.cuda(), dout.cuda()
    out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, scale, d_v=d_v, q_offset=q_offset)
    dq, dkv = ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, scale, q_offset=q_offset)
    ref, lse = O.sparse_mla_fwd(q, kv, idx, scale, d_v=d_v, q_offset=q_offset)
    rdq, rdkv = O.sparse_mla_bwd(q, kv, idx, dout, scale, d_v=d_v, q_offset=q_offset)
    for name, a, b in (("out", out, ref), ("dq", dq, rdq), ("dkv", dkv, rdkv)):
        assert rel_err(a, b) <= TOL, name
    got = (smax.double() + ssum.double().log()).cpu()
    live = torch.isfinite(lse)
    assert torch.equal(torch.isfinite(got), live)
    assert rel_err(got[live], lse[live]) <= TOL
    assert float(out[0, S // 2].abs().sum()) == 0.0 and float(dq[0, S // 2].abs().sum()) == 0.0


def test_f32_attention_unselected_rows_not_finite():
    """Rows that no slot selects do not reach the results, whatever they hold."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    S, H, K, D = 20, 5, 40, 64
    g = torch.Generator().manual_seed(2)
    q, kv, dout = torch.randn(1, S, H, D, generator=g), torch.randn(1, S, D, generator=g), torch.randn(1, S, H, D, generator=g)
    idx = rand_indices(S, K, seed=3)
    idx[idx == 0] = -1
    runs = []
    for bad in (0.0, float("inf"), float("nan")):
        kv[0, 0] = bad
        qd, kvd, idd, dod = q.cuda(), kv.cuda(), idx.cuda(), dout.cuda()
        out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, D ** -0.5, d_v=D)
        runs.append((out, smax, *ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, D ** -0.5)))
    for r in runs[1:]:
        assert torch.equal(r[0], runs[0][0]) and torch.equal(r[1], runs[0][1]) and torch.equal(r[2], runs[0][2])
        assert rel_err(r[3], runs[0][3]) <= 1e-6  # (atomic sums)


def test_f32_attention_sink():
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    S, H, K, D = 50, 18, 48, 64
    g = torch.Generator().manual_seed(7)
    q, kv, dout = torch.randn(1, S, H, D, generator=g), torch.randn(1, S, D, generator=g), torch.randn(1, S, H, D, generator=g)
    sink = torch.randn(H, generator=g)
    idx = rand_indices(S, K, seed=5, holes=0.3)
    idx[0, 3] = -1
    qo, kvo, so = (t.double().requires_grad_(True) for t in (q, kv, sink))
    ref, lse = O.sparse_attn_sink(qo, kvo, so, idx, D ** -0.5)
    rdq, rdkv, rds = torch.autograd.grad(ref, (qo, kvo, so), dout.double())
    out, m2, s2 = ops.sparse_mla_fwd(q.cuda(), kv.cuda(), idx.cuda(), D ** -0.5, d_v=D, sinks=sink.cuda())
    dq, dkv, ds = ops.sparse_mla_bwd(q.cuda(), kv.cuda(), idx.cuda(), out, dout.cuda(), m2, s2, D ** -0.5, sinks=sink.cuda())
    for name, a, b in (("out", out, ref.detach()), ("lse", m2 + s2.log(), lse.detach()), ("dq", dq, rdq),
                       ("dkv", dkv, rdkv), ("dsink", ds, rds)):
        assert rel_err(a, b) <= TOL, name


@pytest.mark.parametrize("S,H,K,seed", [(512, 16, 64, 0), (300, 8, 128, 1), (700, 4, 256, 2)])
def test_f32_attention_gradient_error(S, H, K, seed):
    """dQ and dKV against fp64 on row widths of the model: the backward's S has the forward's bits,
    so its rounding cancels in P.  Measured 5.4e-7 to 6.7e-7 over nine draws; 8.4e-7 to 8.8e-7
    (dQ) with S summed in another order than the forward's."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    g = torch.Generator().manual_seed(seed)
    q, dout = torch.randn(1, S, H, 576, generator=g).cuda(), torch.randn(1, S, H, 512, generator=g).cuda()
    kv, idx = torch.randn(1, S, 576, generator=g).cuda(), rand_indices(S, K, seed=seed).cuda()
    scale = 576 ** -0.5
    out, smax, ssum = ops.sparse_mla_fwd(q, kv, idx, scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, idx, out, dout, smax, ssum, scale)
    qr, kr = q.double().requires_grad_(), kv.double().requires_grad_()
    rows = kr[0][idx[0].long().clamp_min(0)]  # [S, K, 576]
    x = torch.matmul(qr[0], rows.transpose(1, 2)) * scale
    p = torch.softmax(x.masked_fill((idx[0] < 0).unsqueeze(1), float("-inf")), dim=-1)
    rq, rk = torch.autograd.grad(torch.matmul(p, rows[..., :512]), [qr, kr], dout[0].double())
    assert rel_err(dq, rq) <= 7e-7 and rel_err(dkv, rk) <= 8e-7
