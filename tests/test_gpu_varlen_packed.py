"""Packed batches (TND) of enough tokens and few enough heads that tokens share workgroups
(csrc/attn_pack.h): groups cross sequence borders, the batch runs on global key rows
(dsa_tnd_global_indices{,_varlen}) with host and with device bounds, against the per-sequence
oracle and the per-sequence one-token kernels."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O
from tests.dsa_cases import rel_err
from tests.test_gpu_varlen import _local_indices

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = 2e-2  # bf16 attention and its gradients
SCALE = 576 ** -0.5


def _cu(lens):
    return [0] + np.cumsum(lens).tolist()


def _rule(idx, lens_q, lens_k):
    """Each slot by the per-sequence rule (0 <= v < len_k, v <= s_local + max(0, len_k - len_q)),
    offset by the sequence's first key; everything else -1."""
    out, q0, k0 = torch.full_like(idx, -1), 0, 0
    for lq, lk in zip(lens_q, lens_k):
        v = idx[q0:q0 + lq]
        lim = torch.arange(lq).view(lq, 1) + max(0, lk - lq)
        out[q0:q0 + lq] = torch.where((v >= 0) & (v < lk) & (v <= lim), v + k0, -1)
        q0, k0 = q0 + lq, k0 + lk
    return out


@pytest.mark.parametrize("n_seq", [1, 64, 65, 130])  # (64 sequences per launch)
def test_global_indices_from_host_bounds(n_seq):
    from torchtitan_npu_simulator_amd import _lib

    g = torch.Generator().manual_seed(n_seq)
    lens_q, lens_k = (torch.randint(0, 40, (n_seq,), generator=g).tolist() for _ in range(2))
    lens_q[n_seq // 2], lens_k[-1] = 300, 700  # (one much longer than the others)
    if n_seq > 2:
        lens_q[1] = lens_q[n_seq - 2] = 0
        lens_k[0] = 0
    T, K = sum(lens_q), 70
    idx = torch.randint(-3, 45, (T, K), generator=g, dtype=torch.int32)
    src, out = idx.to(DEV), torch.full((T, K), -7, dtype=torch.int32, device=DEV)
    cq, ck = _cu(lens_q), _cu(lens_k)
    _lib.check(_lib.load_library().dsa_tnd_global_indices_varlen(
        _lib.ptr(src), _lib.ptr(out), _lib.host_i32(cq), _lib.host_i32(ck), n_seq, K, _lib.stream_of(DEV)), "global")
    assert torch.equal(out.cpu(), _rule(idx, lens_q, lens_k))


CASES = [
    # lens_q, lens_k, H, K: borders inside groups, an empty sequence, a single token
    ([1, 500, 0, 530, 37], [1, 500, 0, 530, 37], 16, 64),
    ([300, 301, 450], [350, 301, 700], 64, 40),           # more keys than queries: a causal offset
    ([16] * 70, [16] * 70, 32, 16),                       # more than 64 sequences
]


@pytest.mark.parametrize("lens_q,lens_k,H,K", CASES)
@pytest.mark.parametrize("device_bounds", [False, True])
def test_packed_batch(lens_q, lens_k, H, K, device_bounds):
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    T, Tk = sum(lens_q), sum(lens_k)
    lib, far = _lib.load_library(), 1 << 40
    assert lib.dsa_attn_packed_tokens(0, _lib.DSA_BF16, 1, T, Tk, H, K, far) > 1
    assert lib.dsa_attn_packed_tokens(1, _lib.DSA_BF16, 1, T, Tk, H, K, far) > 1
    assert lib.dsa_sparse_mla_bwd_packed(1, T, Tk, H, 576, K, far,
                                         lib.dsa_sparse_mla_bwd_workspace_size(1, T, Tk, H, 576, K)) == 1
    g = torch.Generator().manual_seed(T + H)
    q, dout = torch.randn(T, H, 576, generator=g).bfloat16(), torch.randn(T, H, 512, generator=g).bfloat16()
    kv = torch.randn(Tk, 576, generator=g).bfloat16()
    idx = _local_indices(lens_q, lens_k, K, seed=H)
    qd, kvd, dod, idd = q.to(DEV), kv.to(DEV), dout.to(DEV), idx.to(DEV)
    cq, ck = _cu(lens_q), _cu(lens_k)
    bq, bk = (torch.tensor(c, dtype=torch.int32, device=DEV) for c in (cq, ck)) if device_bounds else (cq, ck)
    out, smax, ssum = ops.sparse_mla_fwd_varlen(qd, kvd, idd, SCALE, bq, bk)
    dq, dkv, mass = ops.sparse_mla_bwd_varlen(qd, kvd, idd, out, dod, smax, ssum, SCALE, bq, bk, return_mass=True)
    mass1 = ops.attn_mass_varlen(qd, kvd, idd, smax, ssum, SCALE, bq, bk)
    # the per-sequence entry point (one token per workgroup)
    o1, m1, s1 = torch.empty_like(out), torch.empty_like(smax), torch.empty_like(ssum)
    _lib.check(lib.dsa_sparse_mla_fwd_varlen(
        _lib.ptr(qd), _lib.ptr(kvd), _lib.ptr(idd), _lib.ptr(o1), _lib.ptr(m1), _lib.ptr(s1), _lib.DSA_BF16,
        _lib.host_i32(cq), _lib.host_i32(ck), len(lens_q), H, 576, 512, K, SCALE, _lib.stream_of(DEV)), "varlen")
    assert torch.equal(smax, m1) and torch.allclose(ssum, s1, rtol=1e-5)
    assert rel_err(out, o1) <= 1e-2
    # the oracle, sequence by sequence
    for i, (lq, lk) in enumerate(zip(lens_q, lens_k)):
        if lq == 0:
            continue
        a, b = slice(cq[i], cq[i] + lq), slice(ck[i], ck[i] + lk)
        off = max(0, lk - lq)
        args = (q[a].unsqueeze(0), kv[b].unsqueeze(0), idx[a].unsqueeze(0))
        ref, lse = O.sparse_mla_fwd(*args, SCALE, q_offset=off)
        rm = O.attn_mass(*args, lse, SCALE, q_offset=off)
        rdq, rdkv = O.sparse_mla_bwd(*args, dout[a].unsqueeze(0), SCALE, q_offset=off)
        if float(ref.abs().max()) == 0.0:  # (a sequence of holes)
            assert not out[a].any() and not mass[a].any()
            continue
        assert rel_err(out[a], ref[0]) <= TOL
        assert rel_err(mass[a], rm[0]) <= TOL and rel_err(mass1[a], rm[0]) <= TOL
        # (a token with a single key has dS = 0 but for rounding: judged against dO)
        small = TOL * float(dout[a].double().norm())
        for got, want in ((dq[a], rdq[0]), (dkv[b], rdkv[0])):
            err = float((got.double().cpu() - want.double()).norm())
            assert err <= TOL * float(want.double().norm()) or (lq < 20 and err <= small)


def test_packed_batch_differentiable():
    """The op on host and on device bounds gives the same results and gradients bit for bit."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    lens, H, K = [700, 1, 399], 32, 48
    T = sum(lens)
    g = torch.Generator().manual_seed(8)
    q = torch.randn(T, H, 576, generator=g).bfloat16().to(DEV).requires_grad_()
    kv = torch.randn(T, 1, 576, generator=g).bfloat16().to(DEV).requires_grad_()
    dout = torch.randn(T, H, 512, generator=g).bfloat16().to(DEV)
    idx = _local_indices(lens, lens, K, seed=1).to(DEV).unsqueeze(1)
    runs = []
    for cu in (_cu(lens), torch.tensor(_cu(lens), dtype=torch.int32, device=DEV)):
        out, smax, ssum = ops.npu_sparse_flash_attention(
            q[..., :512], kv[..., :512], kv[..., :512], idx, query_rope=q[..., 512:], key_rope=kv[..., 512:],
            scale_value=SCALE, layout_query="TND", layout_kv="TND", cu_seqlens_q=cu, cu_seqlens_kv=cu)
        runs.append((out, smax, ssum, *torch.autograd.grad(out, [q, kv], dout)))
    for a, b in zip(*runs):
        assert torch.equal(a, b)


def test_queries_without_keys_are_refused():
    """Host bounds: a sequence with queries and no keys is refused at any batch size."""
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    lens_q, lens_k, H, K = [600, 3, 600], [600, 0, 600], 16, 32
    T, Tk = sum(lens_q), sum(lens_k)
    q, kv = torch.zeros(T, H, 576, dtype=torch.bfloat16, device=DEV), torch.zeros(Tk, 576, dtype=torch.bfloat16, device=DEV)
    idx = torch.zeros(T, K, dtype=torch.int32, device=DEV)
    with pytest.raises(_lib.DSAError, match="no keys"):
        ops.sparse_mla_fwd_varlen(q, kv, idx, SCALE, _cu(lens_q), _cu(lens_k))
