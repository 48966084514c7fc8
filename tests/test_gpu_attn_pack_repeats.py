"""Packed attention (csrc/attn_pack.h) over lists that repeat keys, a few times or as padding:
every occurrence counts, in a fixed order, at a cost that stays near that of distinct lists."""

from __future__ import annotations

import pytest
import torch

from oracle import dsa_oracle as O
from tests.dsa_cases import rand_indices, rel_err

TOL = 2e-2  # bf16 attention and its gradients
SCALE = 576 ** -0.5


def _inputs(S, H, K, kind):
    g = torch.Generator().manual_seed(S + K)
    q, dout = torch.randn(1, S, H, 576, generator=g).bfloat16(), torch.randn(1, S, H, 512, generator=g).bfloat16()
    kv = torch.randn(1, S, 576, generator=g).bfloat16()
    if kind == "drawn with replacement":
        idx = (torch.rand(1, S, K, generator=g) * (torch.arange(S).view(1, S, 1) + 1)).to(torch.int32)
    else:
        idx = rand_indices(S, K, seed=K, shuffle=True)
        if kind == "padded with key 0":
            idx[..., K // 3:] = 0
        elif kind == "padded with the row's last key":
            idx[..., K // 2:] = torch.arange(S, dtype=torch.int32).view(1, S, 1)
        elif kind == "one key":
            idx[:] = 0
        elif kind == "one repeat":
            idx[0, 400, 1] = idx[0, 400, 0] = 17
    return q, kv, dout, idx


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["drawn with replacement", "padded with key 0", "padded with the row's last key",
                                  "one key", "one repeat"])
@pytest.mark.parametrize("S,H,K", [(517, 16, 33), (530, 40, 64)])
def test_packed_repeats(S, H, K, kind):
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    q, kv, dout, idx = _inputs(S, H, K, kind)
    qd, kvd, dod, idd = q.cuda(), kv.cuda(), dout.cuda(), idx.cuda()
    assert _lib.load_library().dsa_sparse_mla_fwd_workspace_size(_lib.DSA_BF16, 1, S, S, H, K, 0) > 0
    runs = []
    for _ in range(2):
        out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, SCALE)
        runs.append((out, smax, ssum, *ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, SCALE, return_mass=True),
                     ops.attn_mass(qd, kvd, idd, smax, ssum, SCALE)))
    for a, b in zip(*runs):
        assert torch.equal(a, b)
    out, smax, ssum, dq, dkv, mass, mass1 = runs[0]
    ref, lse = O.sparse_mla_fwd(q, kv, idx, SCALE)
    assert rel_err(out, ref) <= TOL
    rm = O.attn_mass(q, kv, idx, lse, SCALE)
    assert rel_err(mass, rm) <= TOL and rel_err(mass1, rm) <= TOL
    rdq, rdkv = O.sparse_mla_bwd(q, kv, idx, dout, SCALE)
    # (one key over and over: dS is 0 but for the rounding of P and dP, so the error is taken
    # against the size of dO, whose rows the sums are made of)
    floor = 1e-2 * float(dout.double().norm()) if kind == "one key" else 0.0
    assert float((dq.double().cpu() - rdq.double()).norm()) <= TOL * float(rdq.double().norm()) + floor
    assert float((dkv.double().cpu() - rdkv.double()).norm()) <= TOL * float(rdkv.double().norm()) + floor


@pytest.mark.gpu
def test_packed_repeats_cost():
    """Lists padded with one key take a few times what distinct ones take (one workgroup sums
    that key's rows); a walk over every repeat took more than a hundred times as long."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    S, H, K = 1024, 16, 256
    ms = []
    for kind in ("distinct", "padded with key 0"):
        qd, kvd, dod, idd = (x.cuda() for x in _inputs(S, H, K, kind))
        out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, SCALE)
        best = float("inf")
        for _ in range(4):  # (the first one warms up)
            beg, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            beg.record()
            ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, SCALE)
            end.record()
            end.synchronize()
            best = min(best, beg.elapsed_time(end))
        ms.append(best)
    assert ms[1] <= 12 * ms[0], ms
