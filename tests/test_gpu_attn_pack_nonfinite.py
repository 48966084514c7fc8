"""Rows that are not finite in packed attention (csrc/attn_pack.h): they reach the tokens that
select them and no others, forward and backward, as in the one-token kernels."""

from __future__ import annotations

import math

import pytest
import torch

from tests.dsa_cases import rand_indices, rel_err

INF, NAN = float("inf"), float("nan")
TOL = 1e-2  # packed against one-token kernels: another reference maximum of the bf16 P


def _one_token(ops, q, kv, idx, dout, scale, sinks=None):
    """Forward and backward of the one-token kernels: no forward workspace, a backward
    workspace too small for the packed plan."""
    from torchtitan_npu_simulator_amd import _lib

    B, S, H, D = q.shape
    K = idx.shape[-1]
    out = torch.empty(B, S, H, 512, dtype=q.dtype, device=q.device)
    smax, ssum = (torch.empty(B, S, H, device=q.device) for _ in range(2))
    lib = _lib.load_library()
    _lib.check(lib.dsa_sparse_mla_fwd_ws(
        _lib.ptr(q), _lib.ptr(kv), _lib.ptr(idx), _lib.ptr(sinks), _lib.ptr(out), _lib.ptr(smax), _lib.ptr(ssum),
        _lib.DSA_BF16, B, S, kv.shape[1], H, D, 512, K, scale, 0, None, 0, _lib.stream_of(q.device)), "fwd")
    ws = 1 << 18
    assert lib.dsa_sparse_mla_bwd_packed(B, S, kv.shape[1], H, D, K, 0, ws) == 0
    return (out, smax, ssum, *ops.sparse_mla_bwd(q, kv, idx, out, dout, smax, ssum, scale, sinks=sinks,
                                                 workspace_bytes=ws))


def _close(a, b):
    a, b = a.float(), b.float()
    ok = torch.isfinite(b)
    assert torch.equal(a[~ok], b[~ok])  # (a row without a key has a maximum of -inf; no NaN)
    assert rel_err(a[ok], b[ok]) <= TOL


def _case(H, S, K, width, seed, sinks):
    g = torch.Generator().manual_seed(seed)
    q, dout = torch.randn(1, S, H, width, generator=g).bfloat16(), torch.randn(1, S, H, 512, generator=g).bfloat16()
    kv = torch.randn(1, S, width, generator=g).bfloat16()
    idx = rand_indices(S, K, seed=seed, shuffle=True, holes=0.1)
    return q, kv, dout, idx, torch.randn(H, generator=g) if sinks else None


@pytest.mark.gpu
@pytest.mark.parametrize("H,S,K,width,sinks", [
    (16, 640, 40, 576, False),   # three tokens per group
    (24, 530, 33, 512, True),    # heads padded to 32 rows, an odd slot count, 512 columns, a sink
    (40, 530, 40, 512, False),   # 48 rows per token: a wave's rows belong to two tokens
    (64, 600, 64, 576, False),   # two tokens per group, every row used
])
@pytest.mark.parametrize("where", ["key nan", "key inf", "key -inf last", "query nan", "query inf keyless", "dout nan",
                                   "dout inf", "repeats"])
def test_packed_rows_not_finite(H, S, K, width, sinks, where):
    from torchtitan_npu_simulator_amd import _lib
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    q, kv, dout, idx, sk = _case(H, S, K, width, H + len(where), sinks)
    hit = [401]  # the tokens whose results the rows may reach
    if where.startswith("key") or where == "repeats":  # one key, selected by a few scattered tokens alone
        key, hit = 300, [300, 401, 402, S - 1]
        idx[idx == key] = 7
        idx[0, hit, 3] = key
        kv[0, key, 5] = NAN
        if where == "repeats":  # (a key twice in one list takes slots of its own)
            idx[0, 401, 4] = key
        elif where == "key inf":
            kv[0, key] = INF
        elif where == "key -inf last":  # (a logit of -inf where the query's last column is positive)
            kv[0, key] = 1.0
            kv[0, key, width - 1] = -INF
    elif where == "query nan":
        q[0, 401, 3] = NAN
    elif where == "query inf keyless":
        q[0, 401, 3, 11] = INF
        idx[0, 401] = -1
    else:
        dout[0, 401, 2, 9] = NAN if where == "dout nan" else INF
    scale = 1.0 / math.sqrt(width)
    qd, kvd, idd, dod = q.cuda(), kv.cuda(), idx.cuda(), dout.cuda()
    skd = None if sk is None else sk.cuda()
    lib = _lib.load_library()
    assert lib.dsa_sparse_mla_fwd_workspace_size(_lib.DSA_BF16, 1, S, S, H, K, 0) > 0
    one = _one_token(ops, qd, kvd, idd, dod, scale, skd)
    out, smax, ssum = ops.sparse_mla_fwd(qd, kvd, idd, scale, sinks=skd)
    dq, dkv, *_ = ops.sparse_mla_bwd(qd, kvd, idd, out, dod, smax, ssum, scale, sinks=skd)
    rest = torch.ones(S, dtype=torch.bool)
    rest[hit] = False
    for a, b in zip((out, smax, ssum, dq), (*one[:3], one[3])):
        _close(a[0, rest], b[0, rest])
    keys = torch.ones(S, dtype=torch.bool)  # keys that none of those tokens selected
    for t in hit:
        keys[idx[0, t][idx[0, t] >= 0].long()] = False
    assert int(keys.sum()) > S // 2
    _close(dkv[0, keys], one[4][0, keys])
    if "keyless" not in where:  # the tokens themselves show it
        assert not torch.isfinite(dq[0, 401].float()).all()
        assert not torch.isfinite(dkv[0, ~keys]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("device_bounds", [False, True])
def test_packed_rows_not_finite_across_sequences(device_bounds):
    """A sequence of a packed batch is what it is without its neighbours, whatever they hold."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops

    H, K, lens = 16, 64, [350, 401, 349]
    T = sum(lens)
    g = torch.Generator().manual_seed(1)
    q, dout = torch.randn(T, H, 576, generator=g).bfloat16(), torch.randn(T, H, 512, generator=g).bfloat16()
    kv = torch.randn(T, 576, generator=g).bfloat16()
    idx = torch.cat([rand_indices(m, K, seed=i)[0] for i, m in enumerate(lens)]).cuda()
    cu = [0, 350, 751, 1100]
    bounds = torch.tensor(cu, dtype=torch.int32, device="cuda") if device_bounds else cu
    scale = 576 ** -0.5
    runs = []
    for bad in (False, True):
        if bad:  # keys, a query and a gradient of the middle sequence, at both of its ends
            kv[350], kv[750], q[750, 3], dout[351, 1] = NAN, INF, NAN, INF
        qd, kvd, dod = q.cuda(), kv.cuda(), dout.cuda()
        out, smax, ssum = ops.sparse_mla_fwd_varlen(qd, kvd, idx, scale, bounds, bounds)
        dq, dkv, mass = ops.sparse_mla_bwd_varlen(qd, kvd, idx, out, dod, smax, ssum, scale, bounds, bounds,
                                                  return_mass=True)
        mass1 = ops.attn_mass_varlen(qd, kvd, idx, smax, ssum, scale, bounds, bounds)
        runs.append((out, smax, ssum, dq, dkv, mass, mass1))
    for a, b in zip(*runs):
        for r0, r1 in ((0, 350), (751, 1100)):
            assert torch.isfinite(b[r0:r1].float()).all()
            assert rel_err(b[r0:r1], a[r0:r1]) <= TOL
    assert not torch.isfinite(runs[1][0][350:751].float()).all()
