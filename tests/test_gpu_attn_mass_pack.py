"""Attention mass with several tokens per workgroup, against the one-token kernel and fp64.

Both forms compute a row's scores by the same MFMA chain and differ in the order in which a
slot's H <= 64 probabilities, all positive, are added: at most 2 * 64 roundings, 2^-17
relative.  Against fp64 on the bf16 operands: the scores' fp32 sums of 576 products are within
2^-24 * sqrt(576) * |q||k| * scale < 1e-4 for these inputs, exp2 and the statistics add less:
1e-3 relative."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _case(B, S, s_kv, H, D, K, seed, repeats=False):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn(B, S, H, D, generator=g, device=DEV).bfloat16()
    kv = torch.randn(B, s_kv, D, generator=g, device=DEV).bfloat16()
    idx = torch.stack([torch.randperm(s_kv, generator=g, device=DEV)[torch.arange(K, device=DEV) % s_kv]
                       for _ in range(16)])[torch.randint(0, 16, (B, S), generator=g, device=DEV)].to(torch.int32)
    idx = torch.where(torch.rand(idx.shape, generator=g, device=DEV) < 0.1, -1, idx)
    if repeats:
        idx[:, ::3, K // 2:] = idx[:, ::3, :K - K // 2]
    return q, kv, idx.contiguous()


def _mass(q, kv, idx, mx, sm, scale, q_offset, ws_bytes):
    from torchtitan_npu_simulator_amd._lib import DSA_BF16, check, load_library, ptr, stream_of

    lib = load_library()
    B, S, H, D = q.shape
    K = idx.shape[-1]
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=DEV)
    out = torch.full((B, S, K), float("nan"), device=DEV)
    check(lib.dsa_attn_mass_ws(ptr(q), ptr(kv), ptr(idx), ptr(mx), ptr(sm), ptr(out), DSA_BF16, B, S, kv.shape[1], H,
                               D, K, scale, q_offset, ptr(ws), ws_bytes, stream_of(DEV)), "dsa_attn_mass_ws")
    return out


@pytest.mark.parametrize("B,S,s_kv,H,D,K,repeats", [
    (1, 700, 700, 64, 576, 96, False), (2, 513, 600, 16, 512, 64, True), (1, 1030, 500, 1, 576, 33, True),
    (1, 640, 640, 17, 576, 40, False), (2, 300, 310, 40, 512, 31, False), (1, 515, 40, 8, 576, 64, True)])
@pytest.mark.parametrize("causal", [True, False])
def test_packed_mass(B, S, s_kv, H, D, K, repeats, causal):
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops
    from torchtitan_npu_simulator_amd._lib import DSA_BF16, load_library

    q, kv, idx = _case(B, S, s_kv, H, D, K, S + H, repeats)
    scale, off = D ** -0.5, 0 if causal else s_kv
    need = int(load_library().dsa_attn_mass_workspace_size(DSA_BF16, B, S, s_kv, H, K, off))
    assert (need > 0) == (B * S >= (512 if causal else 1024))
    _, mx, sm = ops.sparse_mla_fwd(q, kv, idx, scale, q_offset=off)
    plain = _mass(q, kv, idx, mx, sm, scale, off, 0)
    got = _mass(q, kv, idx, mx, sm, scale, off, need)
    torch.testing.assert_close(got, plain, rtol=2.0 ** -17, atol=1e-30)
    assert torch.equal(ops.attn_mass(q, kv, idx, mx, sm, scale, q_offset=off), got)
    limit = torch.arange(S, device=DEV).view(1, S, 1) + off
    ok = (idx >= 0) & (idx <= limit)
    k = kv.double()[torch.arange(B, device=DEV).view(B, 1, 1), idx.clamp(min=0).long()]
    s = torch.matmul(q.double(), k.transpose(2, 3).contiguous()) * scale
    p = torch.exp(s.masked_fill(~ok.unsqueeze(2), -float("inf")) - (mx.double() + sm.double().log()).unsqueeze(-1))
    ref = torch.where(ok, p.sum(2), 0.0)
    assert torch.equal(got == 0, plain == 0)
    assert ((got.double() - ref).abs() <= 1e-3 * ref + 1e-7).all()


def test_packed_mass_in_chunks():
    """More groups than one chunk of the workspace holds."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops
    from torchtitan_npu_simulator_amd._lib import DSA_BF16, load_library

    q, kv, idx = _case(1, 8210, 4096, 16, 512, 2048, 5)
    need = int(load_library().dsa_attn_mass_workspace_size(DSA_BF16, 1, 8210, 4096, 16, 2048, 0))
    assert 8 * 16384 * 4 * ((8210 + 7) // 8) > 1 << 29 and need < 1 << 30
    _, mx, sm = ops.sparse_mla_fwd(q, kv, idx, 512 ** -0.5)
    plain = _mass(q, kv, idx, mx, sm, 512 ** -0.5, 0, 0)
    torch.testing.assert_close(_mass(q, kv, idx, mx, sm, 512 ** -0.5, 0, need), plain, rtol=2.0 ** -17, atol=1e-30)


@pytest.mark.parametrize("B,S,s_kv,H,D,K,repeats", [
    (1, 700, 700, 64, 576, 512, False),   # two tokens per group, a tail of one, slots past the last key
    (2, 513, 600, 16, 512, 512, True),    # five tokens, a tail of three, two batch elements, repeats
    (1, 1030, 500, 1, 576, 515, True),    # one head of 16 rows, an odd slot count
    (1, 640, 640, 17, 576, 600, False),   # heads padded to 32 rows
    (2, 300, 900, 40, 512, 513, False)])  # 48 rows per token: a wave's halves belong to two tokens
def test_packed_mass_long_lists(B, S, s_kv, H, D, K, repeats):
    """Sizes at which the causal call packs: against the one-token kernel, and in the backward."""
    from torchtitan_npu_simulator_amd import torch_npu_ops as ops
    from torchtitan_npu_simulator_amd._lib import DSA_BF16, load_library

    q, kv, idx = _case(B, S, s_kv, H, D, K, S + H, repeats)
    scale, off = D ** -0.5, s_kv - S if s_kv > S else 0
    lib = load_library()
    assert lib.dsa_attn_packed_tokens(1, DSA_BF16, B, S, s_kv, H, K, off) > 1
    need = int(lib.dsa_attn_mass_workspace_size(DSA_BF16, B, S, s_kv, H, K, off))
    out, mx, sm = ops.sparse_mla_fwd(q, kv, idx, scale, q_offset=off)
    plain = _mass(q, kv, idx, mx, sm, scale, off, 0)
    got = _mass(q, kv, idx, mx, sm, scale, off, need)
    torch.testing.assert_close(got, plain, rtol=2.0 ** -17, atol=1e-30)
    assert torch.equal(got == 0, plain == 0)
    assert torch.equal(ops.attn_mass(q, kv, idx, mx, sm, scale, q_offset=off), got)
    dout = torch.randn(out.shape, device=DEV).bfloat16()
    mass = ops.sparse_mla_bwd(q, kv, idx, out, dout, mx, sm, scale, q_offset=off, return_mass=True)[2]
    # (its scores come from 16 x 16 x 32 matrix steps: fp32 sums in another order)
    torch.testing.assert_close(mass, plain, rtol=1e-4, atol=1e-7)
