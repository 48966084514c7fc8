"""The work that a user of this package has it do, as measurable cases.

Each case is one call (or one forward + backward) through the public entry points: the
DSA layer of the ``npu_dsa`` converter, the torch_npu-style ops that it is made of, the
DeepSeek-V4 shared-KV attention, and the producers around them.  ``listed`` are fixed
sizes; ``draw`` gives further cases from the ranges that the listed ones stand for.
"""

import math
import types

import torch

D_QK, D_V, ROPE = 576, 512, 64  # MLA absorb mode: 512 latent + 64 rope columns
H_I, D_I = 64, 128  # the DeepSeek lightning indexer: 64 heads x 128


def listed():
    return [
        # one DeepSeek-V3.2 layer of a training step at the benchmark's shape, through the
        # converter's forward: bf16 indexer + top-k, attention, their backward, indexer loss
        dict(name="layer_train_8192", kind="layer", S=8192, H=128, K=2048),
        # the attention op on one tensor-parallel rank of eight (128 / 8 heads)
        dict(name="attn_train_16_heads", kind="attn", B=1, S=4096, H=16, K=2048),
        # a packed batch of ragged sequences (lengths on the device), tensor parallel four
        dict(name="attn_train_packed", kind="packed", lens="1,777,1500,301,2411,1090", H=32, K=1024),
        # generation: one new token of each sequence against its cached keys
        dict(name="decode_4x16384", kind="decode", B=4, S=1, s_kv=16384, H=128, K=2048),
        # the tiny fp32 layer that parity checks and debugging runs use
        dict(name="attn_train_fp32", kind="attn32", S=512, H=16, K=64),
        # the lightning indexer + top-k alone, bf16, a whole sequence
        dict(name="indexer_bf16_8192", kind="indexer", B=1, S=8192, s_k=8192, fp8=False, K=2048),
        # fp8: quantise the rows, then index a context-parallel share of the queries over
        # the whole key prefix
        dict(name="indexer_fp8_share", kind="indexer", B=1, S=2048, s_k=16384, fp8=True, K=2048),
        # the indexer KL loss op called on its own (evaluation of the indexer)
        dict(name="indexer_kl_4096", kind="kl", S=4096, H=128, K=2048),
        # the V4 block compressor over a long sequence, with norm and RoPE
        dict(name="compressor_32768", kind="compress", S=32768, D=512, ratio=4),
        # the indexer's query producer: RoPE + Hadamard + fp8
        dict(name="indexer_prep_8192", kind="prep", S=8192, heads=64, v4=False),
        # the absorbed MLA projections around the attention, forward + backward
        dict(name="absorb_train_4096", kind="absorb", S=4096, H=128),
        # one DeepSeek-V4 attention layer: window 128 + top-1024 compressed rows + sink
        dict(name="v4_train_4096", kind="v4", S=4096, H=128, K=1024, ratio=4),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer", "attn", "attn", "packed", "decode", "attn32", "indexer", "indexer", "kl", "compress",
                       "prep", "absorb", "v4"])
    heads = rng.choice([8, 16, 32, 64, 128])
    topk = rng.choice([64, 256, 512, 1000, 1024, 2048])
    if kind == "layer":
        return dict(kind=kind, S=_log_int(rng, 100, 4096), H=heads, K=topk)
    if kind == "attn":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), S=_log_int(rng, 50, 3000), H=heads, K=topk)
    if kind == "packed":
        lens = [_log_int(rng, 1, 2000) for _ in range(rng.randint(1, 6))]
        return dict(kind=kind, lens=",".join(map(str, lens)), H=heads, K=topk)
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 1, 16), S=rng.choice([1, 1, 1, 2, 4]), s_kv=_log_int(rng, 300, 32768),
                    H=heads, K=topk)
    if kind == "attn32":
        return dict(kind=kind, S=_log_int(rng, 32, 768), H=rng.choice([4, 8, 16]), K=rng.choice([16, 50, 64, 128, 256]))
    if kind == "indexer":
        s_k = _log_int(rng, 256, 16384)
        return dict(kind=kind, B=rng.choice([1, 1, 2]), S=_log_int(rng, 16, min(s_k, 8192)), s_k=s_k,
                    fp8=rng.random() < 0.5, K=topk)
    if kind == "kl":
        return dict(kind=kind, S=_log_int(rng, 64, 3000), H=heads, K=topk)
    if kind == "compress":
        ratio = rng.choice([4, 4, 128])
        return dict(kind=kind, S=ratio * _log_int(rng, max(1, 64 // ratio), 32768 // ratio), D=rng.choice([128, 512]),
                    ratio=ratio)
    if kind == "prep":
        return dict(kind=kind, S=_log_int(rng, 64, 8192), heads=rng.choice([1, 64]), v4=rng.random() < 0.5)
    if kind == "absorb":
        return dict(kind=kind, S=_log_int(rng, 64, 4096), H=heads)
    ratio = rng.choice([4, 4, 128])
    return dict(kind=kind, S=128 * _log_int(rng, 2, 24), H=heads, K=rng.choice([128, 512, 1024]), ratio=ratio)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Draws:
    """Seeded inputs drawn on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=self.g, device=self.dev, dtype=torch.float32).to(dtype)

    def head_weights(self, *shape):
        return torch.rand(*shape, generator=self.g, device=self.dev) * (shape[-1] ** -0.5 * D_I ** -0.5)

    def rows_of(self, S, s_kv, K):
        """int32 [S,K]: each query row's random distinct keys among those it may see
        (t <= s + s_kv - S), ascending, -1 after the last, as the top-k returns them."""
        out = torch.empty(S, K, dtype=torch.int32, device=self.dev)
        t = torch.arange(s_kv, device=self.dev)
        k = min(K, s_kv)
        for r0 in range(0, S, 1024):
            s = torch.arange(r0, min(S, r0 + 1024), device=self.dev).view(-1, 1)
            x = torch.rand(s.numel(), s_kv, generator=self.g, device=self.dev)
            x = x.masked_fill(t > s + (s_kv - S), -1.0)
            v, i = x.topk(k, dim=1)
            i = i.masked_fill(v < 0, s_kv).sort(dim=1).values
            out[r0:r0 + s.numel(), :k] = i.masked_fill(i == s_kv, -1).to(torch.int32)
        out[:, k:] = -1
        return out

    def window_of(self, S, n_cmp, K):
        """int32 [1,S,K] compressed rows c < (s + 1) // 4 of each token, offset by S."""
        out = torch.empty(S, K, dtype=torch.int32, device=self.dev)
        t = torch.arange(n_cmp, device=self.dev)
        k = min(K, n_cmp)
        for r0 in range(0, S, 1024):
            s = torch.arange(r0, min(S, r0 + 1024), device=self.dev).view(-1, 1)
            x = torch.rand(s.numel(), n_cmp, generator=self.g, device=self.dev).masked_fill(t >= (s + 1) // 4, -1.0)
            v, i = x.topk(k, dim=1)
            i = i.masked_fill(v < 0, n_cmp).sort(dim=1).values
            out[r0:r0 + s.numel(), :k] = torch.where(i == n_cmp, i.new_full((), -1), i + S).to(torch.int32)
        out[:, k:] = -1
        return out.unsqueeze(0)

    def rope_table(self, n_pos, dim):
        inv = 10000.0 ** (-torch.arange(0, dim, 2, device=self.dev, dtype=torch.float64) / dim)
        ang = torch.arange(n_pos, device=self.dev, dtype=torch.float64).view(-1, 1) * inv
        return torch.polar(torch.ones_like(ang), ang).to(torch.complex64)


def _lens(case):
    return [int(v) for v in case["lens"].split(",")]


def _inputs(case, seed):
    d, kind = _Draws(seed), case["kind"]
    n = types.SimpleNamespace(case=case, kind=kind)
    if kind == "layer":
        S, H = case["S"], case["H"]
        n.q = d.normal(1, S, H, D_QK)
        n.kv = d.normal(1, S, 1, D_QK)
        n.qi, n.ki, n.w = d.normal(1, S, H_I, D_I), d.normal(1, S, 1, D_I), d.head_weights(1, S, H_I)
        n.dout = d.normal(1, S, H, D_V)
    elif kind in ("attn", "attn32"):
        dt = torch.float32 if kind == "attn32" else torch.bfloat16
        B, S, H = case.get("B", 1), case["S"], case["H"]
        n.q, n.kv, n.dout = d.normal(B, S, H, D_QK, dtype=dt), d.normal(B, S, 1, D_QK, dtype=dt), \
            d.normal(B, S, H, D_V, dtype=dt)
        n.idx = torch.stack([d.rows_of(S, S, case["K"]) for _ in range(B)]).unsqueeze(2)
    elif kind == "packed":
        lens = _lens(case)
        T, H = sum(lens), case["H"]
        n.q, n.kv, n.dout = d.normal(T, H, D_QK), d.normal(T, 1, D_QK), d.normal(T, H, D_V)
        n.idx = torch.cat([d.rows_of(m, m, case["K"]) for m in lens]).unsqueeze(1)
        n.cu = torch.tensor([0] + lens, device=d.dev).cumsum(0).to(torch.int32)
    elif kind == "decode":
        B, S, s_kv, H = case["B"], case["S"], case["s_kv"], case["H"]
        n.q, n.kv = d.normal(B, S, H, D_QK), d.normal(B, s_kv, 1, D_QK)
        n.qi, n.ki, n.w = d.normal(B, S, H_I, D_I), d.normal(B, s_kv, 1, D_I), d.head_weights(B, S, H_I)
    elif kind == "indexer":
        B, S, s_k = case["B"], case["S"], case["s_k"]
        n.qi, n.ki, n.w = d.normal(B, S, H_I, D_I), d.normal(B, s_k, 1, D_I), d.head_weights(B, S, H_I)
    elif kind == "kl":
        S, H = case["S"], case["H"]
        n.q, n.kv = d.normal(1, S, H, D_QK), d.normal(1, S, 1, D_QK)
        n.qi, n.ki, n.w = d.normal(1, S, H_I, D_I), d.normal(1, S, 1, D_I), d.head_weights(1, S, H_I)
        n.idx = d.rows_of(S, S, case["K"]).view(1, S, 1, case["K"])
        n.smax, n.ssum = _softmax_stats(n.q[0], n.kv[0, :, 0], n.idx[0, :, 0], D_QK ** -0.5)
    elif kind == "compress":
        S, D, r = case["S"], case["D"], case["ratio"]
        width = 2 * D if r == 4 else D
        n.kv, n.score = d.normal(1, S, width, dtype=torch.float32), d.normal(1, S, width, dtype=torch.float32)
        n.ape = 0.02 * d.normal(r, width, dtype=torch.float32)
        n.norm = 1.0 + 0.1 * d.normal(D, dtype=torch.float32)
        n.freqs = d.rope_table(S, 64)
    elif kind == "prep":
        S, h = case["S"], case["heads"]
        n.x = d.normal(1, S, h, D_I) if h > 1 else d.normal(1, S, D_I)
        n.freqs = d.rope_table(S, 64)
    elif kind == "absorb":
        S, H = case["S"], case["H"]
        n.q_nope, n.q_pe = d.normal(1, S, H, 128), d.normal(1, S, H, ROPE)
        n.w_uk = (d.normal(H, 128, D_V, dtype=torch.float32) * D_V ** -0.5).to(torch.bfloat16)
        n.w_uv = (d.normal(H, D_V, 128, dtype=torch.float32) * D_V ** -0.5).to(torch.bfloat16)
        n.attn = d.normal(1, S, H, D_V)
        n.dq, n.dy = d.normal(1, S, H, D_QK), d.normal(1, S, H, 128)
    elif kind == "v4":
        S, H, r = case["S"], case["H"], case["ratio"]
        n.q, n.kv, n.cmp = d.normal(1, S, H, D_V), d.normal(1, S, D_V), d.normal(1, S // r, D_V)
        n.sinks = d.normal(H, dtype=torch.float32)
        n.idx = d.window_of(S, S // r, case["K"]) if r == 4 else None
        n.dout = d.normal(1, S, H, D_V)
    return n


def prepare(case, seed):
    """Inputs on the GPU, in the layouts that the model code hands over."""
    n = _inputs(case, seed)
    if n.kind == "layer":
        from torchtitan_npu_simulator_amd.converters.dsa import SparseLightningIndexerKLLoss

        n.layer = types.SimpleNamespace(
            config=types.SimpleNamespace(kv_lora_rank=D_V, qk_rope_head_dim=ROPE),
            compute_dsa_indexer_loss=SparseLightningIndexerKLLoss(), layer_number=0, num_layers=1)
        n.dloss = torch.ones((), device=n.q.device)
    for t in ("q", "kv", "qi", "ki", "w", "q_nope", "q_pe", "w_uk", "w_uv", "attn", "cmp", "sinks"):
        if n.kind in ("layer", "attn", "attn32", "packed", "absorb", "v4") and hasattr(n, t):
            getattr(n, t).requires_grad_(True)
    return n


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(n):
    from torchtitan_npu_simulator_amd import torch_npu_ops as npu

    if n.kind == "layer":
        from torchtitan_npu_simulator_amd.converters.dsa import dsa_forward

        q, k = n.q.transpose(1, 2), n.kv.transpose(1, 2)
        loss, out = dsa_forward(n.layer, q, k, k[..., :D_V], scale=D_QK ** -0.5, q_indexer=n.qi, k_indexer=n.ki,
                                weights=n.w, index_topk=n.case["K"])
        return (out, *torch.autograd.grad([loss, out], [n.q, n.kv, n.qi, n.ki, n.w], [n.dloss, n.dout.transpose(1, 2)]))
    if n.kind in ("attn", "attn32", "packed"):
        q_nope, q_pe = torch.split(n.q, [D_V, ROPE], dim=-1)
        k_nope, k_pe = torch.split(n.kv, [D_V, ROPE], dim=-1)
        lay = dict(layout_query="TND", layout_kv="TND", cu_seqlens_q=n.cu, cu_seqlens_kv=n.cu) \
            if n.kind == "packed" else {}
        out, smax, ssum = npu.npu_sparse_flash_attention(q_nope, k_nope, k_nope, n.idx, query_rope=q_pe, key_rope=k_pe,
                                                         scale_value=D_QK ** -0.5, sparse_mode=3, **lay)
        return (out, smax, ssum, *torch.autograd.grad(out, [n.q, n.kv], n.dout))
    if n.kind == "decode":
        idx, _ = npu.npu_lightning_indexer(n.qi, n.ki, n.w, sparse_count=n.case["K"], sparse_mode=3)
        q_nope, q_pe = torch.split(n.q, [D_V, ROPE], dim=-1)
        k_nope, k_pe = torch.split(n.kv, [D_V, ROPE], dim=-1)
        out, _, _ = npu.npu_sparse_flash_attention(q_nope, k_nope, k_nope, idx, query_rope=q_pe, key_rope=k_pe,
                                                   scale_value=D_QK ** -0.5, sparse_mode=3)
        return idx, out
    if n.kind == "indexer":
        if n.case["fp8"]:
            q8, qs = npu.quantize_fp8_per_row(n.qi)
            k8, ks = npu.quantize_fp8_per_row(n.ki.squeeze(2))
            return npu.npu_lightning_indexer(q8, k8, n.w, sparse_count=n.case["K"], sparse_mode=3, return_value=True,
                                             query_scale=qs, key_scale=ks)
        return npu.npu_lightning_indexer(n.qi, n.ki, n.w, sparse_count=n.case["K"], sparse_mode=3, return_value=True)
    if n.kind == "kl":
        q_nope, q_pe = torch.split(n.q, [D_V, ROPE], dim=-1)
        k_nope, k_pe = torch.split(n.kv, [D_V, ROPE], dim=-1)
        return npu.npu_sparse_lightning_indexer_grad_kl_loss(
            q_nope, k_nope, n.qi, n.ki, n.w, n.idx, n.smax, n.ssum, scale_value=D_QK ** -0.5, query_rope=q_pe,
            key_rope=k_pe)
    if n.kind == "compress":
        return npu.compressor_pool(n.kv, n.score, n.ape, n.case["ratio"], norm_weight=n.norm, freqs_cis=n.freqs)
    if n.kind == "prep":
        start, inter = (64, True) if n.case["v4"] else (0, False)
        return npu.indexer_prep(n.x, n.freqs, rope_start=start, interleaved=inter)
    if n.kind == "absorb":
        q = npu.mla_absorb_q(n.q_nope, n.q_pe, n.w_uk)
        y = npu.mla_absorb_out(n.attn, n.w_uv)
        return (q, y, *torch.autograd.grad([q, y], [n.q_nope, n.q_pe, n.w_uk, n.attn, n.w_uv], [n.dq, n.dy]))
    out = npu.npu_sparse_attn_shared_kv(n.q, n.kv, n.cmp, n.idx, n.sinks, D_V ** -0.5, n.case["ratio"])
    return (out, *torch.autograd.grad(out, [n.q, n.kv, n.cmp, n.sinks], n.dout))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _pairs(S, s_kv, K):
    """Usable (row, slot) pairs: min(K, s + 1 + s_kv - S) summed over the rows."""
    a = s_kv - S + 1
    full = max(0, min(S, S - (K - a))) if K > a else S
    head = S - full
    return full * K + head * a + head * (head - 1) // 2


def _attn_work(rows, pairs, keys, H, K, width, es, train):
    q, o, kv = rows * H * width * es, rows * H * D_V * es, keys * width * es
    fwd = dict(bytes=q + o + kv + rows * K * 4 + rows * H * 8, flops=2 * pairs * H * (width + D_V))
    if not train:
        return fwd
    # S again, dP, dQ, dK, dV
    return dict(bytes=fwd["bytes"] + 2 * q + 2 * o + 2 * kv + rows * K * 4 + rows * H * 8,
                flops=fwd["flops"] + 2 * pairs * H * (3 * width + 2 * D_V))


def work(case):
    kind = case["kind"]
    if kind == "layer":
        S, K = case["S"], case["K"]
        a, i, k = (_attn_work(S, _pairs(S, S, K), S, case["H"], K, D_QK, 2, True), work(dict(case, kind="indexer", B=1, s_k=S,
                   fp8=False)), _kl_work(S, _pairs(S, S, K), K))
        return {m: a[m] + i[m] + k[m] for m in a}
    if kind in ("attn", "attn32"):
        B, S, K = case.get("B", 1), case["S"], case["K"]
        w = _attn_work(S, _pairs(S, S, K), S, case["H"], K, D_QK, 4 if kind == "attn32" else 2, True)
        return {m: B * w[m] for m in w}
    if kind == "packed":
        ws = [_attn_work(m, _pairs(m, m, case["K"]), m, case["H"], case["K"], D_QK, 2, True) for m in _lens(case)]
        return {m: sum(w[m] for w in ws) for m in ("bytes", "flops")}
    if kind == "decode":
        B, S, s_kv, K = case["B"], case["S"], case["s_kv"], case["K"]
        p = _pairs(S, s_kv, K)
        a = _attn_work(S, p, min(s_kv, p), case["H"], K, D_QK, 2, False)
        i = work(dict(kind="indexer", B=1, S=S, s_k=s_kv, fp8=False, K=K))
        return {m: B * (a[m] + i[m]) for m in a}
    if kind == "indexer":
        B, S, s_k = case["B"], case["S"], case["s_k"]
        return dict(bytes=B * (2 * (S * H_I + s_k) * D_I + 4 * S * H_I + 8 * S * case["K"]),
                    flops=B * 2 * _pairs(S, s_k, s_k) * H_I * D_I)
    if kind == "kl":
        S, H, K = case["S"], case["H"], case["K"]
        p = _pairs(S, S, K)
        k = _kl_work(S, p, K)
        return dict(bytes=k["bytes"] + 2 * S * (H + 1) * D_QK + 8 * S * H, flops=k["flops"] + 2 * p * H * D_QK)
    if kind == "compress":
        S, D, r = case["S"], case["D"], case["ratio"]
        width = 2 * D if r == 4 else D
        return dict(bytes=8 * S * width + 2 * (S // r) * D, flops=8 * S * width)
    if kind == "prep":
        rows = case["S"] * case["heads"]
        return dict(bytes=rows * D_I * 5 + rows * 4, flops=rows * D_I * 10)
    if kind == "absorb":
        S, H = case["S"], case["H"]
        return dict(bytes=2 * S * H * (2 * 128 + 2 * ROPE + 2 * D_V + 2 * 128 + D_V + D_QK) + 8 * H * 128 * D_V,
                    flops=6 * 2 * S * H * 128 * D_V)
    S, H, r = case["S"], case["H"], case["ratio"]
    p = _pairs(S, S, 128)
    p += sum(min(case["K"] if r == 4 else S, (s + 1) // r) for s in range(S))
    return _attn_work(S, p, S + S // r, H, case["K"] if r == 4 else 1, D_V, 2, True)


def _kl_work(S, pairs, K):
    return dict(bytes=2 * 2 * (S * H_I + S) * D_I + 8 * S * H_I + 4 * S * K, flops=2 * pairs * H_I * D_I * 3)


def tolerance(case):
    kind = case["kind"]
    if kind == "attn32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "compress":
        return {"rel": 5e-3, "max": 0.05}  # bf16 rows, normalised
    if kind == "prep":
        return {"rel": 1e-2, "max": 0.2}  # bf16, then 3-bit mantissas: a rounding is one step of 1/8
    if kind in ("indexer", "decode"):
        # scores that differ in their last fp32 bits swap a few keys at the cut
        return {"rel": 1e-2, "max": 0.3, "differ": 5e-3}
    if kind == "layer":
        return {"rel": 2e-2, "max": 0.9}
    return {"rel": 1e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _softmax_stats(q, kv, idx, scale):
    """(max, sum) [1,S,H] fp32 of each row's softmax over its selected keys."""
    S, H, _ = q.shape
    smax = torch.empty(1, S, H, device=q.device)
    ssum = torch.empty(1, S, H, device=q.device)
    step = max(1, (1 << 28) // (idx.shape[1] * D_QK))
    for r0 in range(0, S, step):
        i = idx[r0:r0 + step].long()
        x = torch.bmm(q[r0:r0 + step].float(), kv[i.clamp(min=0)].float().transpose(1, 2).contiguous()) * scale
        x = x.masked_fill((i < 0).unsqueeze(1), float("-inf"))
        m = x.amax(-1)
        smax[0, r0:r0 + step], ssum[0, r0:r0 + step] = m, torch.exp(x - m.unsqueeze(-1)).sum(-1)
    return smax, ssum


def _attn64(q, kv, idx, scale, dout=None, sinks=None, want_mass=False):
    """q [S,H,W], kv [T,W], idx [S,K] (-1 empty): out, max, sum and, with dout, dq, dkv and
    d sinks; the head-summed probability [S,K] with want_mass."""
    S, H, W = q.shape
    kv64 = kv.double()
    r = types.SimpleNamespace()
    new = lambda *s: torch.zeros(*s, dtype=torch.float64, device=q.device)  # noqa: E731
    r.out, r.smax, r.ssum, r.dq, r.dkv, r.dsinks = new(S, H, D_V), new(S, H), new(S, H), new(S, H, W), new(*kv.shape), new(H)
    r.mass = new(*idx.shape) if want_mass else None
    step = max(1, (1 << 28) // (idx.shape[1] * W))
    for r0 in range(0, S, step):
        sl = slice(r0, r0 + step)
        i = idx[sl].long()
        ok = i >= 0
        kk = kv64[i.clamp(min=0)]
        qd = q[sl].double()
        x = (torch.bmm(qd, kk.transpose(1, 2).contiguous()) * scale).masked_fill(~ok.unsqueeze(1), float("-inf"))
        m = x.amax(-1) if sinks is None else torch.maximum(x.amax(-1), sinks.double())
        m0 = m.masked_fill(m == float("-inf"), 0.0)
        e = torch.exp(x - m0.unsqueeze(-1))
        l = e.sum(-1) if sinks is None else e.sum(-1) + torch.exp(sinks.double() - m0)
        p = e / l.unsqueeze(-1).clamp_min(1e-300)
        out = torch.bmm(p, kk[..., :D_V].contiguous())
        r.out[sl], r.smax[sl], r.ssum[sl] = out, m, l
        if want_mass:
            r.mass[sl] = p.sum(1)
        if dout is None:
            continue
        do = dout[sl].double()
        delta = (do * out).sum(-1)
        if sinks is not None:
            r.dsinks -= (torch.exp(sinks.double() - m0) / l * delta).sum(0)
        ds = p * (torch.bmm(do, kk[..., :D_V].transpose(1, 2).contiguous()) - delta.unsqueeze(-1)) * scale
        r.dq[sl] = torch.bmm(ds, kk)
        c = torch.bmm(ds.transpose(1, 2).contiguous(), qd)
        c[..., :D_V] += torch.bmm(p.transpose(1, 2).contiguous(), do)
        r.dkv.index_add_(0, i[ok], c[ok])
    return r


def _scores64(qi, ki, w, k_rows, limit):
    """Index scores [rows, T] (-inf at masked keys): qi [R,64,128], ki [T,128], w [R,64]."""
    out = torch.empty(qi.shape[0], ki.shape[0], dtype=torch.float64, device=qi.device)
    kt = ki.double().t().contiguous()
    for r0 in range(0, qi.shape[0], 64):
        x = torch.relu(qi[r0:r0 + 64].double() @ kt)
        out[r0:r0 + 64] = torch.bmm(w[r0:r0 + 64].double().unsqueeze(1), x).squeeze(1)
    t = torch.arange(ki.shape[0], device=qi.device)
    return out.masked_fill(t > limit.view(-1, 1), float("-inf"))


def _topk64(sc, K):
    k = min(K, sc.shape[1])
    v, i = sc.topk(k, dim=1)
    i = i.masked_fill(v == float("-inf"), sc.shape[1]).sort(dim=1).values
    idx = torch.full((sc.shape[0], K), -1, dtype=torch.int64, device=sc.device)
    idx[:, :k] = i.masked_fill(i == sc.shape[1], -1)
    vals = torch.gather(sc, 1, idx.clamp(min=0)).masked_fill(idx < 0, float("-inf"))
    return idx, vals


def _indexer64(qi, ki, w, K):
    S, T = qi.shape[0], ki.shape[0]
    idx, vals = [], []
    for r0 in range(0, S, 1024):
        r1 = min(S, r0 + 1024)
        lim = torch.arange(r0, r1, device=qi.device) + (T - S)
        i, v = _topk64(_scores64(qi[r0:r1], ki, w[r0:r1], T, lim), K)
        idx.append(i)
        vals.append(v)
    return torch.cat(idx), torch.cat(vals)


def _kl64(qi, ki, w, idx, mass, upstream, eps=1e-8):
    """(dq, dk, dw, loss) of the indexer KL loss (token sum), gradients times upstream."""
    S = qi.shape[0]
    new = lambda *s: torch.zeros(*s, dtype=torch.float64, device=qi.device)  # noqa: E731
    dq, dk, dw, loss = new(*qi.shape), new(*ki.shape), new(*w.shape), 0.0
    step = max(1, (1 << 27) // (idx.shape[1] * H_I))
    for r0 in range(0, S, step):
        sl = slice(r0, r0 + step)
        i = idx[sl].long()
        ok = i >= 0
        kk, q, wd = ki[i.clamp(min=0)].double(), qi[sl].double(), w[sl].double()
        x = torch.bmm(q, kk.transpose(1, 2).contiguous())  # [c,64,K]
        sc = (torch.relu(x) * wd.unsqueeze(-1)).sum(1).masked_fill(~ok, float("-inf"))
        z = mass[sl].double().masked_fill(~ok, 0.0).clamp_min(0)
        zs = z.sum(-1, keepdim=True)
        t = z / zs.clamp_min(eps)
        ls = torch.log_softmax(sc, dim=-1)
        good = (zs > eps)
        lt = torch.where(t > 0, t * (t.clamp_min(eps).log() - ls.masked_fill(~ok, 0.0)), torch.zeros_like(t))
        loss += float((zs * lt.sum(-1, keepdim=True)).sum())
        g = torch.where(good & ok, zs * upstream * (torch.exp(ls) * t.sum(-1, keepdim=True) - t), torch.zeros_like(t))
        dw[sl] = (torch.relu(x) * g.unsqueeze(1)).sum(-1)
        e = g.unsqueeze(1) * wd.unsqueeze(-1) * (x > 0)
        dq[sl] = torch.bmm(e, kk)
        c = torch.bmm(e.transpose(1, 2).contiguous(), q)
        dk.index_add_(0, i[ok], c[ok])
    return dq, dk, dw, loss


def _rope64(x, ang):
    """x [.., 2n] in interleaved pairs, ang [.., n] complex128."""
    z = torch.view_as_complex(x.reshape(*x.shape[:-1], -1, 2).contiguous()) * ang
    return torch.view_as_real(z).reshape(x.shape)


def exact(case, seed):
    n, kind = _inputs(case, seed), case["kind"]
    scale = D_QK ** -0.5
    if kind == "layer":
        S = case["S"]
        idx, _ = _indexer64(n.qi[0], n.ki[0, :, 0], n.w[0], case["K"])
        a = _attn64(n.q[0], n.kv[0, :, 0], idx, scale, n.dout[0], want_mass=True)
        dqi, dki, dw, _ = _kl64(n.qi[0], n.ki[0, :, 0], n.w[0], idx, a.mass, 1.0 / S)
        return (a.out.unsqueeze(0).transpose(1, 2), a.dq.unsqueeze(0), a.dkv.view(n.kv.shape), dqi.unsqueeze(0),
                dki.view(n.ki.shape), dw.unsqueeze(0))
    if kind in ("attn", "attn32"):
        rs = [_attn64(n.q[b], n.kv[b, :, 0], n.idx[b, :, 0], scale, n.dout[b]) for b in range(n.q.shape[0])]
        out, smax, ssum, dq, dkv = (torch.stack([getattr(r, f) for r in rs]) for f in ("out", "smax", "ssum", "dq", "dkv"))
        return out, smax, ssum, dq, dkv.view(n.kv.shape)
    if kind == "packed":
        rs, t0 = [], 0
        for m in _lens(case):
            sl = slice(t0, t0 + m)
            rs.append(_attn64(n.q[sl], n.kv[sl, 0], n.idx[sl, 0], scale, n.dout[sl]))
            t0 += m
        out, smax, ssum, dq, dkv = (torch.cat([getattr(r, f) for r in rs]) for f in ("out", "smax", "ssum", "dq", "dkv"))
        return out, smax, ssum, dq, dkv.view(n.kv.shape)
    if kind == "decode":
        idx = [_indexer64(n.qi[b], n.ki[b, :, 0], n.w[b], case["K"])[0] for b in range(n.q.shape[0])]
        out = [_attn64(n.q[b], n.kv[b, :, 0], idx[b], scale).out for b in range(n.q.shape[0])]
        return torch.stack(idx).unsqueeze(2), torch.stack(out)
    if kind == "indexer":
        if case["fp8"]:
            return None  # the selection is a function of the 8-bit rows, not of the inputs
        r = [_indexer64(n.qi[b], n.ki[b, :, 0], n.w[b], case["K"]) for b in range(n.qi.shape[0])]
        return torch.stack([x[0] for x in r]).unsqueeze(2), torch.stack([x[1] for x in r]).unsqueeze(2)
    if kind == "kl":
        mass = _attn64(n.q[0], n.kv[0, :, 0], n.idx[0, :, 0], scale, want_mass=True).mass
        dqi, dki, dw, loss = _kl64(n.qi[0], n.ki[0, :, 0], n.w[0], n.idx[0, :, 0], mass, 1.0)
        return dqi.unsqueeze(0), dki.view(n.ki.shape), dw.unsqueeze(0), torch.tensor([loss], dtype=torch.float64)
    if kind == "compress":
        S, D, r = case["S"], case["D"], case["ratio"]
        kv, sc = (t[0].double().view(S // r, r, -1) for t in (n.kv, n.score))
        sc = sc + n.ape.double()
        if r == 4:
            prev = lambda t, fill: torch.cat([torch.full_like(t[:1, :, :D], fill), t[:-1, :, :D]])  # noqa: E731
            kv, sc = torch.cat([prev(kv, 0.0), kv[..., D:]], 1), torch.cat([prev(sc, float("-inf")), sc[..., D:]], 1)
        x = (kv * sc.softmax(1)).sum(1)
        x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * n.norm.double()
        x[:, D - 64:] = _rope64(x[:, D - 64:], n.freqs[::r].to(torch.complex128))
        return x.unsqueeze(0)
    if kind == "prep":
        x = n.x[0].double().clone()
        ang = n.freqs.to(torch.complex128)
        ang = ang.unsqueeze(1) if x.dim() == 3 else ang
        if case["v4"]:
            x[..., 64:] = _rope64(x[..., 64:], ang)
        else:  # blocked pairs (i, i + 32)
            y = _rope64(torch.stack([x[..., :32], x[..., 32:64]], -1).flatten(-2), ang).unflatten(-1, (32, 2))
            x[..., :32], x[..., 32:64] = y[..., 0], y[..., 1]
        h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
        while h.shape[0] < D_I:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)])
        y = (x @ h * D_I ** -0.5).unsqueeze(0)
        return y, None, y.abs().amax(-1) / 448.0
    if kind == "absorb":
        qn, at, dq, dy = (t[0].double().transpose(0, 1).contiguous() for t in (n.q_nope, n.attn, n.dq, n.dy))
        wk, wv = n.w_uk.double(), n.w_uv.double()
        tr = lambda t: t.transpose(1, 2).contiguous()  # noqa: E731
        back = lambda t: t.transpose(0, 1).unsqueeze(0)  # noqa: E731
        dql = dq[..., :D_V].contiguous()
        return (torch.cat([back(torch.bmm(qn, wk)), n.q_pe.double()], -1), back(torch.bmm(at, wv)),
                back(torch.bmm(dql, tr(wk))), n.dq[..., D_V:].double(), torch.bmm(tr(qn), dql),
                back(torch.bmm(dy, tr(wv))), torch.bmm(tr(at), dy))
    S, r = case["S"], case["ratio"]
    s = torch.arange(S, device=n.q.device).view(S, 1)
    win = s - 127 + torch.arange(128, device=n.q.device)
    if r == 4:
        cmp = n.idx[0].long()
    else:
        c = torch.arange(S // r, device=n.q.device)
        cmp = torch.where(c < (s + 1) // r, c + S, -1)
    rows = torch.cat([n.kv[0], n.cmp[0]])
    a = _attn64(n.q[0], rows, torch.cat([win.clamp(min=-1), cmp], 1), D_V ** -0.5, n.dout[0], n.sinks)
    return a.out.unsqueeze(0), a.dq.unsqueeze(0), a.dkv[:S].unsqueeze(0), a.dkv[S:].unsqueeze(0), a.dsinks
