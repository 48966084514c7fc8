// Block KV compressor (DeepSeek-V4): softmax-gated pooling of ratio-token blocks.
//
// out[b, c, f] = sum_i softmax_i(g_i) x_i over the block's slots, where slot i of block c
//   without overlap: x = kv[b, c*r + i, f],        g = score[b, c*r + i, f] + ape[i, f]
//   with overlap (coff = 2), 2r slots: i < r  -> previous block's features 0..D
//                   x = kv[b, (c-1)*r + i, f],     g = score[...] + ape[i, f]   (absent for c = 0)
//                                       i >= r -> current block's features D..2D
//                   x = kv[b, c*r + i-r, D + f],   g = score[...] + ape[i-r, D + f]
// then optionally RMSNorm over f of the bf16-rounded pooled row times norm_weight, and
// optionally RoPE on the last rope_dim features (interleaved pairs (2i, 2i+1), angle i at
// the block's position, in fp32 on the row as stored: bf16-rounded when the output is
// bf16), as Compressor._forward_bsnd / _forward_tnd apply it after the norm.  The block's
// position is that of its first token: c * ratio, or positions[first token] when token
// positions are given (rows whose position falls outside the cos/sin table keep their
// features).
//
// Packed varlen ("TND") batches give each block's first token explicitly (block_starts,
// whole r-token blocks inside one request): block c pools tokens block_starts[c] + i, and
// with overlap its first r slots come from the previous listed block, block_starts[c-1],
// when c > 0 and the block's position (positions[block_starts[c]]) is at least r.
//
// HBM-bound streaming: a lane owns four consecutive features (16-byte loads, coalesced along
// the row) and D/4 lanes a row.  Each input row is read once per block that uses it (the
// overlap re-read of the previous block's first half comes from L2).  The softmax is online
// per feature in fp32 with expf, four slots at a time: their loads go out together and the
// running maximum moves once for the four (five expf instead of eight).
//
// What bounds it is the number of rows in flight.  With ratio 4 there are enough blocks, and
// a lane goes over its block's slots alone.  With ratio 128 one lane per feature was a serial
// chain of 128 slots on nb * D / 4 lanes, so `parts` lanes share a feature's slots (their
// softmax states meet by shuffles inside a wave and in LDS between waves).
// Measured, before and now: S=32768 D=512 ratio 128 94 -> 31 us, S=4096 75 -> 17.5, S=512
// 51 -> 15.6 and with D=128 50 -> 10.3; ratio 4 S=32768 D=512 (280 MB) 56.1 -> 53.9, of which
// batches of four instead of one slot give 4 us (two: 54.6; registers held to 8 waves a SIMD
// for them: spills, 65).  Rows sliced over workgroups as well, with the norm in a second
// launch, took 2 us off 4 to 32 blocks' kernels and put the same into the launch.
#include "dsa_common.h"

namespace dsa {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxThreads = 1024;
constexpr int kBatch = 4;

struct Args {
  const float *kv, *score, *ape, *norm_w;
  void* out;
  int out_bf16;
  int64_t n_blocks_total;
  int nb, D, r, overlap;
  float eps;
  const int64_t* block_starts;
  const int32_t* positions;
  int64_t n_tokens;
  const float* rope_cs;
  int64_t n_pos;
  int rope_dim;
};

struct Block {
  int64_t cur, prev;  // first token of the block and of the block whose first half overlaps it
  bool usable, has_prev;
  int c;
};

__device__ Block locate(const Args& a, int64_t blk) {
  const int64_t b = blk / a.nb;
  Block k{0, 0, true, false, (int)(blk - b * a.nb)};
  if (a.block_starts) {
    k.cur = a.block_starts[k.c];
    k.usable = k.cur >= 0 && k.cur <= a.n_tokens - a.r;  // out-of-range starts pool nothing
    if (k.usable && a.overlap && k.c > 0 && a.positions[k.cur] >= a.r) {
      k.prev = a.block_starts[k.c - 1];
      k.has_prev = k.prev >= 0 && k.prev <= a.n_tokens - a.r;
    }
  } else {
    k.cur = b * (int64_t)a.nb * a.r + (int64_t)k.c * a.r;
    k.prev = k.cur - a.r;
    k.has_prev = a.overlap && k.c > 0;
  }
  return k;
}

// Softmax state of one feature: a maximum of -inf holds nothing yet, and is shifted by 0 so
// that slots of -inf weigh 0 whichever slots they share a batch or a part with.
struct Pool {
  float m = -INFINITY, s = 0.f, acc = 0.f;
  __device__ void join(float m2, float s2, float acc2) {
    const float mn = fmaxf(m, m2);
    const float sh = mn == -INFINITY ? 0.f : mn;
    const float e1 = expf(m - sh), e2 = expf(m2 - sh);
    s = s * e1 + s2 * e2;
    acc = acc * e1 + acc2 * e2;
    m = mn;
  }
};

template <int N>
__device__ __forceinline__ void consume(Pool (&p)[4], const float* x, const float* g, const float* a, int64_t pitch) {
  float4 xr[N], gr[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    xr[i] = *reinterpret_cast<const float4*>(x + i * pitch);
    gr[i] = *reinterpret_cast<const float4*>(g + i * pitch);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float4 av = *reinterpret_cast<const float4*>(a + i * pitch);
    gr[i].x += av.x;
    gr[i].y += av.y;
    gr[i].z += av.z;
    gr[i].w += av.w;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float mn = p[u].m;
#pragma unroll
    for (int i = 0; i < N; ++i) mn = fmaxf(mn, (&gr[i].x)[u]);
    const float sh = mn == -INFINITY ? 0.f : mn;
    const float sc = expf(p[u].m - sh);
    p[u].s *= sc;
    p[u].acc *= sc;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float e = expf((&gr[i].x)[u] - sh);
      p[u].s += e;
      p[u].acc += e * (&xr[i].x)[u];
    }
    p[u].m = mn;
  }
}

// Rows [i0, i1) of the r tokens from `tok`; `off` is the lane's feature within the input row.
__device__ __forceinline__ void consume_rows(Pool (&p)[4], const Args& a, int64_t tok, int off, int i0, int i1) {
  const int64_t pitch = (int64_t)(a.overlap ? 2 : 1) * a.D;
  int i = i0;
  for (; i + kBatch <= i1; i += kBatch)
    consume<kBatch>(p, a.kv + (tok + i) * pitch + off, a.score + (tok + i) * pitch + off, a.ape + i * pitch + off,
                    pitch);
  for (; i < i1; ++i)
    consume<1>(p, a.kv + (tok + i) * pitch + off, a.score + (tok + i) * pitch + off, a.ape + i * pitch + off, pitch);
}

// RMSNorm of the bf16-rounded row (fp32 arithmetic) over its `lanes` lanes; `red` holds one
// float per wave of the row.  Every thread of the workgroup comes here; `writes` marks those
// whose values count.
__device__ void norm_row(float (&v)[4], const Args& a, int lanes, int l, float* red, bool writes) {
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    v[u] = bf16_to_f(f_to_bf16(v[u]));
    ss += v[u] * v[u];
  }
  if (lanes >= 64) {
    ss = wave_sum(ss);
    if (writes && (l & 63) == 0) red[l / 64] = ss;
    __syncthreads();
    ss = 0.f;
    for (int w = 0; w < lanes / 64; ++w) ss += red[w];
  } else {
    for (int mk = lanes >> 1; mk >= 1; mk >>= 1) ss += __shfl_xor(ss, mk, 64);
  }
  const float inv = rsqrtf(ss / (float)a.D + a.eps);
  const float4 w4 = *reinterpret_cast<const float4*>(a.norm_w + 4 * l);
  v[0] *= inv * w4.x;
  v[1] *= inv * w4.y;
  v[2] *= inv * w4.z;
  v[3] *= inv * w4.w;
}

__device__ __forceinline__ void rope_row(float (&v)[4], const Args& a, const Block& k, int f) {
  if (!a.rope_cs || !k.usable || f < a.D - a.rope_dim) return;
  // RoPE of the stored row: this lane's features are the pairs (f, f+1), (f+2, f+3)
  const int64_t pos = a.positions ? (int64_t)a.positions[k.cur] : (int64_t)k.c * a.r;
  if (pos < 0 || pos >= a.n_pos) return;
  if (a.out_bf16)
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = bf16_to_f(f_to_bf16(v[u]));
  const float4 cs4 = *reinterpret_cast<const float4*>(a.rope_cs + pos * a.rope_dim + (f - (a.D - a.rope_dim)));
  const float a0 = v[0], b0 = v[1], a1 = v[2], b1 = v[3];
  v[0] = a0 * cs4.x - b0 * cs4.y;
  v[1] = a0 * cs4.y + b0 * cs4.x;
  v[2] = a1 * cs4.z - b1 * cs4.w;
  v[3] = a1 * cs4.w + b1 * cs4.z;
}

__device__ __forceinline__ void store_row(const float (&v)[4], const Args& a, int64_t blk, int f) {
  const int64_t o = blk * (int64_t)a.D + f;
  if (a.out_bf16) {
    uint2 w;
    w.x = pack_bf16x2(v[0], v[1]);
    w.y = pack_bf16x2(v[2], v[3]);
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.out) + o) = w;
  } else {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.out) + o) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// A workgroup holds blockDim / (lanes * parts) blocks of lanes = D / 4 times `parts` threads;
// all three are powers of two, and a block of more than one wave in parts is alone in its
// workgroup.
template <bool kSplit>
__global__ void __launch_bounds__(kSplit ? kMaxThreads : kThreads)
compressor_kernel(Args a, int parts_arg) {
  extern __shared__ float smem[];
  const int lanes = a.D / 4, parts = kSplit ? parts_arg : 1;
  const int l = threadIdx.x & (lanes - 1);
  const int part = (threadIdx.x / lanes) & (parts - 1);
  const int g = threadIdx.x / (lanes * parts);
  const int64_t blk = (int64_t)blockIdx.x * (blockDim.x / (lanes * parts)) + g;
  const bool active = blk < a.n_blocks_total;
  const int f = 4 * l;
  const Block k = active ? locate(a, blk) : Block{0, 0, false, false, 0};

  Pool p[4];
  if (k.usable) {
    // the previous block's slots and this block's are divided over the parts alike
    const int per = (a.r + parts - 1) / parts;
    const int i0 = part * per, i1 = i0 + per < a.r ? i0 + per : a.r;
    if (k.has_prev) consume_rows(p, a, k.prev, f, i0, i1);
    consume_rows(p, a, k.cur, (a.overlap ? a.D : 0) + f, i0, i1);
  }
  if (kSplit) {
    const int in_wave = lanes * parts < 64 ? lanes * parts : 64;
    for (int d = lanes; d < in_wave; d <<= 1)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        p[u].join(__shfl_xor(p[u].m, d, 64), __shfl_xor(p[u].s, d, 64), __shfl_xor(p[u].acc, d, 64));
    if (lanes * parts > 64) {  // the block is the workgroup's only one
      const int span = lanes < 64 ? 64 : lanes;  // lanes that hold a state each
      const int n = lanes * parts / span, me = threadIdx.x / span, t = threadIdx.x & (span - 1);
      float4* box = reinterpret_cast<float4*>(smem);  // [n - 1][m, s, acc][span]
      if (me > 0) {
        box[((me - 1) * 3 + 0) * span + t] = make_float4(p[0].m, p[1].m, p[2].m, p[3].m);
        box[((me - 1) * 3 + 1) * span + t] = make_float4(p[0].s, p[1].s, p[2].s, p[3].s);
        box[((me - 1) * 3 + 2) * span + t] = make_float4(p[0].acc, p[1].acc, p[2].acc, p[3].acc);
      }
      __syncthreads();
      if (me == 0) {
        float top[4], sh[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) top[u] = p[u].m;
        for (int w = 0; w < n - 1; ++w) {
          const float4 m4 = box[(w * 3 + 0) * span + t];
#pragma unroll
          for (int u = 0; u < 4; ++u) top[u] = fmaxf(top[u], (&m4.x)[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          sh[u] = top[u] == -INFINITY ? 0.f : top[u];
          const float e = expf(p[u].m - sh[u]);
          p[u].s *= e;
          p[u].acc *= e;
        }
        for (int w = 0; w < n - 1; ++w) {
          const float4 m4 = box[(w * 3 + 0) * span + t], s4 = box[(w * 3 + 1) * span + t],
                       a4 = box[(w * 3 + 2) * span + t];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float e = expf((&m4.x)[u] - sh[u]);
            p[u].s += (&s4.x)[u] * e;
            p[u].acc += (&a4.x)[u] * e;
          }
        }
      }
      __syncthreads();  // smem is the norm's from here on
    }
  }
  float v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = p[u].s > 0.f ? p[u].acc / p[u].s : 0.f;
  if (a.norm_w) norm_row(v, a, lanes, l, smem + g * (lanes / 64 + 1), part == 0);
  rope_row(v, a, k, f);
  if (active && part == 0) store_row(v, a, blk, f);
}

// The split of a block: a part keeps at least one batch of slots.  With ratio 4 there is one
// part and 256 threads, with ratio 128 and D=512 eight parts and 1024.
int launch(const Args& a, const char* what, hipStream_t stream) {
  const int lanes = a.D / 4;
  int parts = 1;
  while (parts * 2 <= a.r / kBatch && lanes * parts * 2 <= kMaxThreads) parts *= 2;
  const int span = lanes * parts, held = lanes < 64 ? 64 : lanes;
  // blocks share a workgroup only where each has one part or sits inside one wave
  const int threads = parts > 1 && span > 64 ? span : kThreads;
  const int64_t per_wg = threads / span;
  const int64_t grid = (a.n_blocks_total + per_wg - 1) / per_wg;
  if (grid > INT32_MAX) return set_error(DSA_ERR_INVALID_ARG, "%s: too many blocks", what);
  const size_t norm_shm = (size_t)per_wg * (lanes / 64 + 1) * sizeof(float);
  const TimedLaunch tl("compressor_kernel", stream);
  if (parts > 1) {
    const size_t join_shm = span > 64 ? (size_t)(span / held - 1) * 3 * held * sizeof(float4) : 0;
    compressor_kernel<true><<<(unsigned)grid, threads, norm_shm > join_shm ? norm_shm : join_shm, stream>>>(a, parts);
  } else {
    compressor_kernel<false><<<(unsigned)grid, threads, norm_shm, stream>>>(a, 1);
  }
  return check_launch(what);
}

}  // namespace
}  // namespace dsa

namespace dsa {
namespace {
int check_rope(const char* what, const float* rope_cs, int64_t n_pos, int64_t rope_dim, int64_t d) {
  if (!rope_cs) return DSA_OK;
  if (rope_dim <= 0 || rope_dim % 4 != 0 || rope_dim > d || n_pos <= 0)
    return set_error(DSA_ERR_INVALID_ARG, "%s: rope_dim=%lld with %lld positions (needs a multiple of 4 <= D)", what,
                     (long long)rope_dim, (long long)n_pos);
  return DSA_OK;
}
}  // namespace
}  // namespace dsa

extern "C" int dsa_compressor_fwd(const float* kv, const float* score, const float* ape, const float* norm_weight,
                                  void* out, int out_dtype, int64_t batch, int64_t s, int64_t d, int64_t ratio,
                                  int overlap, float norm_eps, const float* rope_cs, int64_t n_pos, int64_t rope_dim,
                                  const int32_t* positions, void* stream) {
  using namespace dsa;
  if (!kv || !score || !ape || !out) return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd: null pointer");
  if (int rc = check_rope("dsa_compressor_fwd", rope_cs, n_pos, rope_dim, d)) return rc;
  if (batch <= 0 || s <= 0 || d <= 0 || ratio <= 0)
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd: bad sizes");
  if (s % ratio != 0)
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd: seqlen (%lld) must be divisible by ratio (%lld)",
                     (long long)s, (long long)ratio);
  if (d < 4 || d > 4 * kThreads || (d & (d - 1)) != 0)  // row groups tile the workgroup exactly
    return set_error(DSA_ERR_UNSUPPORTED, "dsa_compressor_fwd: D=%lld (needs a power of two in [4, 1024])",
                     (long long)d);
  if (out_dtype != DSA_F32 && out_dtype != DSA_BF16)
    return set_error(DSA_ERR_UNSUPPORTED, "dsa_compressor_fwd: out dtype %d", out_dtype);
  const int64_t nb = s / ratio;
  if (nb > INT32_MAX || ratio > 65536) return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd: sizes out of range");
  return launch({kv, score, ape, norm_weight, out, out_dtype == DSA_BF16, batch * nb, (int)nb, (int)d, (int)ratio,
                 overlap ? 1 : 0, norm_eps, nullptr, positions, batch * s, rope_cs, n_pos, (int)rope_dim},
                "dsa_compressor_fwd", (hipStream_t)stream);
}

extern "C" int dsa_compressor_fwd_tnd(const float* kv, const float* score, const float* ape,
                                      const float* norm_weight, void* out, int out_dtype, int64_t n_tokens, int64_t d,
                                      int64_t ratio, int overlap, const int64_t* block_starts, int64_t n_blocks,
                                      const int32_t* positions, float norm_eps, const float* rope_cs, int64_t n_pos,
                                      int64_t rope_dim, void* stream) {
  using namespace dsa;
  if (!kv || !score || !ape || !out || (n_blocks > 0 && !block_starts))
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd_tnd: null pointer");
  if (int rc = check_rope("dsa_compressor_fwd_tnd", rope_cs, n_pos, rope_dim, d)) return rc;
  if (rope_cs && !positions)
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd_tnd: RoPE needs the token positions");
  if (overlap && !positions)
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd_tnd: overlap needs the token positions");
  if (n_tokens <= 0 || d <= 0 || ratio <= 0 || n_blocks < 0)
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd_tnd: bad sizes");
  if (d < 4 || d > 4 * kThreads || (d & (d - 1)) != 0)
    return set_error(DSA_ERR_UNSUPPORTED, "dsa_compressor_fwd_tnd: D=%lld (needs a power of two in [4, 1024])",
                     (long long)d);
  if (out_dtype != DSA_F32 && out_dtype != DSA_BF16)
    return set_error(DSA_ERR_UNSUPPORTED, "dsa_compressor_fwd_tnd: out dtype %d", out_dtype);
  if (n_blocks > INT32_MAX || ratio > 65536)
    return set_error(DSA_ERR_INVALID_ARG, "dsa_compressor_fwd_tnd: sizes out of range");
  if (n_blocks == 0) return DSA_OK;
  return launch({kv, score, ape, norm_weight, out, out_dtype == DSA_BF16, n_blocks, (int)n_blocks, (int)d, (int)ratio,
                 overlap ? 1 : 0, norm_eps, block_starts, positions, n_tokens, rope_cs, n_pos, (int)rope_dim},
                "dsa_compressor_fwd_tnd", (hipStream_t)stream);
}
