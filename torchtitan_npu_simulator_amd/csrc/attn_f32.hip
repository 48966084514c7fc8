// Gathered sparse attention in fp32 on v_mfma_f32_16x16x4_f32 (forward and backward), for row
// widths that are multiples of 16 up to 576; other widths run the scalar kernels of
// sparse_mla_fwd.hip / sparse_mla_bwd.hip.
//
// One workgroup = one token x 16 heads, 4 waves.  The token's selected rows are gathered in
// blocks of 32 into an LDS tile (the next block's rows are held in registers meanwhile), Q
// and dO of the 16 heads stay in LDS.  MFMA k-slots are assigned so that lane group g's four
// steps use four consecutive elements: one 16-byte LDS read per lane feeds four MFMAs, for the
// columns of S = K Q^T as for the keys of P V and dS K.  Bound by the gather's latency and the
// fp32 matrix rate (a 16x16x4 step is 32 cycles); the scalar kernels read every row once per
// head with one thread per key, and added every (head, key) gradient row with atomics of its
// own, where one here adds the sum over 16 heads.  512 tokens, 16 heads, top-64:
// forward 861 -> 39 us, backward 16058 -> 101 us.
#include "attn_f32.h"

namespace dsa {
namespace {

constexpr int kThreads = 256;
constexpr int kBN = 32;        // keys per block
constexpr int kHT = 16;        // heads per workgroup
constexpr int kMaxD = 576;
constexpr int kLd = kMaxD + 4; // LDS row stride in floats (= 4 mod 32: rows 4 apart are 16 banks apart)
constexpr int kPs = kBN + 4;   // row stride of the [head][key] score tiles
constexpr int kMaxTiles = kMaxD / 16 / 4;  // 16-column tiles per wave

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bool f32_slot_ok(int v, int s_kv, int64_t limit) {
  return v >= 0 && v < s_kv && (int64_t)v <= limit;
}

// The block's rows of one wave (8w .. 8w+7; lane l holds float4 columns l, l + 64, l + 128) in
// registers: loads of unusable slots and of columns past the row read valid places; the former
// are stored as zeros (a weight of 0 times a value that is not finite would not be 0), the
// latter not at all.
struct RowRegs {
  f32x4 v[kBN / 4][3];
};
__device__ __forceinline__ void load_rows(RowRegs& r, const float* __restrict__ kvb, int slot_key, int wave, int lane,
                                          int d) {
  const int nc = d >> 2;
#pragma unroll
  for (int i = 0; i < kBN / 4; ++i) {
    const int key = __shfl(slot_key, 8 * wave + i, 64);
    const f32x4* src = reinterpret_cast<const f32x4*>(kvb + (int64_t)key * d);
#pragma unroll
    for (int c = 0; c < 3; ++c) r.v[i][c] = src[min(lane + 64 * c, nc - 1)];
  }
}
__device__ __forceinline__ void store_rows(const RowRegs& r, float* tile, uint32_t vmask, int wave, int lane, int d) {
  const int nc = d >> 2;
#pragma unroll
  for (int i = 0; i < kBN / 4; ++i)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (lane + 64 * c < nc)
        *reinterpret_cast<f32x4*>(tile + (8 * wave + i) * kLd + 4 * (lane + 64 * c)) =
            (vmask >> (8 * wave + i) & 1u) ? r.v[i][c] : (f32x4){0.f, 0.f, 0.f, 0.f};
}
// rows of 16 heads -> LDS (zero rows for absent heads)
__device__ __forceinline__ void load_heads(float* dst, const float* __restrict__ src, int nh, int d, int tid) {
  const int nc = d >> 2;
  for (int i = tid; i < kHT * nc; i += kThreads) {
    const int r = i / nc, c = i - r * nc;
    const f32x4 v = *reinterpret_cast<const f32x4*>(src + (int64_t)min(r, nh - 1) * d + 4 * c);
    *reinterpret_cast<f32x4*>(dst + r * kLd + 4 * c) = r < nh ? v : (f32x4){0.f, 0.f, 0.f, 0.f};
  }
}
// acc[16 rows of a x 16 rows of b] += a b^T over columns [c0, c1) (multiples of 16)
__device__ __forceinline__ f32x4 dot_rows(const float* a, const float* b, int c0, int c1, int col, int g) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const float* pa = a + col * kLd + 4 * g;
  const float* pb = b + col * kLd + 4 * g;
#pragma unroll 4
  for (int c = c0; c < c1; c += 16) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(pa + c), y = *reinterpret_cast<const f32x4*>(pb + c);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mfma_f32(x[j], y[j], acc);
  }
  return acc;
}

// slots of the block: key (0 for an unusable one) in every lane < 32, and their validity bits
__device__ __forceinline__ uint32_t block_slots(const int32_t* __restrict__ ridx, int blk, int K, int s_kv,
                                                int64_t limit, int lane, int& key) {
  const int j = blk * kBN + (lane & (kBN - 1));
  const int v = ridx[min(j, K - 1)];
  const bool ok = j < K && f32_slot_ok(v, s_kv, limit);
  key = ok ? v : 0;
  return (uint32_t)__ballot(ok);  // (lanes 32..63 repeat the block)
}

__global__ void __launch_bounds__(kThreads, 1)
attn_f32_fwd_kernel(const float* __restrict__ q, const float* __restrict__ kv, const int32_t* __restrict__ idx,
                    float* __restrict__ out, float* __restrict__ smax, float* __restrict__ ssum, int S, int s_kv, int H,
                    int K, int dqk, int dv, float scale, int64_t q_offset, const float* __restrict__ sinks) {
  __shared__ __align__(16) float tile[kBN * kLd];
  __shared__ __align__(16) float qs[kHT * kLd];
  __shared__ __align__(16) float ps[2][kHT * kPs];  // partial scores of the two column halves; P in the first
  __shared__ float alpha[kHT];
  const int tok = blockIdx.x, h0 = blockIdx.y * kHT, b = blockIdx.z, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int64_t row_id = (int64_t)b * S + tok;
  const int32_t* ridx = idx + row_id * K;
  const int64_t limit = tok + q_offset;
  const float* kvb = kv + (int64_t)b * s_kv * dqk;
  const int nh = min(kHT, H - h0);
  const int nblk = (K + kBN - 1) / kBN;
  int key;
  uint32_t vm = block_slots(ridx, 0, K, s_kv, limit, lane, key);
  RowRegs rr;
  load_rows(rr, kvb, key, wave, lane, dqk);
  load_heads(qs, q + (row_id * H + h0) * dqk, nh, dqk, tid);
  // wave w: scores of key tile w & 1 over column half w >> 1; output columns of tiles w, w + 4, ..
  const int kt = wave & 1, half = wave >> 1, mid = (dqk / 16 / 2) * 16;
  const int nt = dv / 16;
  f32x4 o[kMaxTiles];  // heads 4g + r, column 16 (wave + 4 t) + col
#pragma unroll
  for (int t = 0; t < kMaxTiles; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // softmax: thread = (head tid / 16, keys 2 (tid % 16), + 1)
  const int sh = tid >> 4, sk = 2 * (tid & 15);
  float m = -INFINITY, l = 0.f;
  for (int blk = 0; blk < nblk; ++blk) {
    store_rows(rr, tile, vm, wave, lane, dqk);
    const uint32_t vmask = vm;
    __syncthreads();
    if (blk + 1 < nblk) {
      vm = block_slots(ridx, blk + 1, K, s_kv, limit, lane, key);
      load_rows(rr, kvb, key, wave, lane, dqk);
    }
    if (vmask == 0u) {  // (workgroup-uniform) no usable key
      __syncthreads();
      continue;
    }
    {
      const f32x4 s = dot_rows(tile + 16 * kt * kLd, qs, half ? mid : 0, half ? dqk : mid, col, g);
      *reinterpret_cast<f32x4*>(&ps[half][col * kPs + 16 * kt + 4 * g]) = s;  // keys 16 kt + 4g + r of head col
    }
    __syncthreads();
    {
      float x[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        x[e] = (vmask >> (sk + e) & 1u) ? (ps[0][sh * kPs + sk + e] + ps[1][sh * kPs + sk + e]) * scale : -INFINITY;
      float bm = fmaxf(x[0], x[1]);
      bm = fmaxf(bm, lane_xor<1>(bm));
      bm = fmaxf(bm, lane_xor<2>(bm));
      bm = fmaxf(bm, lane_xor<4>(bm));
      bm = fmaxf(bm, lane_xor<8>(bm));
      const float mn = fmaxf(m, bm);
      const float mr = mn == -INFINITY ? 0.f : mn;  // (every logit so far is -inf: exp gives 0)
      const float a = m == -INFINITY ? 0.f : expf(m - mn);
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        x[e] = expf(x[e] - mr);
        sum += x[e];
      }
      sum += lane_xor<1>(sum);
      sum += lane_xor<2>(sum);
      sum += lane_xor<4>(sum);
      sum += lane_xor<8>(sum);
      l = l * a + sum;
      m = mn;
      // (every thread reads only the two scores it overwrites)
      *reinterpret_cast<float2*>(&ps[0][sh * kPs + sk]) = make_float2(x[0], x[1]);
      if ((tid & 15) == 0) alpha[sh] = a;
    }
    __syncthreads();
    f32x4 p4[2];  // P of head col, keys 16 s + 4g .. +3
#pragma unroll
    for (int s = 0; s < 2; ++s) p4[s] = *reinterpret_cast<const f32x4*>(&ps[0][col * kPs + 16 * s + 4 * g]);
    float al[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) al[r] = alpha[4 * g + r];
#pragma unroll
    for (int t = 0; t < kMaxTiles; ++t) {
      const int ct = wave + 4 * t;
      if (ct < nt) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[t][r] *= al[r];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int j = 0; j < 4; ++j) o[t] = mfma_f32(p4[s][j], tile[(16 * s + 4 * g + j) * kLd + 16 * ct + col], o[t]);
      }
    }
    __syncthreads();  // the tile and the scores are rewritten
  }
  // row statistics, with the sink's logit (no value) joining the sum
  __shared__ float inv_s[kHT];
  if ((tid & 15) == 0) {
    float m_out = m, l_out = l, fold = 1.f;
    if (sinks && sh < nh) {
      const float s = sinks[h0 + sh];
      m_out = fmaxf(m, s);
      const float a = l > 0.f ? l * expf(m - m_out) : 0.f;
      l_out = a + expf(s - m_out);
      fold = a / l_out;
    }
    inv_s[sh] = l > 0.f ? fold / l : 0.f;
    if (sh < nh) {
      smax[row_id * H + h0 + sh] = m_out;
      ssum[row_id * H + h0 + sh] = l_out;
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kMaxTiles; ++t) {
    const int ct = wave + 4 * t;
    if (ct >= nt) break;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * g + r < nh) out[(row_id * H + h0 + 4 * g + r) * dv + 16 * ct + col] = o[t][r] * inv_s[4 * g + r];
  }
}

__global__ void __launch_bounds__(kThreads, 1)
attn_f32_bwd_kernel(const float* __restrict__ q, const float* __restrict__ kv, const int32_t* __restrict__ idx,
                    const float* __restrict__ out, const float* __restrict__ dout, const float* __restrict__ smax,
                    const float* __restrict__ ssum, float* __restrict__ dq, float* __restrict__ dkv, int S, int s_kv,
                    int H, int K, int dqk, int dv, float scale, int64_t q_offset, const float* __restrict__ sinks,
                    float* __restrict__ dsink) {
  __shared__ __align__(16) float tile[kBN * kLd];
  __shared__ __align__(16) float qs[kHT * kLd], dos[kHT * kLd];
  __shared__ __align__(16) float ps[kHT * kPs], ds[kHT * kPs];  // S, then P | dP, then dS: [head][key]
  __shared__ int keys[kBN];
  const int tok = blockIdx.x, h0 = blockIdx.y * kHT, b = blockIdx.z, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int64_t row_id = (int64_t)b * S + tok;
  const int32_t* ridx = idx + row_id * K;
  const int64_t limit = tok + q_offset;
  const float* kvb = kv + (int64_t)b * s_kv * dqk;
  float* dkvb = dkv + (int64_t)b * s_kv * dqk;
  const int nh = min(kHT, H - h0);
  const int nblk = (K + kBN - 1) / kBN;
  int key;
  uint32_t vm = block_slots(ridx, 0, K, s_kv, limit, lane, key);
  RowRegs rr;
  load_rows(rr, kvb, key, wave, lane, dqk);
  load_heads(qs, q + (row_id * H + h0) * dqk, nh, dqk, tid);
  load_heads(dos, dout + (row_id * H + h0) * dv, nh, dv, tid);
  // thread = (head tid / 16, keys 2 (tid % 16), + 1): the row's lse and delta = dO . O
  const int sh = tid >> 4, sk = 2 * (tid & 15);
  const int64_t hr = row_id * H + h0 + min(sh, nh - 1);
  const float sm = ssum[hr];
  const float lse = (sh < nh && sm > 0.f) ? smax[hr] + logf(sm) : INFINITY;  // +inf -> P = 0
  float delta = 0.f;
  for (int c = 4 * (tid & 15); c < dv; c += 64) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(out + hr * dv + c), y = *reinterpret_cast<const f32x4*>(dout + hr * dv + c);
#pragma unroll
    for (int r = 0; r < 4; ++r) delta = fmaf(x[r], y[r], delta);
  }
  delta += lane_xor<1>(delta);
  delta += lane_xor<2>(delta);
  delta += lane_xor<4>(delta);
  delta += lane_xor<8>(delta);
  if (sinks && (tid & 15) == 0 && sh < nh) atomicAdd(&dsink[h0 + sh], -expf(sinks[h0 + sh] - lse) * delta);
  const int nt = dqk / 16, ntv = dv / 16;
  f32x4 dqa[kMaxTiles];  // heads 4g + r, column 16 (wave + 4 t) + col
#pragma unroll
  for (int t = 0; t < kMaxTiles; ++t) dqa[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int blk = 0; blk < nblk; ++blk) {
    store_rows(rr, tile, vm, wave, lane, dqk);
    const uint32_t vmask = vm;
    if (tid < kBN) keys[tid] = key;
    __syncthreads();
    if (blk + 1 < nblk) {
      vm = block_slots(ridx, blk + 1, K, s_kv, limit, lane, key);
      load_rows(rr, kvb, key, wave, lane, dqk);
    }
    if (vmask == 0u) {  // (workgroup-uniform) no usable key
      __syncthreads();
      continue;
    }
    {  // waves 0, 1: S of key tiles 0, 1; waves 2, 3: dP of them.  In two column halves, which
       // gives S the forward's bits (the rounding of S then cancels in P = exp(S - lse): dQ is off by
       // 5.4e-7 from fp64, 8.7e-7 with S in one chain) and dP a shorter chain
      const int kt = wave & 1, d = wave < 2 ? dqk : dv, mid = (d / 16 / 2) * 16;
      const float* rows = wave < 2 ? qs : dos;
      const f32x4 x = dot_rows(tile + 16 * kt * kLd, rows, 0, mid, col, g) +
                      dot_rows(tile + 16 * kt * kLd, rows, mid, d, col, g);
      *reinterpret_cast<f32x4*>(&(wave < 2 ? ps : ds)[col * kPs + 16 * kt + 4 * g]) = x;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = sh * kPs + sk + e;
      const float p = (vmask >> (sk + e) & 1u) ? expf(ps[i] * scale - lse) : 0.f;
      const float d = p * (ds[i] - delta);
      ps[i] = p;
      ds[i] = d;
    }
    __syncthreads();
    f32x4 d4[2];  // dS of head col, keys 16 s + 4g .. +3
#pragma unroll
    for (int s = 0; s < 2; ++s) d4[s] = *reinterpret_cast<const f32x4*>(&ds[col * kPs + 16 * s + 4 * g]);
    // operands of the key gradients: key 16 s + col, heads 4g + j
    float dk4[2][4], pk4[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dk4[s][j] = ds[(4 * g + j) * kPs + 16 * s + col] * scale;
        pk4[s][j] = ps[(4 * g + j) * kPs + 16 * s + col];
      }
#pragma unroll
    for (int t = 0; t < kMaxTiles; ++t) {
      const int ct = wave + 4 * t;
      if (ct >= nt) break;
      const int cc = 16 * ct + col;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) dqa[t] = mfma_f32(d4[s][j], tile[(16 * s + 4 * g + j) * kLd + cc], dqa[t]);
      f32x4 c[2] = {(f32x4){0.f, 0.f, 0.f, 0.f}, (f32x4){0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float qv = qs[(4 * g + j) * kLd + cc];
#pragma unroll
        for (int s = 0; s < 2; ++s) c[s] = mfma_f32(dk4[s][j], qv, c[s]);
      }
      if (ct < ntv) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float ov = dos[(4 * g + j) * kLd + cc];
#pragma unroll
          for (int s = 0; s < 2; ++s) c[s] = mfma_f32(pk4[s][j], ov, c[s]);
        }
      }
      // keys 16 s + 4g + r, column cc: the sum over the 16 heads
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int kk = 16 * s + 4 * g + r;
          if (vmask >> kk & 1u) atomicAdd(&dkvb[(int64_t)keys[kk] * dqk + cc], c[s][r]);
        }
    }
    __syncthreads();  // the tile, the scores and the keys are rewritten
  }
#pragma unroll
  for (int t = 0; t < kMaxTiles; ++t) {
    const int ct = wave + 4 * t;
    if (ct >= nt) break;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * g + r < nh) dq[(row_id * H + h0 + 4 * g + r) * dqk + 16 * ct + col] = dqa[t][r] * scale;
  }
}

bool aligned16(const void* p) { return (uintptr_t)p % 16 == 0; }

}  // namespace

// The tile kernels read rows 16 bytes at a time and columns in steps of 16; a token's heads
// are taken 16 at a time.
bool attn_f32_fits(int64_t d_qk, int64_t d_v, int64_t n_heads) {
  return d_qk % 16 == 0 && d_v % 16 == 0 && d_qk <= kMaxD && d_v <= d_qk && n_heads <= 65535 * kHT;
}

int attn_f32_fwd(const float* q, const float* kv, const int32_t* indices, float* out, float* smax, float* ssum,
                 int64_t batch, int64_t s_q, int64_t s_kv, int64_t n_heads, int64_t d_qk, int64_t d_v, int64_t topk,
                 float scale, int64_t q_offset, const float* sinks, hipStream_t st) {
  const dim3 grid((unsigned)s_q, ceil_div(n_heads, kHT), (unsigned)batch);
  const TimedLaunch tl("attn_f32_fwd_kernel", st);
  attn_f32_fwd_kernel<<<grid, kThreads, 0, st>>>(q, kv, indices, out, smax, ssum, (int)s_q, (int)s_kv, (int)n_heads,
                                                 (int)topk, (int)d_qk, (int)d_v, scale, q_offset, sinks);
  return check_launch("dsa_sparse_mla_fwd(f32)");
}

int attn_f32_bwd(const float* q, const float* kv, const int32_t* indices, const float* out, const float* dout,
                 const float* smax, const float* ssum, float* dq, float* dkv, int64_t batch, int64_t s_q, int64_t s_kv,
                 int64_t n_heads, int64_t d_qk, int64_t d_v, int64_t topk, float scale, int64_t q_offset,
                 const float* sinks, float* dsink, hipStream_t st) {
  const dim3 grid((unsigned)s_q, ceil_div(n_heads, kHT), (unsigned)batch);
  const TimedLaunch tl("attn_f32_bwd_kernel", st);
  attn_f32_bwd_kernel<<<grid, kThreads, 0, st>>>(q, kv, indices, out, dout, smax, ssum, dq, dkv, (int)s_q, (int)s_kv,
                                                 (int)n_heads, (int)topk, (int)d_qk, (int)d_v, scale, q_offset, sinks,
                                                 dsink);
  return check_launch("dsa_sparse_mla_bwd(f32)");
}

bool attn_f32_aligned(const void* a, const void* b, const void* c, const void* d) {
  return aligned16(a) && aligned16(b) && aligned16(c) && aligned16(d);
}

}  // namespace dsa
