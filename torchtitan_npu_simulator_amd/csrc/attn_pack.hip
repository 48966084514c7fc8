// The plan of token-packed attention (attn_pack.h): per group the union of its tokens'
// selected keys, the tokens' bit masks over it, and the slot of every selection.
//
// One workgroup per group.  The union is a bitmap of the keys in LDS (one bit per key); a
// scan of the words' bit counts gives every key its slot.  Bound by the two reads of the
// group's index rows and by the LDS atomics (one per selection and pass).
#include <algorithm>
#include <type_traits>

#include "attn_pack.h"

namespace dsa {
namespace {

constexpr int kPlanThreads = 512;
constexpr int kPlanWaves = kPlanThreads / 64;
constexpr uint32_t kRepeats = 0x80000000u;    // (PackView::sel) the group has repeated slots
constexpr int64_t kPackMaxKeys = 1 << 17;     // bitmap and word offsets: 24 KB of LDS; 8 v + t of a repeat in 31 bits
constexpr int64_t kPackMaxMaskWords = 9216;   // 36 KB of LDS
constexpr int64_t kPlanLds = 63 * 1024;       // dynamic LDS of the plan: the above and room to sort repeats
constexpr int64_t kSortMax = 4096;
static_assert(kPackMaxKeys / 32 * 6 + kPackMaxMaskWords * 4 <= kPlanLds, "the plan fits without a sort buffer");

__device__ __forceinline__ bool plan_slot_ok(int v, int s_kv, int64_t limit) {
  return v >= 0 && v < s_kv && (int64_t)v <= limit;
}

// pairs of a bitonic merge over n elements (half the next power of two)
__device__ __forceinline__ int len_pairs(int n) { return n > 1 ? 1 << (31 - __clz(n - 1)) : 0; }

__global__ void __launch_bounds__(kPlanThreads)
pack_plan_kernel(const int32_t* __restrict__ indices, int S, int s_kv, int K, int64_t q_offset, PackView pk,
                 int32_t* __restrict__ idx_out, uint32_t* __restrict__ mask_out, int32_t* __restrict__ count_out,
                 int sort_cap) {
  extern __shared__ uint32_t lds[];
  __shared__ int wsum[kPlanWaves];
  __shared__ int sh_rep;  // repeats found
  const int nw = (s_kv + 31) >> 5;
  uint32_t* bits = lds;                      // [nw] keys of the union
  uint32_t* mk = lds + nw;                   // [tt][words]
  uint16_t* pre = reinterpret_cast<uint16_t*>(mk + pk.tt * pk.words);  // [nw] slots before the word
  int32_t* srt = reinterpret_cast<int32_t*>(mk + pk.tt * pk.words + (nw + 1) / 2);  // [sort_cap] repeats
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = (int)(gridDim.x - 1u - blockIdx.x), b = blockIdx.y;  // longest rows first
  const int tok0 = grp * pk.tt, nt = min(pk.tt, S - tok0);
  const int64_t row0 = (int64_t)b * S + tok0;
  const int32_t* src = indices + row0 * K;   // nt rows of K, consecutive
  const int n_el = nt * K;
  int32_t* io = idx_out + ((int64_t)b * pk.groups + grp) * pk.cap;
  uint32_t* mo = mask_out + ((int64_t)b * pk.groups + grp) * pk.tt * pk.words;

  for (int i = tid; i < nw + pk.tt * pk.words; i += kPlanThreads) lds[i] = 0u;
  if (tid < 4) pk.redo[((int64_t)b * pk.groups + grp) * 4 + tid] = 0u;
  if (tid == 0) {
    sh_rep = 0;
    if (pk.suspect) pk.suspect[(int64_t)b * pk.groups + grp] = 0;
  }
  __syncthreads();
  // every load of a batch is issued before the first use
  constexpr int kU = 8;
  auto for_each = [&](auto&& f) {
    for (int e0 = 0; e0 < n_el; e0 += kPlanThreads * kU) {
      int v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = src[min(e0 + tid + kPlanThreads * u, n_el - 1)];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int e = e0 + tid + kPlanThreads * u;
        if (e < n_el) {
          const int t = (int)((unsigned)e / (unsigned)K);
          f(e, t, v[u], plan_slot_ok(v[u], s_kv, (int64_t)(tok0 + t) + q_offset));
        }
      }
    }
  };
  for_each([&](int, int, int v, bool ok) {
    if (ok) atomicOr(&bits[v >> 5], 1u << (v & 31));
  });
  __syncthreads();
  // slots before each word: every thread owns a run of consecutive words
  const int per = (nw + kPlanThreads - 1) / kPlanThreads;
  const int w0 = min(nw, tid * per), w1 = min(nw, w0 + per);
  int mine = 0;
  for (int w = w0; w < w1; ++w) mine += __popc(bits[w]);
  int inc = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(inc, d, 64);
    if (lane >= d) inc += o;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int base = inc - mine, n = 0;
  for (int w = 0; w < kPlanWaves; ++w) {
    if (w < wave) base += wsum[w];
    n += wsum[w];
  }
  for (int w = w0; w < w1; ++w) {
    pre[w] = (uint16_t)base;
    base += __popc(bits[w]);
  }
  __syncthreads();
  auto slot_of = [&](int v) -> int {
    return (int)pre[v >> 5] + __popc(bits[v >> 5] & ((1u << (v & 31)) - 1u));
  };
  // keys out, one thread per 32-key word
  for (int w = tid; w < nw; w += kPlanThreads) {
    uint32_t m = bits[w];
    int p = pre[w];
    if (pk.sel) pk.sel[((int64_t)b * nw + w) * pk.groups + grp] = make_uint2(m, (uint32_t)p);
    while (m) {
      io[p++] = 32 * w + __builtin_ctz(m);
      m &= m - 1u;
    }
  }
  for_each([&](int e, int t, int v, bool ok) {
    int p = -1;
    if (ok) {
      p = slot_of(v);
      const uint32_t bit = 1u << (p & 31);
      if (atomicOr(&mk[t * pk.words + (p >> 5)], bit) & bit) io[n + atomicAdd(&sh_rep, 1)] = 8 * v + t;
    }
    if (pk.pos) pk.pos[row0 * K + e] = ok ? (uint16_t)p : kPackNoSlot;
  });
  __syncthreads();
  const int rep = sh_rep;
  if (rep > 0) {
    // some token lists a key more than once (top-k output never does).  Every further occurrence
    // takes a slot of its own after the union, ordered by key and token, so the slots do not
    // depend on the order in which the threads ran (pos keeps the key's first slot, whose
    // probability is the repeat's too), and a key's reduction finds its run.  A bitonic sort
    // in place, every comparison ascending (the first step of a merge pairs mirrored
    // elements), so places past the last one count as +inf; in LDS where they fit.  1024 tokens,
    // 16 heads, 256 keys drawn with replacement: forward 330 us with one thread that walked
    // the lists, 116 now (distinct keys: 82).
    int32_t* ex = io + n;
    auto sort = [&](auto* x) __attribute__((always_inline)) {
      for (int len = 2; len < 2 * rep; len <<= 1)
        for (int j = len >> 1; j > 0; j >>= 1) {
          const bool mirror = 2 * j == len;
          for (int i = tid; i < len_pairs(rep); i += kPlanThreads) {
            const int o = i & (j - 1), base = 2 * (i - o);
            const int lo = base + o, hi = mirror ? base + 2 * j - 1 - o : lo + j;
            if (hi < rep) {
              const int u = x[lo], w = x[hi];
              if (u > w) {
                x[lo] = w;
                x[hi] = u;
              }
            }
          }
          __syncthreads();
        }
    };
    auto give = [&](int i, int x) {  // the i-th repeat's slot
      const int t = x & 7, p = n + i;
      ex[i] = x >> 3;
      atomicOr(&mk[t * pk.words + (p >> 5)], 1u << (p & 31));
    };
    if (rep <= sort_cap) {  // in LDS
      for (int i = tid; i < rep; i += kPlanThreads) srt[i] = ex[i];
      __syncthreads();
      sort(srt);
      for (int i = tid; i < rep; i += kPlanThreads) give(i, srt[i]);
    } else {
      sort(ex);
      for (int i = tid; i < rep; i += kPlanThreads) give(i, ex[i]);
    }
    __syncthreads();
    if (pk.sel)
      for (int w = tid; w < nw; w += kPlanThreads)
        pk.sel[((int64_t)b * nw + w) * pk.groups + grp] = make_uint2(bits[w], (uint32_t)pre[w] | kRepeats);
    if (pk.distinct && tid == 0) pk.distinct[(int64_t)b * pk.groups + grp] = n;
    n += rep;
  }
  const int used = (n + 31) >> 5;
  for (int i = tid; i < pk.tt * used; i += kPlanThreads) {
    const int t = i / used, w = i - t * used;
    mo[t * pk.words + w] = mk[t * pk.words + w];
  }
  for (int j = n + tid; j < 32 * used; j += kPlanThreads) io[j] = -1;
  if (tid == 0) count_out[(int64_t)b * pk.groups + grp] = n;
}

// one workgroup per token of the chunk
__global__ void __launch_bounds__(256)
pack_mass_gather_kernel(PackView pk, float* __restrict__ mass, int S, int K, int g0, int n) {
  const int tok = g0 * pk.tt + blockIdx.x, b = blockIdx.y;
  const int lg = (int)blockIdx.x / pk.tt, t = (int)blockIdx.x - lg * pk.tt;
  const float* src = pk.mass + (((int64_t)b * n + lg) * pk.tt + t) * pk.cap;
  const int64_t row = ((int64_t)b * S + tok) * K;
  for (int j = threadIdx.x; j < K; j += 256) {
    const uint16_t p = pk.pos[row + j];
    mass[row + j] = p == kPackNoSlot ? 0.f : src[p];
  }
}

// One workgroup per key, its four waves on a quarter of the groups each: the groups are looked
// at 64 at a time (one sel entry per lane), and the contribution rows of those that hold the
// key are summed in fp32, eight rows in flight; the waves' sums meet in LDS.  A row is read
// once, non-temporally; the key has one owner, so no atomics are issued and the order of the
// sum is fixed.  (One wave per key left the chip idle with few keys: 700 tokens, 64 heads,
// top-1000 90 -> 44 us.)  (A token-major pair list as dsa_csr.h builds it would be read
// and sorted at the lists' capacity, several times the union.)
template <int kChunks>
__global__ void __launch_bounds__(256)
pack_dkv_reduce_kernel(PackView pk, const uint16_t* __restrict__ cbuf, float* __restrict__ acc_out, int s_kv, int g0,
                       int n) {
  constexpr int kWidth = kChunks * 8;
  constexpr int kRows = 8;
  __shared__ float sums[3][kWidth];  // waves 1..3
  __shared__ int held;
  const int k = blockIdx.x, b = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (threadIdx.x == 0) held = 0;
  __syncthreads();
  // (whole steps of 64 groups per wave)
  const int per = ((n + 3) / 4 + 63) / 64 * 64, n0 = min(n, wave * per), n1 = min(n, n0 + per);
  const uint2* sel = pk.sel + ((int64_t)b * pk.key_words + (k >> 5)) * pk.groups + g0;
  const uint32_t bit = 1u << (k & 31);
  const uint16_t* cb = cbuf + (int64_t)b * n * pk.cap * kWidth;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // chunk `lane`
  float acc2[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // (72 chunks) chunk 64 + (lane & 7)
  auto add8 = [](float (&a)[8], const u32x4& v) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a[2 * r] += bf16_lo(v[r]);
      a[2 * r + 1] += bf16_hi(v[r]);
    }
  };
  auto add8_times = [](float (&a)[8], const u32x4& v, float x) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a[2 * r] = fmaf(x, bf16_lo(v[r]), a[2 * r]);
      a[2 * r + 1] = fmaf(x, bf16_hi(v[r]), a[2 * r + 1]);
    }
  };
  // adds, for every lane g of m, the row of group gb + g at that lane's slot (that lane's `times`
  // times), in order, kRows rows in flight
  auto add_rows = [&](uint64_t m, int gb, int slot, auto timed, float times) __attribute__((always_inline)) {
    constexpr bool kTimed = decltype(timed)::value;
    while (m) {
      u32x4 v[kRows], w[kRows];
      float x[kRows];
      int cnt = 0, g = 0;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        if (m) {  // (past the last one the row before is read again and not added)
          g = __builtin_ctzll(m);
          m &= m - 1;
          ++cnt;
        }
        const uint16_t* row = cb + ((int64_t)(gb + g) * pk.cap + __builtin_amdgcn_readlane(slot, g)) * kWidth;
        if constexpr (kTimed) x[u] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(times), g));
        v[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + 8 * lane));
        if constexpr (kChunks == 72)
          w[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + 512 + 8 * (lane & 7)));
      }
#pragma unroll
      for (int u = 0; u < kRows; ++u)
        if (u < cnt) {
          if constexpr (kTimed) {
            add8_times(acc, v[u], x[u]);
            if constexpr (kChunks == 72) add8_times(acc2, w[u], x[u]);
          } else {
            add8(acc, v[u]);
            if constexpr (kChunks == 72) add8(acc2, w[u]);
          }
        }
    }
  };
  bool any = false;
  for (int gb = n0; gb < n1; gb += 64) {
    const uint2 e = gb + lane < n1 ? sel[gb + lane] : make_uint2(0u, 0u);
    const int slot = (int)(e.y & ~kRepeats) + __popc(e.x & (bit - 1u));
    uint64_t m = __ballot((e.x & bit) != 0u);
    any |= m != 0;
    add_rows(m, gb, slot, std::false_type{}, 1.f);
    if (__ballot((e.y & kRepeats) != 0u) == 0) continue;
    // groups with repeated keys: each lane finds the key's run among its group's slots after the
    // union (ordered by key and token), and in it the slots of one token after the other, whose
    // rows are the same: one is read, times their number.  (A walk over every repeat for every
    // key: backward of 2048 tokens, 16 heads, 1024 keys of which half are key 0 218 ms, now 1.8;
    // 4096 tokens with 512 keys drawn with replacement 50 -> 1.7 ms; distinct keys 1.0.)
    const int64_t pg = (int64_t)b * pk.groups + g0 + min(gb + lane, n - 1);
    const int32_t* list = pk.idx + pg * pk.cap;
    auto first = [&](int a, int z, auto&& before) {  // the first slot of [a, z) that is not `before`
      while (a < z) {
        const int mid = (a + z) >> 1;
        if (before(mid)) a = mid + 1;
        else z = mid;
      }
      return a;
    };
    int lo = 0, hi = 0;
    if (e.y & kRepeats) {
      const int end = pk.count[pg];
      lo = first(pk.distinct[pg], end, [&](int j) { return list[j] < k; });
      hi = first(lo, end, [&](int j) { return list[j] == k; });
    }
    for (int t = 0; t < pk.tt; ++t) {
      if (__ballot(lo < hi) == 0) break;
      const uint32_t* bits = pk.mask + (pg * pk.tt + t) * pk.words;
      const int next = first(lo, hi, [&](int j) { return (bits[j >> 5] >> (j & 31) & 1u) != 0u; });
      add_rows(__ballot(lo < next), gb, lo, std::true_type{}, (float)(next - lo));
      lo = next;
    }
  }
  if (any && lane == 0) held = 1;
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < 8; ++r) sums[wave - 1][8 * lane + r] = acc[r];
    if constexpr (kChunks == 72)
      if (lane < 8)
#pragma unroll
        for (int r = 0; r < 8; ++r) sums[wave - 1][512 + 8 * lane + r] = acc2[r];
  }
  __syncthreads();
  if (wave > 0 || !held) return;
#pragma unroll
  for (int u = 0; u < 3; ++u)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      acc[r] += sums[u][8 * lane + r];
      if constexpr (kChunks == 72) acc2[r] += sums[u][512 + 8 * (lane & 7) + r];
    }
  float* d = acc_out + ((int64_t)b * s_kv + k) * kWidth;
  auto put = [](float* p, const float (&a)[8]) {
    float4* d4 = reinterpret_cast<float4*>(p);
    float4 x = d4[0], y = d4[1];
    x.x += a[0]; x.y += a[1]; x.z += a[2]; x.w += a[3];
    y.x += a[4]; y.y += a[5]; y.z += a[6]; y.w += a[7];
    d4[0] = x;
    d4[1] = y;
  };
  put(d + 8 * lane, acc);
  if constexpr (kChunks == 72)
    if (lane < 8) put(d + 512 + 8 * lane, acc2);
}

int64_t al256(int64_t x) { return (x + 255) / 256 * 256; }

}  // namespace

// Packing never adds gathered blocks (a union is at most the sum of its lists), so it is
// considered wherever a token leaves half of the workgroup's rows idle or more and the tokens
// would run in two rounds of the 256 CUs or more: ceil(tokens / 256) tokens per group keep
// one workgroup per CU.  A call with no causal test (q_offset >= s_kv: the sequences of a
// packed batch on global key rows) packs from 1024 tokens: the union changes the order in
// which a row's keys are summed, and a shorter batch keeps the results of per-sequence calls
// bit for bit.
//
// What a group saves over its tokens is the overlap of their lists, about s_kv / (tt topk) for
// lists drawn at random (top-k lists of neighbours overlap more); the limits below keep calls
// of a causal test whose random lists were not faster packed on the one-token kernels.  (Without
// the test a row's keys lie in its own sequence or window, which s_kv says nothing about.)
// Time of one token over packed, top-k lists at random, 64 | 32 | 16 heads (2 | 4 | 8 tokens):
//   forward, 4096 tokens, top-1024: s_kv 16384 1.02 | 1.12 | 1.29, 32768 0.98 | 1.07 | 1.15,
//     131072 0.93 | 1.02 | 1.07.
//   backward, where every key looks at every group: top-2048, s_kv 16384 1.06 | 1.22 | 1.55,
//     65536 0.95 | 1.02 | 1.10, 131072 0.87 | 0.96 | 1.04; top-256, 16384 1.03 | 1.14 | 1.28,
//     65536 0.86 | 0.96 | 1.10; 1024 tokens (512 | 256 | 256 groups), top-1024, 32768 1.02 |
//     1.08 | 1.10, 65536 0.95 | 1.05 | 1.07, 131072 0.86 | 0.95 | 0.96.
//   mass, whose one-token form runs two workgroups per CU: 1024 tokens and keys, top-64 0.82 |
//     0.84 | 0.84, top-512 1.13 | 1.16 | 1.23; 4096 tokens, s_kv 4096, top-256 0.93 | 1.11 | 1.34,
//     top-2048 1.45 | 2.2 | 3.0; s_kv 32768, top-1024 0.92 | 0.97 | 1.01.
static bool overlap_pays(int64_t batch, int64_t s_q, int64_t s_kv, int64_t topk, int64_t tt, PackParts parts) {
  const int64_t tokens = batch * s_q, lists = tt * topk;
  switch (parts) {
    case PackParts::kForward:
      return tt > 2 || s_kv <= std::max<int64_t>(16384, 16 * topk);
    case PackParts::kBackward:
      return s_kv <= tt * std::max<int64_t>(8192, 8 * topk) || s_kv * batch * pack_groups(s_q, (int)tt) <= (1 << 24);
    default:
      if (topk >= 512 && s_kv <= (tokens >= 2048 ? 2 : 1) * lists) return true;
      if (tokens >= 8192 && s_kv <= 8 * lists) return true;
      return tokens >= 2048 && tt > 2 && (s_kv <= 4 * lists || topk <= (tt >= 6 ? 256 : 64));
  }
}

int pack_tokens(int64_t batch, int64_t s_q, int64_t s_kv, int64_t n_heads, int64_t topk, int64_t q_offset,
                PackParts parts) {
  if (n_heads <= 0 || n_heads > kPackRows / 2 || batch <= 0 || s_q <= 0 || topk <= 0) return 1;
  const bool causal = q_offset < s_kv;
  if (batch * s_q < (causal ? 512 : 1024)) return 1;
  if (s_kv > kPackMaxKeys) return 1;
  int64_t tt = kPackRows / pack_hp(n_heads);
  tt = std::min<int64_t>(tt, (batch * s_q + 255) / 256);
  tt = std::min<int64_t>(tt, s_q);
  tt = std::min<int64_t>(tt, 65504 / topk);  // slots are 16-bit
  while (tt > 1 && tt * (pack_cap(topk, (int)tt) / 32) > kPackMaxMaskWords) --tt;
  if (tt <= 1 || (causal && !overlap_pays(batch, s_q, s_kv, topk, tt, parts))) return 1;
  return (int)tt;
}

int64_t pack_plan_bytes(int64_t batch, int64_t s_q, int64_t s_kv, int64_t topk, int tt, PackParts parts) {
  const int64_t g = pack_groups(s_q, tt) * batch, cap = pack_cap(topk, tt);
  return al256(g * cap * 4) + al256(g * tt * (cap / 32) * 4) + al256(g * 4) + al256(g * 16) +
         (parts != PackParts::kForward ? al256(batch * s_q * topk * 2) : 0) +
         (parts == PackParts::kBackward ? al256(g * ((s_kv + 31) / 32) * 8) + 2 * al256(g * 4) : 0);
}

int pack_plan_build(const int32_t* indices, int64_t batch, int64_t s_q, int64_t s_kv, int64_t n_heads, int64_t topk,
                    int64_t q_offset, int tt, PackParts parts, void* ws, hipStream_t st, PackView* view) {
  PackView pk;
  pk.tt = tt;
  pk.hp = pack_hp(n_heads);
  pk.groups = (int)pack_groups(s_q, tt);
  pk.cap = (int)pack_cap(topk, tt);
  pk.words = pk.cap / 32;
  pk.key_words = (int)((s_kv + 31) / 32);
  const int64_t g = batch * pk.groups;
  char* p = (char*)ws;
  auto take = [&](int64_t bytes) {
    char* r = p;
    p += al256(bytes);
    return r;
  };
  int32_t* idx = (int32_t*)take(g * pk.cap * 4);
  uint32_t* mask = (uint32_t*)take(g * tt * pk.words * 4);
  int32_t* count = (int32_t*)take(g * 4);
  pk.redo = (uint32_t*)take(g * 16);
  if (parts != PackParts::kForward) pk.pos = (uint16_t*)take(batch * s_q * topk * 2);
  if (parts == PackParts::kBackward) {
    pk.sel = (uint2*)take(g * pk.key_words * 8);
    pk.distinct = (int32_t*)take(g * 4);
    pk.suspect = (int32_t*)take(g * 4);
  }
  const int64_t nw = pk.key_words;
  const int64_t used = nw * 4 + (int64_t)tt * pk.words * 4 + (nw + 1) / 2 * 4;
  const int sort_cap = (int)std::min<int64_t>(kSortMax, (kPlanLds - used) / 4);
  const size_t lds = (size_t)(used + sort_cap * 4);
  {
    const TimedLaunch tl("pack_plan_kernel", st);
    pack_plan_kernel<<<dim3((unsigned)pk.groups, (unsigned)batch), kPlanThreads, lds, st>>>(
        indices, (int)s_q, (int)s_kv, (int)topk, q_offset, pk, idx, mask, count, sort_cap);
  }
  pk.idx = idx;
  pk.mask = mask;
  pk.count = count;
  *view = pk;
  return check_launch("pack_plan");
}

int pack_dkv_reduce(const PackView& view, const uint16_t* cbuf, float* acc, int64_t batch, int64_t s_kv, int64_t width,
                    int64_t g0, int64_t n, hipStream_t st) {
  const dim3 grid((unsigned)s_kv, (unsigned)batch);
  const TimedLaunch tl(width == 576 ? "pack_dkv_reduce_kernel<72>" : "pack_dkv_reduce_kernel<64>", st);
  if (width == 576)
    pack_dkv_reduce_kernel<72><<<grid, 256, 0, st>>>(view, cbuf, acc, (int)s_kv, (int)g0, (int)n);
  else
    pack_dkv_reduce_kernel<64><<<grid, 256, 0, st>>>(view, cbuf, acc, (int)s_kv, (int)g0, (int)n);
  return check_launch("pack_dkv_reduce");
}

int pack_mass_gather(const PackView& view, float* mass, int64_t batch, int64_t s_q, int64_t topk, int64_t g0, int64_t n,
                     hipStream_t st) {
  const int64_t toks = std::min<int64_t>(n * view.tt, s_q - g0 * view.tt);
  const TimedLaunch tl("pack_mass_gather_kernel", st);
  pack_mass_gather_kernel<<<dim3((unsigned)toks, (unsigned)batch), 256, 0, st>>>(view, mass, (int)s_q, (int)topk,
                                                                                (int)g0, (int)n);
  return check_launch("pack_mass_gather");
}

}  // namespace dsa
