// Token packing for the gathered-attention kernels: a workgroup of those kernels holds 128
// query rows (head lanes).  With fewer heads a token fills only part of it, so several
// consecutive tokens of one batch element share a workgroup ("group"): the group gathers the
// union of its tokens' selected keys once, and every row masks the keys its own token did
// not select.
//
// What bounds the one-token kernels with few heads is the gather and the G / C round trips,
// which cost the same whatever the head count; a group shares them (and the dKV contribution
// rows are summed over its tokens before they reach memory).  Forward + backward, one token
// per workgroup against packed: S = 4096, 16 heads, top-2048 8.00 -> 1.67 ms (the forward
// 1.76 -> 0.38, scores 1.69 -> 0.38, dQ 0.95 -> 0.21, contributions 2.07 -> 0.39, reduction
// 1.27 -> 0.22, plan 2 x 0.055); 6080 tokens in six sequences, 32 heads, top-1024
// 5.70 -> 2.26 ms.
//
// A group of tt tokens has rows (token, head) at lane row hp * token + head, hp = the head
// count rounded up to 16.  Its plan is
//   idx[cap]          the union's keys in ascending order (a key repeated inside one token's
//                     list appears again at the end, once per extra occurrence, these by key
//                     and token), -1 from the last to the end of its 32-slot block;
//   mask[tt][words]   bit j of word j / 32: slot j of idx is selected by the token;
//   count             used slots;
//   redo[4]           (cleared by the plan) the rows whose O the forward found not finite, as bits;
//   pos[tt][K]        (mass, backward) the slot of the token's j-th selection, kPackNoSlot if
//                     unusable;
//   sel[word]         (backward, stored word-major over the groups) the union's keys
//                     32 word .. +31 as bits, with the slot of the first of them; bit 31 of
//                     the latter marks a group with repeats;
//   distinct          (backward) slots before the repeats;
//   suspect           (backward, cleared by the plan) bwd_dqk_kernel found a dQ of the group
//                     that is not finite before it redid it.
// cap = tt * K rounded up to whole 32-slot blocks always holds the union with its repeats.
//
// A key that a row's token did not select has weight 0 there, but 0 times an infinity or a NaN
// is a NaN: a row that is not finite would reach every token of its group (earlier tokens,
// other sequences of a packed batch).  Every sum over the union is therefore looked at once
// it is complete, and where it is not finite it is formed again from the token's own slots
// alone (O by the forward's fixup pass, dQ in bwd_dqk_kernel's epilogue, dKV at the end of
// bwd_contrib_kernel where the group is suspect).  The look takes 2 us of 430 in the forward
// kernel and in the backward's (6080 tokens, 32 heads, top-1024); S = 4096, 16 heads,
// top-2048 with one NaN key that half of the tokens select: the sums again take 7 ms
// (forward; formed in the kernel's own epilogue 17 ms, and 3 % of its time on finite data for
// the registers) and 19 ms (backward).
#pragma once
#include "dsa_common.h"

namespace dsa {

constexpr int kPackRows = 128;
constexpr uint16_t kPackNoSlot = 0xffff;

// device-side view, passed to the kernels by value
struct PackView {
  const int32_t* idx = nullptr;    // [batch][groups][cap]
  const uint32_t* mask = nullptr;  // [batch][groups][tt][words]
  const int32_t* count = nullptr;  // [batch][groups]
  uint32_t* redo = nullptr;        // [batch][groups][4]
  uint16_t* pos = nullptr;         // [batch][S][K]: mass and backward; the next three: backward
  uint2* sel = nullptr;            // [batch][key words][groups]
  int32_t* distinct = nullptr;     // [batch][groups]
  int32_t* suspect = nullptr;      // [batch][groups]
  float* mass = nullptr;           // [batch][chunk groups][tt][cap]: per-token head sums by slot (backward)
  int tt = 1, hp = kPackRows, cap = 0, words = 0, groups = 0, key_words = 0;
};

inline int pack_hp(int64_t n_heads) { return (int)((n_heads + 15) / 16 * 16); }
inline int64_t pack_groups(int64_t s_q, int tt) { return (s_q + tt - 1) / tt; }
inline int64_t pack_cap(int64_t topk, int tt) { return (topk * tt + 31) / 32 * 32; }

// Parts of the plan: the forward takes idx, mask, count and redo, the mass pos too, the backward
// all of it.
enum class PackParts { kForward, kMass, kBackward };
// Tokens per group for a problem (1: the unpacked kernels serve it).
int pack_tokens(int64_t batch, int64_t s_q, int64_t s_kv, int64_t n_heads, int64_t topk, int64_t q_offset,
                PackParts parts);
// Workspace of the plan (256-byte aligned parts).
int64_t pack_plan_bytes(int64_t batch, int64_t s_q, int64_t s_kv, int64_t topk, int tt, PackParts parts);
// Enqueues the plan into ws and fills *view.
int pack_plan_build(const int32_t* indices, int64_t batch, int64_t s_q, int64_t s_kv, int64_t n_heads, int64_t topk,
                    int64_t q_offset, int tt, PackParts parts, void* ws, hipStream_t st, PackView* view);
// For the n groups from g0 of every batch element:
// mass[token][j] = view.mass[token's group][token][pos[token][j]] (0 at unusable slots)
int pack_mass_gather(const PackView& view, float* mass, int64_t batch, int64_t s_q, int64_t topk, int64_t g0, int64_t n,
                     hipStream_t st);
// acc[key] += sum over the groups, in order, of their contribution row at the key's slot:
// cbuf [batch][n][cap][width] bf16, acc [batch][s_kv][width] fp32 (width 576 or 512)
int pack_dkv_reduce(const PackView& view, const uint16_t* cbuf, float* acc, int64_t batch, int64_t s_kv, int64_t width,
                    int64_t g0, int64_t n, hipStream_t st);

// row r of a group: its token (within the group) and head
__device__ __forceinline__ void pack_row(const PackView& pk, int r, int& t, int& head) {
  t = r / pk.hp;
  head = r - t * pk.hp;
}

// The mask words of row r's token (r wave-uniform): read through the constant address space,
// so that a kernel's loop takes them by scalar loads (the plan is complete before the kernel
// starts; a vector load there would be waited for together with the row DMAs).
typedef const __attribute__((address_space(4))) uint32_t pack_word;
__device__ __forceinline__ const pack_word* pack_mask_token(const PackView& pk, int64_t pgrp, int t) {
  return (const pack_word*)(uintptr_t)(pk.mask + (pgrp * pk.tt + t) * pk.words);
}
__device__ __forceinline__ const pack_word* pack_mask_row(const PackView& pk, int64_t pgrp, int r) {
  return pack_mask_token(pk, pgrp, min(r / pk.hp, pk.tt - 1));
}

}  // namespace dsa
