// Exact block top-k by (ordered BF16 score desc, ID asc) of n <= 8 x SEL_BLOCK
// items held in registers: thread t holds the octet of items 8t .. 8t+7 as
// packed 16-bit ordered scores (0 = excluded or absent).
//
// Two histogram passes over the registers find the k-th best score v and the
// count of items above it: 4096 bins of the top 12 bits (LDS atomics), then
// 16 bins of the low 4 bits of the chosen bin.  No candidate list and no
// second read of memory.  Items tied at v are members in ID order (TieRule),
// up to FS_TIE_RANK ties ranked by comparison; beyond that ok = false and the
// caller runs the full selection.
#pragma once

#include "skv_fastsel.h"

namespace skv {

constexpr int OCT_ITEMS = 8 * SEL_BLOCK;  // largest n held one octet per thread

// Half e (0..7, a compile-time constant after unrolling) of an octet.
__device__ __forceinline__ uint32_t oct_half(const u32x4& wv, int e) {
  return (e & 1) ? wv[e >> 1] >> 16 : wv[e >> 1] & 0xffffu;
}

// This thread's octet of a 16-byte aligned row of n ordered scores, items
// beyond n cleared (the row may hold stale values there).
__device__ __forceinline__ uint4 load_oct(const uint16_t* __restrict__ row, int n) {
  const int t = threadIdx.x, valid = n - 8 * t;
  if (valid <= 0) return make_uint4(0, 0, 0, 0);
  const uint4 w = reinterpret_cast<const uint4*>(row)[t];
  if (valid >= 8) return w;
  auto cut = [&](uint32_t x, int q) {  // halves of word q kept: valid - 2q
    const int keep = valid - 2 * q;
    return keep >= 2 ? x : keep == 1 ? (x & 0xffffu) : 0u;
  };
  return make_uint4(cut(w.x, 0), cut(w.y, 1), cut(w.z, 2), cut(w.w, 3));
}

struct OctResult {
  Selection sel;  // v (k-th best score), above (count scoring > v), all
  uint32_t mine;  // member bits of this thread's items (bit 8o + e = item e of octet o)
  bool ok;        // false: too many ties at v to rank here (use the full path), or,
                  // octn_top only, no v found (sel.v = 0: use octn_select)
};

// How items tied at the k-th score are ranked.
enum TieRule {
  TIE_VALUE,  // not at all: only the k-th score is wanted (sel.v)
  TIE_POS,    // the ID is the position: a block scan in thread order, which is
              // position order for one octet per thread
  TIE_ID,     // id(b), the ID of bit b of this thread's items (registers or
              // arithmetic): tied IDs are gathered in LDS, and each is ranked
              // by comparison by the thread that holds it
  TIE_LOAD    // id(position), read from memory: tie_cut
};

// The top k of the NO octets per thread: octet o of thread t holds items
// 8 (t + o SEL_BLOCK) .. +7 (NO = 2: the row's first 8 SEL_BLOCK items, then
// the rest, in the same layout).  hist and ws are cleared (fs_clear, with a
// barrier between), and hold the block's counts on return; the block passes a
// barrier of the caller's before they, or s.tie, are used again.
//
// These selections run on one CU with 16 waves, so their time is the number
// of block-wide phases: six barriers (cleared scratch, counts, two for the
// bin, digit, ties) against 13 when one wave worked out each rank for the
// others and the tied items went through a position list (top-256 of 6000 keys 5.4 -> 4.6 us, threshold and fine selection of
// 8192 centroids 5.9 -> 4.9 us).
template <int NO, TieRule RULE, typename IdFn>
__device__ __forceinline__ OctResult octn_select(const uint4 (&w)[NO], int k, IdFn id,
                                                 uint32_t* hist, SelWords& ws, FastScratch& s,
                                                 int ts = -1) {
  static_assert(NO >= 1 && NO <= 4 && !(RULE == TIE_POS && NO > 1), "octets per thread");
  OctResult res;
  res.ok = true;
  res.mine = 0;
  res.sel.v = 0;
  res.sel.idcut = 0xffffffffu;
  res.sel.above = 0;
  res.sel.all = false;
  u32x4 wv[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) wv[o] = u32x4{w[o].x, w[o].y, w[o].z, w[o].w};
  uint32_t valid = 0;
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t x = oct_half(wv[o], e);
      if (x) {
        atomicAdd(&hist[x >> 4], 1u);
        valid |= 1u << (8 * o + e);
      }
    }
  __syncthreads();
  SKV_TS(ts, 1);
  fs_rank_bin(hist, ws, k);
  __syncthreads();
  SKV_TS(ts, 2);
  const int b1 = ws.sel[0];
  if (b1 < 0) {  // fewer than k valid items: all of them are members
    res.sel.all = true;
    res.sel.above = ws.sel[2];
    res.mine = valid;
    return res;
  }
  const int acc1 = ws.sel[1];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t x = oct_half(wv[o], e);
      if (x && (int)(x >> 4) == b1) atomicAdd(&ws.hist4[x & 15], 1u);
    }
  __syncthreads();
  const DigitRank dr = fs_rank_digit(ws, k, acc1);
  SKV_TS(ts, 3);
  const uint32_t v = ((uint32_t)b1 << 4) | (uint32_t)dr.digit;
  res.sel.v = v;
  res.sel.above = dr.above;
  if (RULE == TIE_VALUE) return res;
  uint32_t gt = 0, eq = 0;
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t x = oct_half(wv[o], e);
      gt |= (uint32_t)(x > v) << (8 * o + e);
      eq |= (uint32_t)(x == v) << (8 * o + e);
    }
  const int need = k - dr.above;  // 1 <= need <= ties
  if (need >= dr.ties) {
    res.mine = gt | eq;
    return res;
  }
  const int c = __popc(eq);
  if (RULE == TIE_POS) {  // ties in position order: thread order, then bit order
    int nt;
    const int exc = block_excl_scan(c, ws.tie_scan, &nt);
    const int take = min(max(need - exc, 0), c);  // this thread's lowest `take` ties
    uint32_t m = 0, rest = eq;
    for (int j = 0; j < take; ++j) {
      m |= rest & (0u - rest);
      rest &= rest - 1;
    }
    res.mine = gt | m;
    return res;
  }
  if (dr.ties > FS_TIE_RANK) {
    res.ok = false;
    return res;
  }
  const int slot0 = c ? atomicAdd(&ws.ntie, c) : 0;
  if constexpr (RULE == TIE_LOAD) {
    int slot = slot0;
    for (uint32_t rest = eq; rest; rest &= rest - 1) {
      const int b = __ffs(rest) - 1;
      s.tie[slot++] = (uint32_t)(8 * ((int)threadIdx.x + (b >> 3) * SEL_BLOCK) + (b & 7));
    }
    __syncthreads();
    const uint32_t idcut = tie_cut(dr.ties, need, id, s, ws);
    slot = slot0;
    for (uint32_t rest = eq; rest; rest &= rest - 1)
      if (s.tie[slot++] <= idcut) gt |= rest & (0u - rest);
    res.mine = gt;
    return res;
  }
  if (c) {
    int slot = slot0;
#pragma unroll
    for (int b = 0; b < 8 * NO; ++b)  // compile-time bit: the IDs may be registers
      if ((eq >> b) & 1u) s.tie[slot++] = id(b);
  }
  __syncthreads();
  int slot = slot0;
  for (uint32_t rest = eq; rest; rest &= rest - 1)  // rank = number of smaller tied IDs
    if (count_below(s.tie, dr.ties, s.tie[slot++]) < need) gt |= rest & (0u - rest);
  res.mine = gt;
  return res;
}

// octn_select for k well below the 8 NO SEL_BLOCK items (NO = 2 or 4): the
// k-th largest thread maximum is at most the k-th largest item (k threads hold
// an item that reaches it), so only items from its bin's floor f up are
// counted, by distance above f (4096 bins of one score step; a few hundred to
// a few thousand LDS additions instead of one per item and a second pass for
// the low digits, which were bound by the additions: threshold and fine
// selection of 32672 centroids 15.4 -> 11.5 us).  hmax and hitem with their
// words are cleared, as for octn_select.  ok = false, with nothing selected
// and sel.v = 0, where the bound says too little and octn_select has to run:
// fewer than k threads hold an item (always for k > SEL_BLOCK; items are then
// not counted, all would land above the last step), or the k-th score lies
// 4095 or more steps above f.  (Select launch with a budget of 2048 out of
// 10240 / 24576 centroids 10.5 / 16.5 us; counting the items all the same, on
// one bin, and selecting over LDS afterwards 36.4 / 54.8.)  ok = false with
// sel.v: too many ties.
template <int NO, TieRule RULE, typename IdFn>
__device__ __forceinline__ OctResult octn_top(const uint4 (&w)[NO], int k, IdFn id, uint32_t* hmax,
                                              uint32_t* hitem, FastScratch& s, int ts = -1) {
  static_assert(RULE == TIE_VALUE || RULE == TIE_ID, "ties by ID");
  OctResult res;
  res.ok = true;
  res.mine = 0;
  res.sel.v = 0;
  res.sel.idcut = 0xffffffffu;
  res.sel.above = 0;
  res.sel.all = false;
  u32x4 wv[NO];
  u16x2 mx = {0, 0};
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    wv[o] = u32x4{w[o].x, w[o].y, w[o].z, w[o].w};
    const uint32_t u[4] = {w[o].x, w[o].y, w[o].z, w[o].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) mx = __builtin_elementwise_max(mx, __builtin_bit_cast(u16x2, u[q]));
  }
  const uint32_t top = max((uint32_t)mx[0], (uint32_t)mx[1]);
  if (top) atomicAdd(&hmax[top >> 4], 1u);
  __syncthreads();
  SKV_TS(ts, 1);
  fs_rank_bin(hmax, s.w[0], k);
  __syncthreads();
  SKV_TS(ts, 2);
  const int b1 = s.w[0].sel[0];
  if (__builtin_expect(b1 < 0, 0)) {
    res.ok = false;
    return res;
  }
  const uint32_t f = max((uint32_t)b1 << 4, 1u);  // at least k items reach it
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t x = oct_half(wv[o], e);
      if (x >= f) atomicAdd(&hitem[min(x - f, 4095u)], 1u);
    }
  __syncthreads();
  SKV_TS(ts, 3);
  fs_rank_bin(hitem, s.w[1], k);
  __syncthreads();
  const int bin = s.w[1].sel[0];
  if (__builtin_expect(bin == 4095, 0)) {
    res.ok = false;
    return res;
  }
  const uint32_t v = f + (uint32_t)bin;
  res.sel.v = v;
  res.sel.above = s.w[1].sel[1];
  const int need = k - res.sel.above, ties = (int)hitem[bin];
  if (RULE == TIE_VALUE) return res;
  uint32_t gt = 0, eq = 0;
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t x = oct_half(wv[o], e);
      gt |= (uint32_t)(x > v) << (8 * o + e);
      eq |= (uint32_t)(x == v) << (8 * o + e);
    }
  if (need >= ties) {
    res.mine = gt | eq;
    return res;
  }
  if (__builtin_expect(ties > FS_TIE_RANK, 0)) {
    res.ok = false;
    return res;
  }
  const int c = __popc(eq);
  const int slot0 = c ? atomicAdd(&s.w[1].ntie, c) : 0;
  int slot = slot0;
  for (uint32_t rest = eq; rest; rest &= rest - 1) s.tie[slot++] = id(__ffs(rest) - 1);
  __syncthreads();
  slot = slot0;
  for (uint32_t rest = eq; rest; rest &= rest - 1)  // rank = number of smaller tied IDs
    if (count_below(s.tie, ties, s.tie[slot++]) < need) gt |= rest & (0u - rest);
  res.mine = gt;
  return res;
}

// One octet per thread over the scratch's first histogram, cleared here: for
// the paths that run several selections over the same scratch.
template <TieRule RULE, typename IdFn>
__device__ __forceinline__ OctResult oct_select_clear(const uint4 w, int k, IdFn id, FastScratch& s) {
  __syncthreads();
  fs_clear(s.hist, s.w[0]);
  __syncthreads();
  const uint4 w1[1] = {w};
  return octn_select<1, RULE>(w1, k, id, s.hist, s.w[0], s);
}

}  // namespace skv
