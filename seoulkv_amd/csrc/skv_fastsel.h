// Exact block top-k by (ordered BF16 score desc, ID asc) from a sampled cut.
//
// 1. Sample: 4096 items (all of them when n <= 4096, else the items at
//    floor(j n / 4096)) are histogrammed in LDS (12-bit bins, then the low 4
//    bits of the chosen bin) to find a score `cut` that about
//    k + 4 sqrt(k) + 8 items are expected to reach (exactly the k-th best
//    score when the sample is the whole input).
// 2. Candidates: one pass over all n scores appends (score, position) of
//    every item scoring >= cut to an LDS list (one atomic per wave).  IDs are
//    read later, only for items tied at the k-th score.
// 3. If the list holds fewer than k items (the sample over-estimated the
//    cut) or overflows, the caller runs the full exact selection instead.
//    Otherwise the top k of the input are exactly the top k of the list
//    (every other item scores below cut <= every candidate), found by a
//    histogram over the candidates' scores and, for ties at the k-th score,
//    a rank of the tied IDs.
// The result is therefore identical to a full selection; only the time
// depends on the sample.
#pragma once

#include <cstddef>

#include "skv_select.h"

namespace skv {

constexpr int FS_SAMPLE = 4096;
constexpr int FS_PER = FS_SAMPLE / SEL_BLOCK;  // sample items per thread
constexpr int CAND_CAP = 4096;
constexpr int FS_TIE_RANK = SEL_BLOCK;  // ties ranked by direct comparison up to this count
constexpr int FS_OCT = 4;  // score octets per lane per pass (a 32-bit candidate mask)

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Packed 16-bit steps on both halves of a word.  Written as instructions: from
// vector code the compiler folds the saturating forms below into one compare
// and select per half.  (The tiled top-1600 of 40K keys 10.35 -> 9.85 us, of 60K
// 11.25 -> 10.25; the register selections' masks gained nothing from them and
// keep one compare per item.)
__device__ __forceinline__ uint32_t pk_sub_sat(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_min_u16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ uint32_t pk_dup(uint32_t x) { return x | (x << 16); }
constexpr uint32_t PK_ONE = 0x00010001u;

// Packed test of both halves of w against cut (cm1 = cut - 1 in each half):
// bit 0 = (low half >= cut), bit 16 = (high half >= cut).
__device__ __forceinline__ uint32_t ge_cut2(uint32_t w, uint32_t cm1) {
  return pk_min(pk_sub_sat(w, cm1), PK_ONE);
}

// Masks of an octet (4 words, 8 items): from bits 0 and 16 of word q to bits
// 2q and 2q + 1.
__device__ __forceinline__ uint32_t oct_bits(uint32_t m0, uint32_t m1, uint32_t m2, uint32_t m3) {
  const uint32_t m = m0 | (m1 << 2) | (m2 << 4) | (m3 << 6);
  return (m & 0x55u) | ((m >> 15) & 0xaau);
}
// Bit e: item e scores at least c (cm1 = c - 1 >= 0 in both halves).
__device__ __forceinline__ uint32_t oct_at_least(const u32x4& w, uint32_t cm1) {
  return oct_bits(ge_cut2(w[0], cm1), ge_cut2(w[1], cm1), ge_cut2(w[2], cm1), ge_cut2(w[3], cm1));
}
// Scratch of the register and sampled selections.  hist and hist_b, with
// their small words, let a kernel run two selections in a row with nothing
// cleared in between.
struct SelWords {
  uint32_t hist4[16];
  int sel[4];           // published by fs_rank_bin (0 .. 2) and tie_cut (3)
  int scan[SEL_WAVES];  // its wave totals
  int tie_scan[SEL_WAVES];
  int ntie;
};
struct FastScratch {
  union {
    uint32_t hist[4096];
    KthScratch k;
  };
  union {
    alignas(16) uint64_t cand[CAND_CAP];  // ord << 40 | position
    struct {
      alignas(16) uint32_t hist_b[4096];
      union {
        uint16_t tiles[4096];  // tiles listed by tiled_select
        alignas(16) uint32_t hist_c[4096];
      };
    };
  };
  alignas(16) uint32_t tie[FS_TIE_RANK];  // read as uint4 by count_below
  SelWords w[2];
  int ncand;
  int maxo;
};
static_assert(offsetof(FastScratch, cand) % 16 == 0, "cand is read 16 bytes at a time");
static_assert(offsetof(FastScratch, tie) % 16 == 0, "tie is read 16 bytes at a time");

// Clears a histogram (16-byte aligned) and its small words; a barrier must
// follow before they are used.
__device__ __forceinline__ void fs_clear(uint32_t* hist, SelWords& w) {
  static_assert(4096 == 4 * SEL_BLOCK, "one 16-byte store per thread");
  reinterpret_cast<uint4*>(hist)[threadIdx.x] = make_uint4(0, 0, 0, 0);
  if (threadIdx.x < 16) w.hist4[threadIdx.x] = 0;
  if (threadIdx.x == 0) w.ntie = 0;
}

// Candidate key: ordered score (bits 40..55) | position (bits 0..19); a key
// tied at the k-th score also carries its ID (bits 20..39, flag bit 56).
constexpr uint64_t CAND_HAS_ID = 1ull << 56;
__device__ __forceinline__ uint32_t cand_ord(uint64_t c) { return (uint32_t)(c >> 40) & 0xffffu; }
__device__ __forceinline__ int cand_pos(uint64_t c) { return (int)(c & 0xfffffu); }

// Number of the n entries of a smaller than x; a is a 16-byte aligned LDS
// array.  Four 16-byte reads are in flight per step (a dependent read per
// entry would leave the loop bound by LDS latency).
__device__ __forceinline__ int count_below(const uint32_t* a, int n, uint32_t x) {
  const uint4* a4 = reinterpret_cast<const uint4*>(a);
  const int n4 = n >> 2;
  int r0 = 0, r1 = 0, r2 = 0, r3 = 0, j = 0;
  auto c4 = [x](uint4 w) { return (int)(w.x < x) + (int)(w.y < x) + (int)(w.z < x) + (int)(w.w < x); };
  for (; j + 4 <= n4; j += 4) {
    const uint4 w0 = a4[j], w1 = a4[j + 1], w2 = a4[j + 2], w3 = a4[j + 3];
    r0 += c4(w0);
    r1 += c4(w1);
    r2 += c4(w2);
    r3 += c4(w3);
  }
  for (; j < n4; ++j) r0 += c4(a4[j]);
  for (int i = 4 * n4; i < n; ++i) r1 += a[i] < x;
  return (r0 + r1) + (r2 + r3);
}

struct FastResult {
  Selection sel;  // members: the candidates passing fs_member
  int ncand;      // candidates in FastScratch::cand
  bool ok;        // false: use the full selection
};

// Membership of candidate key c; id(position) is read only for a candidate
// tied at the cut score when not every tie is a member.
template <typename IdFn>
__device__ __forceinline__ bool fs_member(const FastResult& r, uint64_t c, IdFn id) {
  const uint32_t o = cand_ord(c);
  if (o == 0) return false;
  if (r.sel.all || o > r.sel.v) return true;
  if (o < r.sel.v) return false;
  if (r.sel.idcut == 0xffffffffu) return true;
  const uint32_t cid = (c & CAND_HAS_ID) ? (uint32_t)(c >> 20) & 0xfffffu : id(cand_pos(c));
  return cid <= r.sel.idcut;
}

// Score sources: at(i) = ordered score of item i; oct(o) = the 8 ordered
// scores of items 8o .. 8o+7 as packed 16-bit pairs.
struct RowScores {  // a 16-byte aligned row, readable to a multiple of 8 items
  static constexpr int PRE = 8;  // octets per thread fast_select loads at entry
  const uint16_t* __restrict__ row;
  __device__ uint32_t at(int i) const { return row[i]; }
  __device__ uint4 oct(int o) const { return reinterpret_cast<const uint4*>(row)[o]; }
};

struct MaskedScores {  // score[i] where gate[i] >= thr, else 0 (excluded)
  static constexpr int PRE = 4;
  const uint16_t* __restrict__ score;
  const uint16_t* __restrict__ gate;
  uint32_t thr;
  __device__ uint32_t at(int i) const {
    const uint32_t gv = gate[i], sv = score[i];  // both loads issued together
    return gv >= thr ? sv : 0u;
  }
  __device__ uint4 oct(int o) const {
    return pick4(reinterpret_cast<const uint4*>(score)[o], reinterpret_cast<const uint4*>(gate)[o],
                 thr);
  }
  // the 8 packed scores of s4 whose packed gates in g4 reach thr
  __device__ static uint4 pick4(uint4 s4, uint4 g4, uint32_t thr) {
    const uint32_t t16 = thr << 16;
    auto pick = [&](uint32_t sw, uint32_t gw) {
      return ((gw << 16) >= t16 ? (sw & 0xffffu) : 0u) | (gw >= t16 ? (sw & 0xffff0000u) : 0u);
    };
    return make_uint4(pick(s4.x, g4.x), pick(s4.y, g4.y), pick(s4.z, g4.z), pick(s4.w, g4.w));
  }
};


// Descending scan of a 4096-bin histogram (each thread owns 4 bins): the bin
// holding the rank-th largest value and the count in higher bins, in
// w.sel[0..1]; sel[0] = -1 if the histogram holds fewer than rank values.
// w.sel[2] = total count.  One barrier inside; the caller's next barrier
// publishes w.sel.
__device__ __forceinline__ void fs_rank_bin(const uint32_t* hist, SelWords& w, int rank) {
  constexpr int BPT = 4096 / SEL_BLOCK;  // bins per thread, scanned downwards
  static_assert(BPT == 4, "one 16-byte read per thread");
  const int lo = 4096 - BPT * ((int)threadIdx.x + 1);
  const uint4 a = *reinterpret_cast<const uint4*>(&hist[lo]);
  const int cv[BPT] = {(int)a.w, (int)a.z, (int)a.y, (int)a.x};
  const int c = (cv[0] + cv[1]) + (cv[2] + cv[3]);
  int total;
  const int exc = block_excl_scan(c, w.scan, &total);
  if (exc < rank && rank <= exc + c) {
    int acc = exc, bin = lo + BPT - 1;
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
      if (acc + cv[j] >= rank) { bin = lo + BPT - 1 - j; break; }
      acc += cv[j];
    }
    w.sel[0] = bin;
    w.sel[1] = acc;
  }
  if (threadIdx.x == 0) {
    w.sel[2] = total;
    if (total < rank) w.sel[0] = -1;
  }
}

// Digit (0..15) of the rank-th largest value in w.hist4, the count above it
// (acc in higher bins, then higher digits) and the count at it; every wave
// works it out for itself, so no barrier follows.
struct DigitRank {
  int digit, above, ties;
};
__device__ __forceinline__ DigitRank fs_rank_digit(const SelWords& w, int rank, int acc) {
  const int lane = threadIdx.x & 63;
  const int cnt = lane < 16 ? (int)w.hist4[15 - lane] : 0;
  const int inc = acc + row_incl_scan(cnt);
  const uint64_t hit = __ballot(lane < 16 && inc - cnt < rank && rank <= inc);
  const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
  return {15 - l, __builtin_amdgcn_readlane(inc - cnt, l), __builtin_amdgcn_readlane(cnt, l)};
}

// src: the n ordered scores (0 = excluded; see RowScores / MaskedScores).
// id(i): the item's ID (< 2^20), read only for candidates.  VALUE_ONLY: only
// sel.v (the k-th best score) is wanted: no IDs, no tie resolution.
// force_miss places the cut at the best sampled score (a test of the
// fallback: fewer than k candidates unless k ties share it).
// Sample u is item fs_sample_item(n, u).
__device__ __forceinline__ int fs_sample_item(int n, int u) {
  const int j = (int)threadIdx.x + u * SEL_BLOCK;
  return n <= FS_SAMPLE ? j : (int)(((uint64_t)j * (uint64_t)n) >> 12);
}

// Phase 1 of the sampled selection: from this thread's FS_PER sample scores
// sv (0 = excluded), the cut that about k + 4 sqrt(k) + 8 of n items reach
// (the rank-th best sample, rank scaled to the sample).  Returns cut >= 1 (1:
// every valid item).  hist and w are cleared (fs_clear and a barrier).
__device__ __forceinline__ uint32_t fs_cut(const uint32_t (&sv)[FS_PER], int n, int k,
                                           bool force_miss, uint32_t* hist, SelWords& w, int ts) {
#pragma unroll
  for (int u = 0; u < FS_PER; ++u)
    if (sv[u]) atomicAdd(&hist[sv[u] >> 4], 1u);
  __syncthreads();
  SKV_TS(ts, 1);
  int rank = k;
  if (n > FS_SAMPLE) {
    const float e = (float)k * (float)FS_SAMPLE / (float)n;
    rank = (int)ceilf(e + 4.f * sqrtf(e) + 8.f);
  }
  if (force_miss) rank = 1;
  fs_rank_bin(hist, w, rank);
  __syncthreads();
  const int b1 = w.sel[0];
  uint32_t cut = 1;  // every valid item
  if (b1 >= 0) {
    const int acc1 = w.sel[1];
#pragma unroll
    for (int u = 0; u < FS_PER; ++u)
      if (sv[u] && (int)(sv[u] >> 4) == b1) atomicAdd(&w.hist4[sv[u] & 15], 1u);
    __syncthreads();
    cut = ((uint32_t)b1 << 4) | (uint32_t)fs_rank_digit(w, rank, acc1).digit;
  }
  SKV_TS(ts, 2);
  return cut;
}

// Phases 3 on: the exact top-k among the candidates s.cand[0 .. s.ncand)
// (every item scoring >= cut; s.maxo their best score).
template <bool VALUE_ONLY, typename IdFn>
__device__ FastResult fs_finish(int k, IdFn id, FastScratch& s, uint32_t cut, int ts) {
  FastResult res;
  res.ok = true;
  res.ncand = 0;
  res.sel.idcut = 0xffffffffu;
  res.sel.all = false;
  res.sel.above = 0;
  SelWords& w = s.w[1];
  SKV_TS(ts, 3);
  const int nc = s.ncand;
  res.ncand = nc;
  if (nc > CAND_CAP || (cut > 1 && nc < k)) {
    res.ok = false;
    return res;
  }
  if (cut == 1 && nc <= k) {  // fewer valid items than k: all are members
    res.sel.all = true;
    res.sel.v = 0;
    res.sel.above = nc;
    return res;
  }
  SKV_TS(ts, 4);
  // ---- 3. exact k-th score among the candidates (nc >= k here)
  const uint32_t maxo = (uint32_t)s.maxo;
  int shift = 0;
  while (((maxo - cut) >> shift) >= 4096u) ++shift;
  fs_clear(s.hist, w);
  __syncthreads();
  for (int c = threadIdx.x; c < nc; c += SEL_BLOCK)
    atomicAdd(&s.hist[(cand_ord(s.cand[c]) - cut) >> shift], 1u);
  __syncthreads();
  fs_rank_bin(s.hist, w, k);
  __syncthreads();
  const int b2 = w.sel[0];
  int above = w.sel[1];
  // the IDs of the candidates in the k-th score's bin (the only possible
  // ties), loaded now so that they arrive while the score itself is found
  constexpr int CPT = CAND_CAP / SEL_BLOCK;  // candidates per thread
  uint32_t pid[CPT];
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int c = (int)threadIdx.x + u * SEL_BLOCK;
    pid[u] = 0u;
    if (!VALUE_ONLY && c < nc) {
      const uint64_t key = s.cand[c];
      if ((int)((cand_ord(key) - cut) >> shift) == b2) pid[u] = id(cand_pos(key));
    }
  }
  uint32_t v;
  int ties;
  if (shift == 0) {
    v = cut + (uint32_t)b2;
    ties = (int)s.hist[b2];
  } else {
    const uint32_t lowmask = (1u << shift) - 1u;
    for (int c = threadIdx.x; c < nc; c += SEL_BLOCK) {
      const uint32_t d = cand_ord(s.cand[c]) - cut;
      if ((int)(d >> shift) == b2) atomicAdd(&w.hist4[d & lowmask], 1u);
    }
    __syncthreads();
    const DigitRank r = fs_rank_digit(w, k, above);
    v = cut + (((uint32_t)b2 << shift) | (uint32_t)r.digit);
    above = r.above;
    ties = r.ties;
  }
  __syncthreads();
  res.sel.v = v;
  res.sel.above = above;
  SKV_TS(ts, 5);
  const int need = k - above;
  if (VALUE_ONLY || need >= ties) return res;  // every tie is a member

  // ---- ties at v: the `need` lowest IDs win (tied keys keep their ID for
  // fs_member)
  if (ties <= FS_TIE_RANK) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int c = (int)threadIdx.x + u * SEL_BLOCK;
      if (c >= nc) break;
      const uint64_t key = s.cand[c];
      if (cand_ord(key) == v) {
        s.tie[atomicAdd(&w.ntie, 1)] = pid[u];
        s.cand[c] = key | CAND_HAS_ID | ((uint64_t)pid[u] << 20);
      }
    }
    __syncthreads();
    if ((int)threadIdx.x < ties) {  // rank = number of smaller tied IDs
      const uint32_t x = s.tie[threadIdx.x];
      if (count_below(s.tie, ties, x) == need - 1) w.sel[2] = (int)x;
    }
    __syncthreads();
    res.sel.idcut = (uint32_t)w.sel[2];
    __syncthreads();
    return res;
  }
  auto val = [&](int c, uint64_t* out) {
    const uint64_t key = s.cand[c];
    if (cand_ord(key) != v) return false;
    *out = 0xfffffu - id(cand_pos(key));
    return true;
  };
  const uint64_t kth = block_kth<24>(nc, need, val, s.k);
  res.sel.idcut = 0xfffffu - (uint32_t)kth;
  return res;
}

template <bool VALUE_ONLY = false, typename Src, typename IdFn>
__device__ __forceinline__ FastResult fast_select(const Src& src, int n, int k, IdFn id, FastScratch& s,
                                                  bool force_miss = false, int ts = -1) {
  // ---- 1. sample
  uint32_t sv[FS_PER];
#pragma unroll
  for (int u = 0; u < FS_PER; ++u) {
    const int i = fs_sample_item(n, u);
    sv[u] = i >= n ? 0u : src.at(i);
  }
  // the candidate pass's first Src::PRE octets per thread, loaded now so that
  // they arrive while the cut is computed
  static_assert(Src::PRE % FS_OCT == 0, "prefetch whole passes");
  const int no = (n + 7) >> 3;
  uint4 pre[Src::PRE];
#pragma unroll
  for (int q = 0; q < Src::PRE; ++q) {
    const int o = (int)threadIdx.x + q * SEL_BLOCK;
    pre[q] = o < no ? src.oct(o) : make_uint4(0, 0, 0, 0);
  }
  __syncthreads();  // the scratch may have served another selection
  fs_clear(s.hist, s.w[0]);
  if (threadIdx.x == 0) {
    s.ncand = 0;
    s.maxo = 0;
  }
  __syncthreads();
  const uint32_t cut = fs_cut(sv, n, k, force_miss, s.hist, s.w[0], ts);

  // ---- 2. candidate positions: packed compares into a per-lane bit mask
  // (cut >= 1, so excluded items never pass), then one LDS append per set bit
  {
    const int lane = threadIdx.x & 63;
    const int base0 = threadIdx.x & ~63;
    const uint32_t cm1 = pk_dup(cut - 1);  // cut >= 1
    uint32_t mx = 0;
    auto pass = [&](const uint4 (&w)[FS_OCT], int base) {
      uint32_t mask = 0;
#pragma unroll
      for (int r = 0; r < FS_OCT; ++r) {
        // bit 2e: low half of word e >= cut; bit 2e + 1: high half
        const uint32_t m = ge_cut2(w[r].x, cm1) | (ge_cut2(w[r].y, cm1) << 2) |
                           (ge_cut2(w[r].z, cm1) << 4) | (ge_cut2(w[r].w, cm1) << 6);
        uint32_t m8 = (m & 0x55u) | ((m >> 15) & 0xaau);
        const int valid = n - 8 * (base + r * SEL_BLOCK + lane);
        if (valid < 8) m8 &= valid > 0 ? (1u << valid) - 1u : 0u;
        mask |= m8 << (8 * r);
      }
      const int cnt = __popc(mask);
      const int inc = wave_incl_scan(cnt);
      int wbase = 0;
      if (lane == 63) wbase = atomicAdd(&s.ncand, inc);
      wbase = __builtin_amdgcn_readlane(wbase, 63);
      int slot = wbase + inc - cnt;
#pragma unroll
      for (int r = 0; r < FS_OCT; ++r) {  // compile-time octet: no indexed arrays
        uint32_t m8 = (mask >> (8 * r)) & 0xffu;
        const u32x4 wv = {w[r].x, w[r].y, w[r].z, w[r].w};
        const int pos0 = 8 * (base + r * SEL_BLOCK + lane);
        while (m8) {
          const int e = __ffs(m8) - 1;
          m8 &= m8 - 1;
          const uint32_t word = wv[e >> 1];
          const uint32_t o = (e & 1) ? word >> 16 : word & 0xffffu;
          mx = max(mx, o);
          if (slot < CAND_CAP) s.cand[slot] = ((uint64_t)o << 40) | (uint64_t)(pos0 + e);
          ++slot;
        }
      }
    };
    // passes over the octets loaded at entry, then over the rest
#pragma unroll
    for (int p = 0; p < Src::PRE / FS_OCT; ++p) {
      const int base = base0 + p * FS_OCT * SEL_BLOCK;
      if (base >= no) break;  // wave-uniform
      const uint4 w[FS_OCT] = {pre[FS_OCT * p], pre[FS_OCT * p + 1], pre[FS_OCT * p + 2],
                               pre[FS_OCT * p + 3]};
      pass(w, base);
    }
    for (int base = base0 + Src::PRE * SEL_BLOCK; base < no; base += FS_OCT * SEL_BLOCK) {
      uint4 w[FS_OCT];
#pragma unroll
      for (int r = 0; r < FS_OCT; ++r) {
        const int o = base + r * SEL_BLOCK + lane;
        w[r] = o < no ? src.oct(o) : make_uint4(0, 0, 0, 0);
      }
      pass(w, base);
    }
    mx = (uint32_t)wave_max((int)mx);
    if (lane == 0) atomicMax(&s.maxo, (int)mx);
  }
  __syncthreads();
  return fs_finish<VALUE_ONLY>(k, id, s, cut, ts);
}

// 16-item tiles of a 16-byte aligned row of ordered scores.
struct RowTiles {
  const uint16_t* __restrict__ row;
  __device__ void tile(int t, uint4 (&w)[2]) const {
    const uint4* r4 = reinterpret_cast<const uint4*>(row) + 2 * t;
    w[0] = r4[0];
    w[1] = r4[1];
  }
};
// 16-item tiles of MaskedScores (score where gate >= thr, else excluded).
struct MaskedTiles {
  const uint16_t* __restrict__ score;
  const uint16_t* __restrict__ gate;
  uint32_t thr;
  __device__ void tile(int t, uint4 (&w)[2]) const {
    const uint4* s4 = reinterpret_cast<const uint4*>(score) + 2 * t;
    const uint4* g4 = reinterpret_cast<const uint4*>(gate) + 2 * t;
    const uint4 s0 = s4[0], s1 = s4[1], g0 = g4[0], g1 = g4[1];
    w[0] = MaskedScores::pick4(s0, g0, thr);
    w[1] = MaskedScores::pick4(s1, g1, thr);
  }
};

// The need-th smallest ID of the `ties` (<= FS_TIE_RANK) items whose
// positions s.tie holds (written before a barrier); s.tie holds their IDs on
// return.  One ID load per tie, all in flight together (an owner reading its
// own ties one after another waited for each: +1.8 us at 80 ties), and one
// comparison rank per tie.
template <typename IdFn>
__device__ __forceinline__ uint32_t tie_cut(int ties, int need, IdFn id, FastScratch& s,
                                            SelWords& w) {
  uint32_t x = 0;
  if ((int)threadIdx.x < ties) {
    x = id((int)s.tie[threadIdx.x]);
    s.tie[threadIdx.x] = x;
  }
  __syncthreads();
  // IDs are distinct, so one thread has the rank
  if ((int)threadIdx.x < ties && count_below(s.tie, ties, x) == need - 1) w.sel[3] = (int)x;
  __syncthreads();
  return (uint32_t)w.sel[3];
}

// Exact top-k of n (FS_SAMPLE < n <= 64 x SEL_BLOCK) ordered scores whose
// producer also wrote an upper bound of every 16-item tile (tmx, e.g. the
// tile's max): from this thread's fast_select sample sv the same cut as
// fast_select, then only the tiles whose bound reaches the cut are read, one
// tile per thread and round, and stay in registers: their items at or above
// the cut are counted by distance above it (4096 bins of one score step), so
// the k-th score is a bin, and every thread forms its tiles' member masks
// from its registers (emit(tile, 16-bit mask), once per tile with members).
// No candidate list is written or read (12.7 -> 10.8 us for the top-1600 of
// 40K keys).  id(position): an item's ID, read for items tied at the k-th
// score only.  A k-th score 4095 or more steps above the cut (scores on both
// sides of zero) takes two more passes over the registers, and more than
// FS_TIE_RANK ties at it are cut by a digit count of their IDs, so neither
// needs another selection (top-1600 of 20K keys, 1650 of them above zero 25.8
// -> 18.8 us, 2500 of them tied 32.3 -> 20.6 us against selecting again; both
// branches are marked unlikely: pools without them keep 9.9-10.0 us).  Returns false, with nothing emitted, when the
// sample's cut missed (fewer than k items reach it): the caller runs another
// selection.  The scratch is cleared by tiled_clear and a barrier.
__device__ __forceinline__ void tiled_clear(FastScratch& s) {
  fs_clear(s.hist, s.w[0]);
  fs_clear(s.hist_b, s.w[1]);
}

template <typename TileSrc, typename IdFn, typename EmitFn>
__device__ __forceinline__ bool tiled_select(const TileSrc& src, const uint16_t* __restrict__ tmx,
                                             const uint32_t (&sv)[FS_PER], int n, int k, IdFn id,
                                             FastScratch& s, bool force_miss, int ts, EmitFn emit) {
  // ---- 1. this thread's 4 tile bounds (loaded with the caller's sample)
  const int ntile = (n + 15) >> 4;
  const int t4 = 4 * (int)threadIdx.x;
  const uint2 tm = t4 < ntile ? *reinterpret_cast<const uint2*>(tmx + t4) : make_uint2(0, 0);
  const uint32_t cut = fs_cut(sv, n, k, force_miss, s.hist, s.w[0], ts);
  // ---- 2. the tiles whose max reaches the cut, listed
  const uint32_t tv[4] = {tm.x & 0xffffu, tm.x >> 16, tm.y & 0xffffu, tm.y >> 16};
  uint32_t hot = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) hot |= (uint32_t)(t4 + e < ntile && tv[e] >= cut) << e;
  int nhot;
  int at = block_excl_scan(__popc(hot), s.w[0].tie_scan, &nhot);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if ((hot >> e) & 1u) s.tiles[at++] = (uint16_t)(t4 + e);
  __syncthreads();
  SKV_TS(ts, 7);
  // ---- 3. the items at or above the cut.  The tiles of every round (at most
  // TL_ROUNDS: the caller bounds the row to 4 x SEL_BLOCK tiles) are loaded
  // before the first is scanned, so the rounds share one memory latency;
  // the loads are branch-free (an unlisted slot reloads tile 0, unused).
  constexpr int TL_ROUNDS = 4;
  int tl[TL_ROUNDS];
  u32x4 tw[TL_ROUNDS][2];
#pragma unroll
  for (int r = 0; r < TL_ROUNDS; ++r) {
    const int i = r * SEL_BLOCK + (int)threadIdx.x;
    tl[r] = i < nhot ? (int)s.tiles[i] : -1;
  }
#pragma unroll
  for (int r = 0; r < TL_ROUNDS; ++r) {
    uint4 w2[2];
    src.tile(max(tl[r], 0), w2);
#pragma unroll
    for (int q = 0; q < 2; ++q) tw[r][q] = u32x4{w2[q].x, w2[q].y, w2[q].z, w2[q].w};
  }
  // bit e: item e of the tile scores at least c (c >= 1)
  auto at_least = [&](int r, uint32_t c) {
    const uint32_t cm1 = pk_dup(c - 1);
    return oct_at_least(tw[r][0], cm1) | (oct_at_least(tw[r][1], cm1) << 8);
  };
  uint32_t cand[TL_ROUNDS];  // the tiles' items at or above the cut
  // f(score) of the items of round r in mask
  auto scores_in = [&](int r, uint32_t mask, auto f) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {  // compile-time octet: no indexed arrays
      uint32_t m8 = (mask >> (8 * q)) & 0xffu;
      while (m8) {
        const int e = __ffs(m8) - 1;
        m8 &= m8 - 1;
        const uint32_t word = tw[r][q][e >> 1];
        f((e & 1) ? word >> 16 : word & 0xffffu);
      }
    }
  };
#pragma unroll
  for (int r = 0; r < TL_ROUNDS; ++r) {
    cand[r] = 0;
    if (r * SEL_BLOCK >= nhot) continue;  // block-uniform
    uint32_t mask = at_least(r, cut);
    if (tl[r] < 0) mask = 0;
    else if (n - 16 * tl[r] < 16) mask &= (1u << (n - 16 * tl[r])) - 1u;
    cand[r] = mask;
    scores_in(r, mask, [&](uint32_t o) { atomicAdd(&s.hist_b[min(o - cut, 4095u)], 1u); });
  }
  __syncthreads();
  SKV_TS(ts, 8);
  fs_rank_bin(s.hist_b, s.w[1], k);
  __syncthreads();
  SKV_TS(ts, 5);
  const int bin = s.w[1].sel[0];
  uint32_t v = 1;   // members: above v, and `need` of those at v (all, when
  int need = 0;     // fewer than k items are valid)
  int ties = 0;
  if (bin < 0) {
    if (cut > 1) return false;  // the cut missed
  } else if (__builtin_expect(bin < 4095, 1)) {
    v = cut + (uint32_t)bin;
    need = k - s.w[1].sel[1];
    ties = (int)s.hist_b[bin];
  } else {  // the k best lie above the last step: 12 bits, then 4 (as octn_select)
    SelWords& w = s.w[0];
    fs_clear(s.hist, w);  // last read before the barriers since the cut
    __syncthreads();
#pragma unroll
    for (int r = 0; r < TL_ROUNDS; ++r)
      scores_in(r, cand[r], [&](uint32_t o) {
        if (o - cut >= 4095u) atomicAdd(&s.hist[o >> 4], 1u);
      });
    __syncthreads();
    fs_rank_bin(s.hist, w, k);
    __syncthreads();
    const uint32_t b = (uint32_t)w.sel[0];
    const int acc = w.sel[1];
#pragma unroll
    for (int r = 0; r < TL_ROUNDS; ++r)
      scores_in(r, cand[r], [&](uint32_t o) {
        if (o - cut >= 4095u && o >> 4 == b) atomicAdd(&w.hist4[o & 15], 1u);
      });
    __syncthreads();
    const DigitRank d = fs_rank_digit(w, k, acc);
    v = (b << 4) | (uint32_t)d.digit;
    need = k - d.above;
    ties = d.ties;
  }
  const bool rank = bin >= 0 && need < ties;  // only some of the ties are members
  uint32_t mem[TL_ROUNDS], eq[TL_ROUNDS];
  int neq = 0;
#pragma unroll
  for (int r = 0; r < TL_ROUNDS; ++r) {
    mem[r] = eq[r] = 0;
    if (r * SEL_BLOCK >= nhot) continue;  // block-uniform
    mem[r] = at_least(r, v) & cand[r];
    if (rank) {
      // v <= 0xffff; a score never exceeds it, so nothing lies above 0xffff
      const uint32_t gt = v < 0xffffu ? at_least(r, v + 1) & cand[r] : 0u;
      eq[r] = mem[r] & ~gt;
      mem[r] = gt;
      neq += __popc(eq[r]);
    }
  }
  if (__builtin_expect(rank && ties > FS_TIE_RANK, 0)) {
    // too many to compare: the need-th lowest ID (< 2^20) by its upper 12 and
    // lower 8 bits, counted from the largest complement
    SelWords& w = s.w[0];
    uint32_t found = 0;
    int left = need;
#pragma unroll 1
    for (int low = 0; low < 2; ++low) {
      __syncthreads();  // (second pass: every thread has read the first's counts)
      fs_clear(s.hist, w);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < TL_ROUNDS; ++r)
        for (uint32_t rest = eq[r]; rest; rest &= rest - 1) {
          const uint32_t c = 0xfffffu - id(16 * tl[r] + __ffs(rest) - 1);
          if (!low) atomicAdd(&s.hist[c >> 8], 1u);
          else if (c >> 8 == found) atomicAdd(&s.hist[c & 255u], 1u);
        }
      __syncthreads();
      fs_rank_bin(s.hist, w, left);
      __syncthreads();
      found = (found << 8) | (uint32_t)w.sel[0];
      left -= w.sel[1];
    }
    const uint32_t idcut = 0xfffffu - found;
#pragma unroll
    for (int r = 0; r < TL_ROUNDS; ++r)
      for (uint32_t rest = eq[r]; rest; rest &= rest - 1)
        if (id(16 * tl[r] + __ffs(rest) - 1) <= idcut) mem[r] |= rest & (0u - rest);
  } else if (rank) {  // the `need` lowest IDs among the ties win
    const int slot0 = neq ? atomicAdd(&s.w[1].ntie, neq) : 0;
    int slot = slot0;
#pragma unroll
    for (int r = 0; r < TL_ROUNDS; ++r)
      for (uint32_t rest = eq[r]; rest; rest &= rest - 1)
        s.tie[slot++] = (uint32_t)(16 * tl[r] + __ffs(rest) - 1);
    __syncthreads();
    const uint32_t idcut = tie_cut(ties, need, id, s, s.w[1]);
    slot = slot0;
#pragma unroll
    for (int r = 0; r < TL_ROUNDS; ++r)
      for (uint32_t rest = eq[r]; rest; rest &= rest - 1)
        if (s.tie[slot++] <= idcut) mem[r] |= rest & (0u - rest);
  }
  SKV_TS(ts, 6);
#pragma unroll
  for (int r = 0; r < TL_ROUNDS; ++r)
    if (mem[r]) emit(tl[r], mem[r]);
  return true;
}

}  // namespace skv
