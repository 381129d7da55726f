// Dense FP8 decode over every key of the cache (interface in skv_dense.h).
//
// k_dense: block (b, g) covers an even share of KV group g's pairs of 16-key
// tiles.  Per tile, one wave scores its 16 keys for the group's 4 query heads
// with two FP8 matrix-core steps (16 x 16 x 128): the A operand is the K half
// of the records as stored, the B operand holds each head's BF16 query split
// into four FP8 terms (column 4h + s carries term s, weight 2^-4s), so the
// products are those of the BF16 query and the FP8 keys.  The V half is
// summed by BF16 matrix-core steps over the pair's 32 keys in FP32, the
// probabilities split exactly into three BF16 terms (dn_pair).  Waves and
// blocks are merged by the usual max/sum rescaling; k_dense_merge folds the
// per-block partials of each query head into the BF16 output.
#include <mutex>

#include "../../include/seoulkv4_hip.h"
#include "skv_dense.h"
#include "skv_device.h"

namespace skv {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr float DN_LOG2E = 1.4426950408889634f;
// A row's running max moves only when a logit exceeds it by more than this
// (log2 units), so the accumulators are rescaled rarely; p <= 2^DN_TAU.
constexpr float DN_TAU = 8.f;

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ uint32_t f32_fp8_byte(float x) {
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x, 0.f, 0, false) & 0xffu;
}
__device__ __forceinline__ float fp8_byte_f32(uint32_t b) {
  typedef float v2f __attribute__((ext_vector_type(2)));
  const v2f f = __builtin_amdgcn_cvt_pk_f32_fp8((int)b, false);
  return f[0];
}

// B operand image of the score step, [m][lane][i]: lane l (column c = l % 16
// = 4h + s, key block kb = l / 16) takes word i of MFMA m, dims
// dn_dim(m, i, kb) + [0, 4).  Term s of head h is FP8(r_s) with
// r_0 = q_h * 2^E_h and r_{s+1} = (r_s - FP8(r_s)) * 16, where 2^E_h scales
// max|q_h| into [128, 256).  Returned: zc = 2^(-4s - E_h) * log2(e) / 16,
// which turns the column's dot product into its share of the logit in log2
// units.  Each wave forms its share of the words: split over the block's
// waves (every wave formed the whole image before, ~1500 vector
// instructions, which was most of a short context's kernel).
constexpr int DN_QWAVES = 8;  // waves that form the image, one word of each MFMA's 8 each
static_assert(DN_WAVES >= DN_QWAVES, "the query's image is formed by the first 8 waves");
typedef uint32_t DenseImage[2][WAVE][8];

__device__ __forceinline__ int dn_dim(int m, int i, int kb) {
  return m * 128 + (i >> 2) * 64 + kb * 16 + (i & 3) * 4;
}

// The query words a wave needs, loaded ahead of the first tiles: 16 elements
// of head lane / 16 (for the maxima), and the 4 elements of each of its two
// image words.
struct DenseQuery {
  uint4 mx[2];
  uint2 w[2];
};

__device__ __forceinline__ DenseQuery dense_query_load(const uint16_t* __restrict__ qg, int lane,
                                                       int wave) {
  const uint4* row = reinterpret_cast<const uint4*>(qg + (lane >> 4) * D + 16 * (lane & 15));
  const uint16_t* qh = qg + ((lane & 15) >> 2) * D;
  DenseQuery q;
  q.mx[0] = row[0];
  q.mx[1] = row[1];
#pragma unroll
  for (int m = 0; m < 2; ++m)
    q.w[m] = *reinterpret_cast<const uint2*>(qh + dn_dim(m, wave & 7, lane >> 4));
  return q;
}

__device__ __forceinline__ float dense_query_form(const DenseQuery& q, int lane, int wave,
                                                  DenseImage& img) {
  const int col = lane & 15, h = col >> 2, s = col & 3;
  const uint32_t mw[8] = {q.mx[0].x, q.mx[0].y, q.mx[0].z, q.mx[0].w,
                          q.mx[1].x, q.mx[1].y, q.mx[1].z, q.mx[1].w};
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    mx = fmaxf(mx, fmaxf(fabsf(bf16_f32(mw[i] & 0xffffu)), fabsf(bf16_f32(mw[i] >> 16))));
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  mx = __shfl(mx, 16 * h);
  int E = 0;
  if (mx > 0.f) {
    int e;
    (void)frexpf(mx, &e);
    E = 8 - e;
  }
  if (wave < DN_QWAVES) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      uint32_t word = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t pair = j < 2 ? q.w[m].x : q.w[m].y;
        float x = ldexpf(bf16_f32((j & 1) ? pair >> 16 : pair & 0xffffu), E);
        uint32_t t = f32_fp8_byte(x);
#pragma unroll
        for (int r = 1; r < 4; ++r) {  // term r, kept by the lanes with s >= r
          x = (x - fp8_byte_f32(t)) * 16.f;
          const uint32_t u = f32_fp8_byte(x);
          t = r <= s ? u : t;
        }
        word |= t << (8 * j);
      }
      img[m][lane][wave] = word;
    }
  }
  return ldexpf(DN_LOG2E / 16.f, -4 * s - E);
}

// Two 16-key tiles of a wave.  k: A operand of the score step, for key row
// l % 16 of tile a the K bytes 64 j + 16 kb + [0, 16) (an instruction reads
// whole 64-byte runs; the dims' order is dn_dim's); v: V dims 16c..16c+15 of
// keys 4kb + r of tile a.
struct DnPair {
  uint4 k[2][4], v[2][4];
};

// V is read with streaming loads: a row's 256 bytes are used by one
// instruction, once.  (K rows come in 64-byte runs, two instructions per
// cache line, and lose more than they gain: T = 2^20 347 us with neither
// streamed, 330 K, 311 V, 324 both; T = 131072 49.9, 53.1, 48.1, 53.0.)
__device__ __forceinline__ uint4 load_stream(const uint8_t* p) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const u4 v = __builtin_nontemporal_load(reinterpret_cast<const u4*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

// tile0, tile1: the records of the tiles' first keys.  TAIL: the context's
// last pair when it is not whole; last0, last1: the index of the last key in
// reach from the tiles' first (rows past it read that key, masked later).
template <bool TAIL>
__device__ __forceinline__ void dn_load_k(DnPair& x, const uint8_t* __restrict__ tile0,
                                          const uint8_t* __restrict__ tile1, int last0, int last1,
                                          int lane) {
  const int row = lane & 15, kb = lane >> 4;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const uint8_t* kr = (a ? tile1 : tile0) + 256;
    const int ko = (TAIL ? min(row, a ? last1 : last0) : row) * 512 + kb * 16;
#pragma unroll
    for (int j = 0; j < 4; ++j) x.k[a][j] = *reinterpret_cast<const uint4*>(kr + ko + 64 * j);
  }
}
template <bool TAIL>
__device__ __forceinline__ void dn_load_v(DnPair& x, const uint8_t* __restrict__ tile0,
                                          const uint8_t* __restrict__ tile1, int last0, int last1,
                                          int lane) {
  const int row = lane & 15, kb = lane >> 4;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const uint8_t* vr = a ? tile1 : tile0;
    const int vo = 4 * kb * 512 + 16 * row;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      x.v[a][r] = load_stream(
          vr + (TAIL ? min(4 * kb + r, a ? last1 : last0) * 512 + 16 * row : vo + 512 * r));
  }
}

__device__ __forceinline__ v8i as_v8i(uint4 a, uint4 b) {
  return v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, (int)b.z, (int)b.w};
}

// The high halves of two words, b's in the low half: two BF16 values.
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(a, b, 0x07060302u);
}

// Two FP8 bytes of w (bytes 0, 1 or 2, 3) as two BF16 values (exact).
template <bool HI>
__device__ __forceinline__ int fp8_bf16x2(uint32_t w) {
  return __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w, 1.f, HI));
}

// The 32 keys t0 .. of a pair: scores, online softmax, P V sums.
//
// P V runs on the matrix cores as 16 products [16 dims x 32 keys][32 keys x
// 16 columns]: product i has dim 16c + i of lane l = 16 kb + c as its row c,
// so the lane's own V bytes (8 keys x 16 dims), transposed 4 x 4 in
// registers and widened to BF16 (exact), are its row operand, and the
// column operand of lane (kb, 4h + s) is made from the scores that the lane
// itself holds (head h, the same 8 keys): no value moves between lanes.  A
// probability enters as three BF16 terms (8 + 8 + 8 significant bits) in the
// columns s = 0, 1, 2 (s = 3: zero), exactly down to 2^-110, where the third
// term's last bit reaches BF16's smallest step (2^-133); the epilogue adds the
// columns.  (exp2 is the bare instruction: a p below 2^-126 is 0.)  The
// products are exact and summed in FP32.  m is the running max of head h over
// all the wave's keys (it moves by more than DN_TAU or not at all), l the sum
// over this lane's keys.
template <bool TAIL, typename NextK>
__device__ __forceinline__ void dn_pair(DnPair& x, int t0, int T, int lane, const DenseImage& img,
                                        float zc, v4f (&o)[16], float& m, float& l, NextK next_k) {
  const int kb = lane >> 4, s = lane & 3;
  // the query operand, read from LDS for every pair: held in registers it
  // would leave too few for the pair in flight
  int at = lane;
  asm volatile("" : "+v"(at));
  v8i bq[2];
#pragma unroll
  for (int mm = 0; mm < 2; ++mm) {
    const uint4* w = reinterpret_cast<const uint4*>(&img[mm][at][0]);
    bq[mm] = as_v8i(w[0], w[1]);
  }
  float z[8];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
      acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
          as_v8i(x.k[a][2 * mm], x.k[a][2 * mm + 1]), bq[mm], acc, 0, 0, 0, 0, 0, 0);
    // logits (log2 units) of keys t0 + 16 a + 4kb + r for head h: the four
    // split columns of a head are adjacent lanes
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = acc[r] * zc;
      v += dpp_f<0xB1>(v);  // quad_perm [1,0,3,2]
      v += dpp_f<0x4E>(v);  // quad_perm [2,3,0,1]
      z[4 * a + r] = v;
    }
  }
  next_k();
  if (TAIL) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (t0 + 16 * (e >> 2) + 4 * kb + (e & 3) >= T) z[e] = -INFINITY;
  }
  float tm = z[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) tm = fmaxf(tm, z[e]);
  if (__ballot(tm > m + DN_TAU)) {
    tm = fmaxf(tm, __shfl_xor(tm, 16));
    tm = fmaxf(tm, __shfl_xor(tm, 32));
    const bool grow = tm > m + DN_TAU;
    const float mn = grow ? tm : m;
    const float al = grow ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
    l *= al;
    m = mn;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[i][j] *= al;
  }
  float p[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {  // (a masked key: 0, also while m = -inf)
    const float x = __builtin_amdgcn_exp2f(z[e] - m);
    p[e] = z[e] == -INFINITY ? 0.f : x;
  }
  l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
  // this column's term of every p (selected by bit masks: no branches)
  const uint32_t m0 = s == 0 ? ~0u : 0u, m1 = s == 1 ? ~0u : 0u, m2 = s == 2 ? ~0u : 0u;
  uint32_t t[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float r1 = p[e] - __uint_as_float(__float_as_uint(p[e]) & 0xffff0000u);
    const float r2 = r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
    t[e] = (__float_as_uint(p[e]) & m0) | (__float_as_uint(r1) & m1) | (__float_as_uint(r2) & m2);
  }
  const v4i pb = {(int)high_halves(t[1], t[0]), (int)high_halves(t[3], t[2]),
                  (int)high_halves(t[5], t[4]), (int)high_halves(t[7], t[6])};
#pragma unroll
  for (int w = 0; w < 4; ++w) {  // dims 16c + 4w .. + 3
    uint32_t d[2][4];  // d[a][i]: the 4 keys' bytes of dim 4w + i
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const uint32_t y[4] = {(&x.v[a][0].x)[w], (&x.v[a][1].x)[w], (&x.v[a][2].x)[w],
                             (&x.v[a][3].x)[w]};
      const uint32_t lo01 = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u);
      const uint32_t hi01 = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u);
      const uint32_t lo23 = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
      const uint32_t hi23 = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
      d[a][0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
      d[a][1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
      d[a][2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
      d[a][3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4i va = {fp8_bf16x2<false>(d[0][i]), fp8_bf16x2<true>(d[0][i]),
                      fp8_bf16x2<false>(d[1][i]), fp8_bf16x2<true>(d[1][i])};
      o[4 * w + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(v8bf, va), __builtin_bit_cast(v8bf, pb), o[4 * w + i], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);  // one word's operands live at a time
  }
}

// The partials: [G][nb][H] rows of 256 unnormalised outputs, then as many
// (max in log2 units, sum) pairs.
__device__ __forceinline__ float2* dense_stats(float* part, int nb) {
  return reinterpret_cast<float2*>(part + (size_t)G * nb * H * D);
}

// PAGED: the records are read through the page table (table, shift).
//
// Bound by the record stream: 12 waves per CU (168 registers each), every
// wave with one pair in registers whose K half is reloaded after the scores
// and whose V half after the sums, so other waves' loads are in flight while
// one computes.  (A double-buffered pair in 8 waves of 256 registers, or
// three pairs in 4 waves of 512, spilled.)  Whole call with the merge, back
// to back, against V sums on the vector ALUs (half of every SIMD's cycles)
// with the query formed by every wave: T = 1000 16.6 -> 8.5 us, 40009 27 ->
// 18, 131072 51-55 -> 45-47 (43 without the merge), 2^20 374 -> 310
// (6.9 TB/s), with the reload below.
// The arguments are DenseArgs' fields as scalars, preloaded at dispatch: the
// first loads need not wait for an argument block.
template <bool PAGED>
__global__ __launch_bounds__(DN_BLOCK) void k_dense(const uint16_t* q, const uint8_t* kv8,
                                                    const int* table, float* part, int T, int rows,
                                                    int nb, int share, int extra, int shift) {
  const int g = blockIdx.y, b = blockIdx.x;
  // (scalar wave index: the tile addresses and loop bounds stay in scalar registers)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  const uint8_t* __restrict__ kv = kv8 + (size_t)g * rows * 512;
  __shared__ float s_o[DN_WAVES][H][D];
  __shared__ float s_m[DN_WAVES][H], s_l[DN_WAVES][H];
  __shared__ __align__(16) DenseImage s_q;

  // pair i of wave w of block b is pair b + nb (w + DN_WAVES i) of the
  // context: the blocks sweep one front through the records together, so at
  // any time the reads spread over all memory channels (T = 2^20: 357 us with
  // a contiguous share per block, whose starts lie a power of two apart, 346
  // with the common front)
  const int mine = share + (b < extra ? 1 : 0);
  const int n = wave < mine ? (mine - wave + DN_WAVES - 1) / DN_WAVES : 0;
  auto key0 = [&](int i) { return (b + nb * (wave + DN_WAVES * i)) * 2 * DN_TILE; };
  // the first key of the second tile of pair i, moved back into the context
  // when the tile lies past it (its scores are masked by the true position)
  auto key1 = [&](int i) { return min(key0(i) + DN_TILE, (T - 1) & ~(DN_TILE - 1)); };
  const DenseQuery qw = dense_query_load(q + (size_t)g * H * D, lane, wave);
  // paged: lane i holds the record index of the first key of either tile of
  // the wave's pair i (a wave has at most DN_PAGED_MAX_PAIRS pairs: T <=
  // 2^20); loaded before the query is formed, so the first tile loads need
  // not wait for the table
  static_assert(DN_PAGED_MAX_PAIRS == WAVE, "one pair per lane");
  uint32_t prow[2] = {0u, 0u};
  if (PAGED && lane < n) {
    prow[0] = kv_row_paged(table, shift, g, key0(lane));
    prow[1] = kv_row_paged(table, shift, g, key1(lane));
  }
  // a page holds a power-of-two number (>= DN_TILE) of consecutive tokens, so
  // the 16 keys of an aligned tile are consecutive records of one page
  auto tile0 = [&](int i) {
    return PAGED ? kv8 + (size_t)__builtin_amdgcn_readlane(prow[0], i) * 512
                 : kv + (size_t)key0(i) * 512;
  };
  auto tile1 = [&](int i) {
    return PAGED ? kv8 + (size_t)__builtin_amdgcn_readlane(prow[1], i) * 512
                 : kv + (size_t)key1(i) * 512;
  };
  // the wave's whole pairs; its last one may be the context's ragged end
  const bool ragged = n > 0 && key0(n - 1) + 2 * DN_TILE > T;
  const int whole = n - (ragged ? 1 : 0);
  auto load_k = [&](DnPair& x, int i) {
    dn_load_k<false>(x, tile0(i), tile1(i), 0, 0, lane);
  };
  auto load_v = [&](DnPair& x, int i) {
    dn_load_v<false>(x, tile0(i), tile1(i), 0, 0, lane);
  };
  DnPair x;
  if (whole > 0) {
    load_k(x, 0);
    load_v(x, 0);
  }

  const float zc = dense_query_form(qw, lane, wave, s_q);
  __syncthreads();

  v4f o[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // running max / this lane's sum of head col / 4

  // each half of the pair's registers is reloaded once it is used; the other
  // waves of the CU cover the rest of the latency.  No reload after the last
  // pair: reading it again instead of branching fetched its streamed V half
  // from memory once more, 290 MB for 268 MB at T = 131072, where a wave has
  // 5.3 pairs (24577 keys 17.0 -> 14.6 us, 40009 20.3 -> 18.2, 131072 44.4 ->
  // 43.3, 2^20 the same; with the branch on V alone 15.2, 19.5, 43.1).
#pragma nounroll
  for (int i = 0; i < whole; ++i) {
    dn_pair<false>(x, key0(i), T, lane, s_q, zc, o, m, l, [&] {
      if (i + 1 < whole) load_k(x, i + 1);
    });
    if (i + 1 < whole) load_v(x, i + 1);
  }
  if (ragged) {
    const int i = n - 1;
    dn_load_k<true>(x, tile0(i), tile1(i), T - 1 - key0(i), T - 1 - key1(i), lane);
    dn_load_v<true>(x, tile0(i), tile1(i), T - 1 - key0(i), T - 1 - key1(i), lane);
    dn_pair<true>(x, key0(i), T, lane, s_q, zc, o, m, l, [] {});
  }

  // the wave's partial: l over its four key blocks, o over the three columns
  // of a head; o[i][j] of lane (kb, 4h + s) is dim 16 (4kb + j) + i, and the
  // lane stores the dims of j = s
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  const int h = col >> 2, s = col & 3;
  const uint32_t ms[4] = {s == 0 ? ~0u : 0u, s == 1 ? ~0u : 0u, s == 2 ? ~0u : 0u, s == 3 ? ~0u : 0u};
  float os[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    uint32_t mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v = o[i][j] + dpp_f<0xB1>(o[i][j]);
      v += dpp_f<0x4E>(v);
      mine |= __float_as_uint(v) & ms[j];
    }
    os[i] = __uint_as_float(mine);
  }
#pragma unroll
  for (int i = 0; i < 16; i += 4)
    *reinterpret_cast<float4*>(&s_o[wave][h][16 * (4 * kb + s) + i]) =
        make_float4(os[i], os[i + 1], os[i + 2], os[i + 3]);
  if (kb == 0 && s == 0) {
    s_m[wave][h] = m;
    s_l[wave][h] = l;
  }
  __syncthreads();
  // the block's partial, waves merged in wave order: 2 dims per thread
  static_assert(DN_BLOCK >= H * D / 2, "one pass of the block covers the partial");
  if (threadIdx.x < H * D / 2) {
    const int hh = threadIdx.x / (D / 2), d = 2 * (threadIdx.x % (D / 2));
    float Mb = -INFINITY;
#pragma unroll
    for (int w = 0; w < DN_WAVES; ++w) Mb = fmaxf(Mb, s_m[w][hh]);
    float2 O = make_float2(0.f, 0.f);
    float Lb = 0.f;
#pragma unroll
    for (int w = 0; w < DN_WAVES; ++w) {
      const float fx = __builtin_amdgcn_exp2f(s_m[w][hh] - Mb);
      const float fw = s_m[w][hh] == -INFINITY ? 0.f : fx;
      const float2 ow = *reinterpret_cast<const float2*>(&s_o[w][hh][d]);
      O.x = fmaf(fw, ow.x, O.x);
      O.y = fmaf(fw, ow.y, O.y);
      Lb = fmaf(fw, s_l[w][hh], Lb);
    }
    const size_t row = ((size_t)g * nb + b) * H + hh;
    *reinterpret_cast<float2*>(part + row * D + d) = O;
    if (d == 0) dense_stats(part, nb)[row] = make_float2(Mb, Lb);
  }
}

// Query head j = blockIdx.x, dims 32 * blockIdx.y + [0, 32): thread (slice s,
// 4 dims) loads partials s, s + 32, ... (at most DN_MERGE_PER, all in flight
// together), the block agrees on their max, and the slices are added in order.
constexpr int DN_MERGE_PER = (DN_TARGET_BLOCKS + 31) / 32;
constexpr int DN_MERGE_DIMS = D / DN_MERGE_SLICES;
static_assert(DN_MERGE_DIMS == 32, "8 threads of 4 dims per slice");

__global__ __launch_bounds__(256) void k_dense_merge(const float* part, int nb, uint16_t* out) {
  const int j = blockIdx.x, g = j / H, h = j % H;
  const int dl = threadIdx.x & 7, sl = threadIdx.x >> 3;
  const int d = blockIdx.y * DN_MERGE_DIMS + 4 * dl;
  const size_t first = (size_t)g * nb * H + h;
  const float2* __restrict__ stats = dense_stats(const_cast<float*>(part), nb);
  __shared__ float s_max[256 / WAVE];
  __shared__ float4 s_o[32][8];
  __shared__ float s_l[32];
  float2 ml[DN_MERGE_PER];
  float4 po[DN_MERGE_PER];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < DN_MERGE_PER; ++i) {
    const int b = sl + 32 * i;
    ml[i] = make_float2(-INFINITY, 0.f);
    po[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (b < nb) {
      const size_t row = first + (size_t)b * H;
      ml[i] = stats[row];
      po[i] = *reinterpret_cast<const float4*>(part + row * D + d);
    }
    mx = fmaxf(mx, ml[i].x);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = mx;
  __syncthreads();
  float M = s_max[0];
#pragma unroll
  for (int w = 1; w < 256 / WAVE; ++w) M = fmaxf(M, s_max[w]);
  float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
  float L = 0.f;
#pragma unroll
  for (int i = 0; i < DN_MERGE_PER; ++i) {
    const float fx = __builtin_amdgcn_exp2f(ml[i].x - M);
    const float f = ml[i].x == -INFINITY ? 0.f : fx;
    O.x = fmaf(f, po[i].x, O.x);
    O.y = fmaf(f, po[i].y, O.y);
    O.z = fmaf(f, po[i].z, O.z);
    O.w = fmaf(f, po[i].w, O.w);
    L = fmaf(f, ml[i].y, L);
  }
  s_o[sl][dl] = O;
  if (dl == 0) s_l[sl] = L;
  __syncthreads();
  if (threadIdx.x < DN_MERGE_DIMS) {
    const float* so = reinterpret_cast<const float*>(s_o);
    float Ot = 0.f, Lt = 0.f;
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      Ot += so[s * DN_MERGE_DIMS + threadIdx.x];
      Lt += s_l[s];
    }
    out[j * D + blockIdx.y * DN_MERGE_DIMS + threadIdx.x] = (uint16_t)bf16_rne(Ot / Lt);
  }
}

}  // namespace

void launch_dense(const DenseArgs& a, hipStream_t st, int k) {
  if (k == 0)
    hipLaunchKernelGGL(a.table ? k_dense<true> : k_dense<false>, dim3(a.nb, G), dim3(DN_BLOCK), 0,
                       st, a.q, a.kv8, a.table, a.part, a.T, a.rows, a.nb, a.share, a.extra,
                       a.shift);
  else
    hipLaunchKernelGGL(k_dense_merge, dim3(G * H, DN_MERGE_SLICES), dim3(256), 0, st,
                       (const float*)a.part, a.nb, a.out);
}

// ------------------------------------------------ allocation-free dense decode
// The partials of skv_dense_decode_static: one file-scope device array per
// GPU, [G][DN_TARGET_BLOCKS][H][D + 2] FP32 (1 MiB), enough for every context
// up to 2^20 keys (dense_split never gives more than DN_TARGET_BLOCKS blocks
// per group).  Host code never names it in a launch: the device address comes
// from hipGetSymbolAddress, once per device, with that device current.
constexpr size_t DN_SCRATCH_FLOATS = (size_t)G * DN_TARGET_BLOCKS * H * (D + 2);
static __device__ __align__(256) float scratch[DN_SCRATCH_FLOATS];

namespace {

constexpr int DN_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[DN_MAX_DEVICES] = {};

// The calling thread's current device's copy of `scratch` (looked up on the
// first call on that device); NULL with *err set on failure.
float* device_scratch(int* device, hipError_t* err) {
  *err = hipGetDevice(device);
  if (*err != hipSuccess) return nullptr;
  if (*device < 0 || *device >= DN_MAX_DEVICES) {
    *err = hipErrorInvalidDevice;
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[*device]) {
    void* ptr = nullptr;
    *err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (*err != hipSuccess) return nullptr;
    g_scratch_ptr[*device] = static_cast<float*>(ptr);
  }
  return g_scratch_ptr[*device];
}

}  // namespace

}  // namespace skv

extern "C" int skv_dense_decode_static(const void* kv8, int rows, int T, const void* q_dev,
                                       void* out_dev, void* stream) {
  using namespace skv;
  if (!kv8 || !q_dev || !out_dev) return note_call_error(SKV_EINVAL, "NULL records, query or output");
  if (T < 1 || T > (1 << 20))
    return note_call_error(SKV_EINVAL, "context %d outside [1, 2^20] (the static partials hold "
                           "%d blocks per group)", T, DN_TARGET_BLOCKS);
  if (rows < T) return note_call_error(SKV_EINVAL, "rows %d < context %d", rows, T);
  int device = 0;
  hipError_t e = hipSuccess;
  float* part = device_scratch(&device, &e);
  if (!part)
    return note_call_error(SKV_EHIP, "device scratch lookup failed: %s", hipGetErrorString(e));
  // every operand must be device memory of the current device large enough
  // for what the kernels touch (a wrong size or a host pointer is refused
  // here rather than faulting in a kernel)
  const struct { const void* ptr; uint64_t bytes; const char* name; } operands[] = {
      {kv8, (uint64_t)G * rows * 512, "records"},
      {q_dev, 16 * D * 2, "query"},
      {out_dev, 16 * D * 2, "output"}};
  for (const auto& op : operands)
    if (const char* why = device_range_error(op.ptr, op.bytes, device))
      return note_call_error(SKV_EINVAL, "%s (%llu bytes) %s", op.name,
                             (unsigned long long)op.bytes, why);
  (void)hipGetLastError();  // a launch error below is this call's, not an earlier one's
  DenseArgs a{};
  a.kv8 = static_cast<const uint8_t*>(kv8);
  a.q = static_cast<const uint16_t*>(q_dev);
  a.T = T;
  a.rows = rows;
  dense_split(T, a.nb, a.share, a.extra);
  if (a.nb > DN_TARGET_BLOCKS)  // never for T <= 2^20
    return note_call_error(SKV_EINVAL, "context %d needs %d partials per group", T, a.nb);
  a.part = part;
  a.out = static_cast<uint16_t*>(out_dev);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  launch_dense(a, st, 0);
  launch_dense(a, st, 1);
  e = hipGetLastError();
  if (e != hipSuccess) return note_call_error(SKV_EHIP, "dense launch failed: %s", hipGetErrorString(e));
  return SKV_OK;
}
