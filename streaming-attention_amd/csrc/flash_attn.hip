// Causal attention over pairs of contiguous rows, without coreset items: one kernel, three weights of
// a pair (query row i, key j):
//   FLASH_SOFTMAX  exact causal softmax attention, the FlashAttention-style baseline of the reference's GPU
//                  module (_flash_causal_kernel, triton_article_attention.py:372-435;
//                  triton_flash_causal_attention :580-637):
//                  out_i = sum_{j<=i} exp(s q_i.k_j - m_i) v_j / max(sum_{j<=i} exp(s q_i.k_j - m_i), 1e-20),
//                  m_i a running row maximum (online softmax)
//   FLASH_EXP      compressor "none" (fast_article_attention.py:437-464, :596-598), where the Taylor part and the
//                  residual add up to exp itself: out_i = sum_{j<=i} exp(s q_i.k_j) v_j / max(sum, eps)
//   FLASH_TAYLOR   the Taylor part (degree <= 3; fast_article_attention.py:184-285): the partial sums
//                  low_num_i = sum_{j < c(i)} exp_{<=t}(s q_i.k_j) v_j and low_den_i in sta_moments' layout, c(i) the
//                  start of the row's chunk, for sta_block_attention.  A pair costs 2 d + 2 (dv + 1) flop and a
//                  token's moments 4 F (dv + 1) for F features, so the pairs are the cheaper way up to a length that
//                  grows with F: about 5000 tokens at d = dv = 64, degree 2, 20000 at 128, 100000 at 64, degree 3.
//                  A tile's key batches can be dealt out to several workgroups (FlashArgs::nsplit).
// fp32 accumulation, no N x N score matrix.
//
// Matrix-core layout (v_mfma_f32_16x16x32): X^T = K Q^T with A = key rows staged in LDS and B = the wave's
// query rows in registers; the weights P^T stay in the accumulator layout and are the B operand of
// num^T += V^T P^T.  A lane holds one query row (li) and, per 16-key subtile, four keys 4 lg + r; its
// accumulators hold value columns 16 ct + 4 lg + r of the same row.  k-step m of lane group lg covers
// dimensions 32 m + 8 lg + j; the V^T rows hold each pair of 16-key subtiles in contraction order
// (flash_key_pos), so every operand is one 16-byte LDS read.
//
// Products.  gfx950's 16-bit matrix cores run 16x the fp32 rate, so fp32 operands are carried as three bf16
// planes, x = h + m + l (8 bits each, together the 24 of fp32), and a product as the six largest plane
// products (hh, hm, mh, mm, hl, lh): the three left out are at most 2^-23 |x x'| together, and in the sums
// their signs are random (measured against 64 bits the results are closer than with fp32 matrix
// instructions, 4.4e-7 against 5.1e-7 at 8191 keys).  2500 / 6 = 417 TF/s against their 157 TF/s.
// 16-bit inputs are taken as they are (exact products, fp32 sums); their fp32 weights are carried as
// 16-bit planes: hi + lo for the softmax (within 2^-16 P for bf16, 2^-20 P for fp16), three bf16 planes for
// FLASH_EXP, whose fp16 values are two bf16 planes (exact: 11 bits).  Rows that three planes cannot hold
// (infinities, values above 3.396e38, values whose lower planes are subnormal) go through fp32 matrix instructions
// after all, found by their sums: 8 x 8191 fp32 with every seventh key switched off by a dimension of finfo.min
// 1.61 ms (0.92 ms in fp32 instructions alone), the check itself 0 to 0.7 us a call.
//
// What bounds it: fp32 rows the six products (two thirds of the time at d = dv = 64), 16-bit rows the VALU
// work of a pair (exponential, maximum, planes: 6 instructions).  8 heads x 8191 fp32, d = dv = 64: 413 us,
// 351 us = 196 TF/s with three workgroups a tile (fp32 matrix instructions, unbalanced tiles: 858 us); 32 x 65536 fp32:
// 83.4 ms = 211 TF/s, matrix cores 58 % busy; 2 x 16 x 8192 bf16: 467 us = 589 TF/s (710 us with a rescale and 12
// more VALU instructions a pair); FLASH_EXP 4 x 8 x 2048 fp32: 102 us (515 us as moment scan + residual kernel in
// fp32 products); with few tiles, FlashArgs::nsplit workgroups share one: 1 x 8192 fp32 394 -> 73 us, 4 x 8192 bf16
// 180 -> 88.  FLASH_TAYLOR 8 x 16 x 4096 bf16: 0.51 ms (matrix cores 54 % busy) in the place of the moment scan's 1.1.
#include <type_traits>

#include "common.hpp"

namespace sta {

enum FlashWeight : int { FLASH_SOFTMAX = 0, FLASH_EXP = 1, FLASH_TAYLOR = 2 };

struct FlashArgs {
  const void* q;
  const void* k;
  const void* v;
  int dtype;
  int64_t n;
  int d;
  int dv;
  int ldqk;      // row stride (elements) of q and k: a multiple of 4, >= d (columns >= d are ignored)
  int ldv;       // row stride of v: a multiple of 4, >= dv
  float scale2;  // softmax scale times log2(e); FLASH_TAYLOR: the scale
  int n_tiles;   // ceil((n + shift) / FLASH_ROWS)
  int64_t bh;
  float floor;   // smallest denominator
  void* out;     // [BH][n][dv], dense
  int out_dtype;
  int vec_out;  // fp32 output, dv % 4 == 0 and 16-byte aligned: 16-byte stores
  // key batches of a tile are dealt out to nsplit workgroups, each with sums of its own.  FLASH_TAYLOR: partials
  // (below).  The others, nsplit > 1: raw sums low_num [nsplit][BH][n][low_ld] and {denominator, row maximum}
  // low_den [nsplit][BH][n][2], which flash_combine_kernel adds up and normalises
  int nsplit;
  // FLASH_TAYLOR: coefficients of x, x^2, x^3 (the logit, or q.k of 16-bit rows), the row chunk and its offset
  // (c(i) = floor((i + shift) / chunk) chunk - shift; row tiles start at -shift), the partials
  float c1, c2, c3;
  int chunk, shift;
  float* low_num;  // [BH][nsplit][low_rows][low_ld], row i at low_off + i
  float* low_den;  // [BH][nsplit][low_rows]
  int64_t low_rows;
  int low_ld, low_off;
  // 1: row strides so long that a batch's offsets leave the 1 GiB buffers: every row takes the fp32 products; 2: the
  // softmax of 16-bit rows so, which FLASH_EXP's kernel takes (the 16-bit softmax has no fp32 products of its own)
  int direct;
};

constexpr int FLASH_ROWS = 128;  // query rows of a workgroup: 4 waves x 2 strips of 16

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

// Planes of the key / query rows, of the weights and of the values, and keys per LDS stage.
// FLASH_TAYLOR carries fp32 operands as two planes, as the moment scan does, and the weights as three: they are
// near 1, so that two planes' error is 2^-17 of every value (2 x 8 x 3000 fp16 segment means: 4.0e-6 from
// 64 bits in the whole result, against 3.5e-6 with the scan).
__host__ __device__ constexpr int flash_kp(int in, int w) { return in != F32 ? 1 : (w == FLASH_TAYLOR ? 2 : 3); }
__host__ __device__ constexpr int flash_pp(int in, int w) {
  return (in == F32 || w != FLASH_SOFTMAX) ? 3 : 2;
}
__host__ __device__ constexpr int flash_vp(int in, int w) {
  return in == F32 ? flash_kp(in, w) : (in == F16 && w != FLASH_SOFTMAX ? 2 : 1);
}
__host__ __device__ constexpr int flash_dps(int dp) { return dp < 32 ? 32 : dp; }
__host__ __device__ constexpr int flash_stage_bytes(int dp, int dvt, int in, int w, int kb) {
  return 2 * (flash_kp(in, w) * kb * (flash_dps(dp) + 8) + flash_vp(in, w) * dvt * 16 * (kb + 8));
}
__host__ __device__ constexpr int flash_kb(int dp, int dvt, int in, int w) {
  return flash_stage_bytes(dp, dvt, in, w, 64) > 120 * 1024 ? 32 : 64;
}
// Two stages (the next batch is written while this one is read, one barrier a batch) where four workgroups'
// stages fit a compute unit's 160 KiB; one stage (two barriers) otherwise.
__host__ __device__ constexpr int flash_stages(int dp, int dvt, int in, int w) {
  return flash_stage_bytes(dp, dvt, in, w, flash_kb(dp, dvt, in, w)) <= 20 * 1024 ? 2 : 1;
}
// waves per SIMD by the per-wave register arrays (query planes, accumulators, logits, staged units)
__host__ __device__ constexpr int flash_occupancy(int dp, int dvt, int in, int w) {
  const int kb = flash_kb(dp, dvt, in, w);
  const int unit = in == F32 ? 4 : 2;
  const int regs = flash_kp(in, w) * 2 * flash_dps(dp) / 8 + 2 * dvt * 4 + 2 * (kb / 16) * 4 +
                   unit * ((kb * dp / 4 + 255) / 256 + 4 * ((kb / 4 * dvt * 4 + 255) / 256));
  return regs <= (in == F32 && w == FLASH_EXP ? 112 : 100) ? 3 : (regs <= 176 ? 2 : 1);
}

__host__ __device__ constexpr int flash_key_pos(int r) {
  return 32 * (r >> 5) + 8 * ((r >> 2) & 3) + 4 * ((r >> 4) & 1) + (r & 3);
}

template <bool F16M>
__device__ __forceinline__ floatx4 mfma16(const uint4& a, const uint4& b, floatx4 c) {
  if constexpr (F16M)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c,
                                                  0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

// x - (the 16-bit value in half `hi` of p), exact where the half is the rounding of x
template <bool F16M>
__device__ __forceinline__ void sub_pair(uint32_t p, float& a, float& b) {
  if constexpr (F16M) {
    a -= static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(p & 0xffffu)));
    b -= static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(p >> 16)));
  } else {
    uint32_t c0 = 0x0000BF80u, c1 = 0xBF800000u;  // bf16 pairs (-1, 0), (0, -1); see split_pair
    asm("" : "+s"(c0));
    asm("" : "+s"(c1));
    const bf16x2 hp = __builtin_bit_cast(bf16x2, p);
    a = __builtin_amdgcn_fdot2_f32_bf16(hp, __builtin_bit_cast(bf16x2, c0), a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(hp, __builtin_bit_cast(bf16x2, c1), b, false);
  }
}

// two fp32 values as NP packed 16-bit planes (bf16: each plane rounded to nearest even; fp16: toward zero)
template <int NP, bool F16M>
__device__ __forceinline__ void plane_pair(float a, float b, uint32_t (&p)[NP]) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if constexpr (F16M)
      p[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
    else
      p[i] = pk_bf16(a, b);
    if (i + 1 < NP) sub_pair<F16M>(p[i], a, b);
  }
}

// Elements of a 4-element unit starting at column c that lie in [0, width), the rest zero (a select,
// so padding that holds non-finite bits cannot leak in).
template <int ES>
__device__ __forceinline__ uint4 unit_clip(uint4 u, int valid) {
  if constexpr (ES == 4)
    return uint4{valid > 0 ? u.x : 0u, valid > 1 ? u.y : 0u, valid > 2 ? u.z : 0u, valid > 3 ? u.w : 0u};
  else
    return uint4{u.x & (valid > 1 ? 0xffffffffu : (valid > 0 ? 0xffffu : 0u)),
                 u.y & (valid > 3 ? 0xffffffffu : (valid > 2 ? 0xffffu : 0u)), 0u, 0u};
}

// Buffer resource of `bytes` bytes at p: loads beyond it return zero (at most 1 GiB: a batch needs
// a few tens of KiB, and the offset that marks absent units lies behind it).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t flash_rsrc(const void* p, int64_t bytes) {
  const int64_t b = bytes < 0 ? 0 : (bytes > 0x40000000 ? 0x40000000 : bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(b), 0x00020000);
}
template <int ES>
__device__ __forceinline__ uint4 load_buf(__amdgpu_buffer_rsrc_t r, int off) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  if constexpr (ES == 4) {
    const u4 x = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    return uint4{x.x, x.y, x.z, x.w};
  } else {
    const u2 x = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    return uint4{x.x, x.y, 0u, 0u};
  }
}

// Which tile a workgroup takes.  Long tiles first (the last rows have the most keys); the workgroups of one
// XCD (w % 8) share heads when the heads divide by 8.  When about two workgroups fit a compute unit at a
// time the first two rounds are all there is, and plain descending order would give compute unit c the
// c-th longest of both rounds (1.5x the mean for the first): the second round therefore ascends.
__device__ __forceinline__ void flash_tile(const FlashArgs& a, int64_t& bh, int& t, int& split) {
  const int total = gridDim.x, nbh = static_cast<int>(a.bh);
  const bool xcd = (nbh & 7) == 0;
  const int hx = (xcd ? nbh >> 3 : nbh) * a.nsplit;  // (head, split)s of this group of workgroups
  const int j = xcd ? blockIdx.x >> 3 : blockIdx.x;
  const int count = xcd ? total >> 3 : total, round = xcd ? 32 : 256;
  int rank = j;
  if (j >= round && j < 2 * round) {
    const int m = (count < 2 * round ? count : 2 * round) - round;
    if (j - round < m) rank = round + (m - 1 - (j - round));
  }
  const int step = rank / hx, hs = rank - step * hx, h = hs / a.nsplit;
  split = hs - h * a.nsplit;
  t = a.n_tiles - 1 - step;
  bh = xcd ? (blockIdx.x & 7) * (nbh >> 3) + h : h;
}

// One workgroup per (head, tile of FLASH_ROWS query rows); wave w owns 2 strips of 16 rows.  Keys [0, last row
// of the tile] are staged KB at a time (K row-major, V transposed), the next batch's rows loaded into
// registers while the current one computes.  A wave skips batches that lie wholly after its rows and
// applies the causal mask only on batches that straddle them.
template <int DP, int DVT, int IN, int W>
__global__ __launch_bounds__(256, flash_occupancy(DP, DVT, IN, W)) void flash_attn_kernel(const FlashArgs a) {
  constexpr int ES = IN == F32 ? 4 : 2;
  constexpr int RS = 2;
  constexpr int KB = flash_kb(DP, DVT, IN, W);
  constexpr int NSUB = KB / 16;
  constexpr int DPS = flash_dps(DP);  // dimensions in whole 32-element steps
  constexpr int MS = DPS / 32;
  constexpr int KP = flash_kp(IN, W), PP = flash_pp(IN, W), VP = flash_vp(IN, W);
  constexpr int XORD = KP - 1;  // plane products (i, j) with i + j <= order are taken
  constexpr int PORD = (PP > VP ? PP : VP) - 1;
  constexpr bool KF16 = IN == F16, PF16 = IN == F16 && W == FLASH_SOFTMAX;
  // denominators: a column of ones on the matrix cores where the weights' planes keep fp32 accuracy and the
  // matrix cores have room (16-bit inputs; FLASH_TAYLOR of every type, so that 16-bit rows and their fp32
  // values give the same sums), else fp32 VALU sums
  constexpr bool DENM = (IN != F32 || W == FLASH_TAYLOR) && PP == 3;
  // how far (log2) a row may exceed its running maximum before the sums are rescaled; two-plane weights keep
  // the latest maximum, whose own weight 1 is then exact (bf16, 32 heads x 8192: error against 64 bits 1.9e-6
  // and 479 us, with 8 here 2.1e-6 and 450 us)
  constexpr float GROW = PP == 3 ? 8.f : 0.f;
  constexpr int LDK = DPS + 8;      // 16-bit elements per key row: 16 (2 j + 1) bytes
  constexpr int DV = DVT * 16;
  constexpr int LDV = KB + 8;
  constexpr int KPL = KB * LDK, VPL = DV * LDV;  // elements of a plane
  constexpr int STAGE = KP * KPL + VP * VPL;
  constexpr int NST = flash_stages(DP, DVT, IN, W);
  constexpr int KU = DP / 4, VU = DV / 4, KG = KB / 4;
  constexpr int KPT = (KB * KU + 255) / 256, VPT = (KG * VU + 255) / 256;
  __shared__ uint4 stage4[(NST * STAGE + 7) / 8];
  uint16_t* const stage = reinterpret_cast<uint16_t*>(stage4);

  constexpr bool TAYLOR = W == FLASH_TAYLOR;
  int64_t bh;
  int t, split;
  flash_tile(a, bh, t, split);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int n = static_cast<int>(a.n);
  const int r0 = t * FLASH_ROWS - (TAYLOR ? a.shift : 0);
  const int64_t qkbase = bh * a.n * a.ldqk;
  const int64_t vbase = bh * a.n * a.ldv;

  // keys of a row: all up to its own, or those before its chunk
  auto limit = [&](int row) -> int {
    if constexpr (!TAYLOR) return row + 1;
    const int c = (row + a.shift) / a.chunk * a.chunk - a.shift;  // row + shift >= 0
    return c > 0 ? c : 0;
  };

  // the wave's query rows as B operands (8 dimensions per lane and k-step), columns >= d zero.  fp32 rows
  // are scaled before they are split; 16-bit rows keep their exact values and the logits are scaled
  // instead, by |scale| (its sign moves to the queries, so that the largest product is the largest logit;
  // FLASH_TAYLOR's coefficients hold the scale).
  int myrow[RS], lim[RS];  // the row's keys are [0, lim)
  bool rvalid[RS];
  uint4 qB[RS][MS][KP];
  const uint32_t flip = (!TAYLOR && IN != F32 && a.scale2 < 0.f) ? 0x80008000u : 0u;
  const float sc = IN == F32 ? 1.f : (a.scale2 < 0.f ? -a.scale2 : a.scale2);
#pragma unroll
  for (int rs = 0; rs < RS; ++rs) {
    myrow[rs] = r0 + (wave * RS + rs) * 16 + li;
    lim[rs] = limit(myrow[rs]);
    rvalid[rs] = (!TAYLOR || myrow[rs] >= 0) && myrow[rs] < n;
    const int64_t qoff = qkbase + static_cast<int64_t>(rvalid[rs] ? myrow[rs] : 0) * a.ldqk;
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      uint32_t w[KP][4];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int col = 32 * m + 8 * lg + 4 * hh;
        const uint4 raw = unit_clip<ES>(load_unit<ES>(a.q, qoff + min(col, a.ldqk - 4)), rvalid[rs] ? a.d - col : 0);
        if constexpr (IN == F32) {
          const floatx4 f = unit_to_f4<4>(raw, F32, a.scale2);
          uint32_t p[KP];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            plane_pair<KP, false>(f[2 * e], f[2 * e + 1], p);
#pragma unroll
            for (int i = 0; i < KP; ++i) w[i][2 * hh + e] = p[i];
          }
        } else {
          w[0][2 * hh] = raw.x ^ flip;
          w[0][2 * hh + 1] = raw.y ^ flip;
        }
      }
#pragma unroll
      for (int i = 0; i < KP; ++i) qB[rs][m][i] = uint4{w[i][0], w[i][1], w[i][2], w[i][3]};
    }
  }
  const int wlim_lo = limit(r0 + wave * RS * 16), wlim_hi = limit(r0 + wave * RS * 16 + RS * 16 - 1);

  floatx4 num[RS][DVT], dacc[RS];
  float den[RS], mrow[RS];
#pragma unroll
  for (int rs = 0; rs < RS; ++rs) {
    den[rs] = 0.f;
    dacc[rs] = floatx4{0.f, 0.f, 0.f, 0.f};
    mrow[rs] = -1e30f;  // finite: exp2(m_old - m_new) is then 0 or 1, never a NaN
#pragma unroll
    for (int ct = 0; ct < DVT; ++ct) num[rs][ct] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t one2 = PF16 ? 0x3c003c00u : 0x3f803f80u;
  const uint4 ones = uint4{one2, one2, one2, one2};

  auto process = [&](auto diag_tag, int off, const uint16_t* Kst, const uint16_t* Vst) {
    constexpr bool DIAG = decltype(diag_tag)::value;
    floatx4 X[NSUB][RS];
#pragma unroll
    for (int kt = 0; kt < NSUB; ++kt)
#pragma unroll
      for (int rs = 0; rs < RS; ++rs) X[kt][rs] = floatx4{0.f, 0.f, 0.f, 0.f};
    // two key subtiles at a time: 2 RS independent chains of products cover the matrix-core latency
#pragma unroll
    for (int kp = 0; kp < NSUB; kp += 2)
#pragma unroll
      for (int m = 0; m < MS; ++m) {
        uint4 kv[2][KP];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < KP; ++i)
            kv[h][i] = *reinterpret_cast<const uint4*>(Kst + i * KPL + (16 * (kp + h) + li) * LDK + 32 * m + 8 * lg);
#pragma unroll
        for (int o = XORD; o >= 0; --o)  // smallest products first
#pragma unroll
          for (int i = 0; i <= o; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int rs = 0; rs < RS; ++rs)
                if (i < KP && o - i < KP) X[kp + h][rs] = mfma16<KF16>(kv[h][i], qB[rs][m][o - i], X[kp + h][rs]);
      }
    if constexpr (W == FLASH_SOFTMAX) {
      // The weights are relative to a row maximum that is replaced (and the sums rescaled) only when some
      // row of the wave exceeds its own by more than GROW.  Lanes compare their own keys, so a batch that
      // changes no maximum has no cross-lane step.
      bool grow = false;
      float mx[RS];
#pragma unroll
      for (int rs = 0; rs < RS; ++rs) {
        float m0 = -__builtin_huge_valf(), m1 = -__builtin_huge_valf();
#pragma unroll
        for (int kt = 0; kt < NSUB; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x = X[kt][rs][r];
            if constexpr (DIAG) {
              if (off + 16 * kt + 4 * lg + r >= lim[rs]) x = -__builtin_huge_valf();
            }
            float& mm = (r & 1) ? m1 : m0;
            mm = __builtin_amdgcn_fmed3f(mm, x, __builtin_huge_valf());  // max, without quieting its inputs
          }
        mx[rs] = __builtin_amdgcn_fmed3f(m0, m1, __builtin_huge_valf()) * sc;
        grow = grow || mx[rs] > mrow[rs] + GROW;
      }
      if (__any(grow)) {
#pragma unroll
        for (int rs = 0; rs < RS; ++rs) {
          float m0 = fmaxf(mrow[rs], mx[rs]);
          m0 = fmaxf(m0, __shfl_xor(m0, 16));
          m0 = fmaxf(m0, __shfl_xor(m0, 32));
          const float alpha = __builtin_amdgcn_exp2f(mrow[rs] - m0);
          mrow[rs] = m0;
          if constexpr (DENM) dacc[rs] *= alpha;
          den[rs] *= alpha;
#pragma unroll
          for (int ct = 0; ct < DVT; ++ct) num[rs][ct] *= alpha;
        }
      }
    }
#pragma unroll
    for (int sp = 0; sp < NSUB / 2; ++sp) {
      uint4 pB[RS][PP];
#pragma unroll
      for (int rs = 0; rs < RS; ++rs) {
        uint32_t w[PP][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float p[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int kt = 2 * sp + (e >> 1), r = 2 * (e & 1) + h;
            const float x = X[kt][rs][r];
            float y;
            if constexpr (W == FLASH_SOFTMAX)
              y = IN == F32 ? x - mrow[rs] : fmaf(x, sc, -mrow[rs]);
            else
              y = IN == F32 ? x : x * sc;
            p[h] = TAYLOR ? fmaf(x, fmaf(x, fmaf(x, a.c3, a.c2), a.c1), 1.f) : __builtin_amdgcn_exp2f(y);
            if constexpr (DIAG) {
              if (off + 16 * kt + 4 * lg + r >= lim[rs]) p[h] = 0.f;
            }
            if constexpr (!DENM) den[rs] += p[h];
          }
          uint32_t pl[PP];
          plane_pair<PP, PF16>(p[0], p[1], pl);
#pragma unroll
          for (int i = 0; i < PP; ++i) w[i][e] = pl[i];
        }
#pragma unroll
        for (int i = 0; i < PP; ++i) pB[rs][i] = uint4{w[i][0], w[i][1], w[i][2], w[i][3]};
      }
      if constexpr (DENM) {
#pragma unroll
        for (int i = PP - 1; i >= 0; --i)
#pragma unroll
          for (int rs = 0; rs < RS; ++rs) dacc[rs] = mfma16<PF16>(ones, pB[rs][i], dacc[rs]);
      }
      constexpr int CG = DVT % 2 == 0 ? 2 : 1;  // value columns in pairs, as the key subtiles above
#pragma unroll
      for (int cp = 0; cp < DVT; cp += CG) {
        uint4 vv[CG][VP];
#pragma unroll
        for (int h = 0; h < CG; ++h)
#pragma unroll
          for (int i = 0; i < VP; ++i)
            vv[h][i] = *reinterpret_cast<const uint4*>(Vst + i * VPL + (16 * (cp + h) + li) * LDV + 32 * sp + 8 * lg);
#pragma unroll
        for (int o = PORD; o >= 0; --o)
#pragma unroll
          for (int i = 0; i <= o; ++i)
#pragma unroll
            for (int h = 0; h < CG; ++h)
#pragma unroll
              for (int rs = 0; rs < RS; ++rs)
                if (i < VP && o - i < PP)
                  num[rs][cp + h] = mfma16<PF16>(vv[h][i], pB[rs][o - i], num[rs][cp + h]);
      }
    }
  };

  const int row_hi = (r0 + FLASH_ROWS < n ? r0 + FLASH_ROWS : n) - 1;  // r0 < n: t < ceil(n / FLASH_ROWS)
  const int kend = limit(row_hi);
  const int step = a.nsplit;  // this workgroup's batches: split, split + step, ...
  const int nb_all = (kend + KB - 1) / KB;
  const int nb_own = (nb_all - split + step - 1) / step;
  constexpr bool FP32_ROWS = !TAYLOR && (IN == F32 || W == FLASH_EXP);  // has fp32 products of its own (below)
  const int nb = FP32_ROWS && a.direct ? 0 : nb_own;
  auto offset = [&](int b) { return (split + b * step) * KB; };

  // Staging registers: this thread's 4-element units of the next batch's rows, raw: key rows unit by unit,
  // value rows as blocks of 4 keys x 4 columns (the transposed write is then 8 bytes).  Offsets inside
  // a batch are fixed per thread; the batch moves the buffer's base, whose size is the rows the tile
  // needs, so rows behind them (and units behind the columns) read as zero.
  int koff[KPT], voff[VPT];
#pragma unroll
  for (int i = 0; i < KPT; ++i) {
    const int e = tid + 256 * i, r = e / KU, u = e - r * KU;
    koff[i] = (e < KB * KU && 4 * u < a.d) ? (r * a.ldqk + 4 * u) * ES : 0x7ffffff0;
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int e = tid + 256 * i, g = e % KG, u = e / KG;  // key-fast: conflict-light transposed writes
    voff[i] = (e < KG * VU && 4 * u < a.dv) ? (4 * g * a.ldv + 4 * u) * ES : 0x7ffffff0;
  }
  const bool kclip = (a.d & 3) != 0, vclip = (a.dv & 3) != 0;
  const char* const kp0 = static_cast<const char*>(a.k) + qkbase * ES;
  const char* const vp0 = static_cast<const char*>(a.v) + vbase * ES;
  uint4 pk[KPT], pv[VPT][4];
  auto prefetch = [&](int off) {
    const __amdgpu_buffer_rsrc_t kr = flash_rsrc(kp0 + static_cast<int64_t>(off) * a.ldqk * ES,
                                                 static_cast<int64_t>(kend - off) * a.ldqk * ES);
    const __amdgpu_buffer_rsrc_t vr = flash_rsrc(vp0 + static_cast<int64_t>(off) * a.ldv * ES,
                                                 static_cast<int64_t>(kend - off) * a.ldv * ES);
#pragma unroll
    for (int i = 0; i < KPT; ++i) pk[i] = load_buf<ES>(kr, koff[i]);
#pragma unroll
    for (int i = 0; i < VPT; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        pv[i][c] = load_buf<ES>(vr, voff[i] == 0x7ffffff0 ? voff[i] : voff[i] + c * a.ldv * ES);
  };
  auto commit = [&](uint16_t* Kst, uint16_t* Vst) {
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int e = tid + 256 * i, r = e / KU, u = e - r * KU;
      if (KB * KU % 256 != 0 && e >= KB * KU) continue;
      uint4 x = pk[i];
      if (kclip) x = unit_clip<ES>(x, a.d - 4 * u);
      if constexpr (IN == F32) {
        const floatx4 f = unit_to_f4<4>(x, F32, 1.f);
        uint32_t p0[KP], p1[KP];
        plane_pair<KP, false>(f[0], f[1], p0);
        plane_pair<KP, false>(f[2], f[3], p1);
#pragma unroll
        for (int j = 0; j < KP; ++j) *reinterpret_cast<uint2*>(Kst + j * KPL + r * LDK + 4 * u) = uint2{p0[j], p1[j]};
      } else {
        *reinterpret_cast<uint2*>(Kst + r * LDK + 4 * u) = uint2{x.x, x.y};
      }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int e = tid + 256 * i, g = e % KG, u = e / KG;
      if (KG * VU % 256 != 0 && e >= KG * VU) continue;
      uint4 x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[c] = vclip ? unit_clip<ES>(pv[i][c], a.dv - 4 * u) : pv[i][c];
      uint16_t* const dst = Vst + 4 * u * LDV + flash_key_pos(4 * g);
      if constexpr (VP == 1) {
        // 16-bit 4 x 4 transpose: column m of the 4 keys
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const uint32_t sel = (m & 1) ? 0x07060302u : 0x05040100u;
          const uint32_t k0 = m < 2 ? x[0].x : x[0].y, k1 = m < 2 ? x[1].x : x[1].y;
          const uint32_t k2 = m < 2 ? x[2].x : x[2].y, k3 = m < 2 ? x[3].x : x[3].y;
          *reinterpret_cast<uint2*>(dst + m * LDV) =
              uint2{__builtin_amdgcn_perm(k1, k0, sel), __builtin_amdgcn_perm(k3, k2, sel)};
        }
      } else {
        floatx4 f[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) f[c] = unit_to_f4<ES>(x[c], IN, 1.f);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          uint32_t p0[VP], p1[VP];
          plane_pair<VP, false>(f[0][m], f[1][m], p0);
          plane_pair<VP, false>(f[2][m], f[3][m], p1);
#pragma unroll
          for (int j = 0; j < VP; ++j) *reinterpret_cast<uint2*>(dst + j * VPL + m * LDV) = uint2{p0[j], p1[j]};
        }
      }
    }
  };

  if constexpr (DPS != DP) {  // dimensions [DP, DPS) of the key rows are never written: zero them
    for (int s = 0; s < NST; ++s)
      for (int e = tid; e < KP * KPL; e += 256) stage[s * STAGE + e] = 0;
    __syncthreads();
  }
  auto compute = [&](int b, const uint16_t* st) {
    const int off = offset(b);
    if (off < wlim_hi) {
      if (off + KB > wlim_lo)
        process(std::true_type{}, off, st, st + KP * KPL);
      else
        process(std::false_type{}, off, st, st + KP * KPL);
    }
  };
  if (nb > 0) prefetch(offset(0));
  if constexpr (NST == 2) {
    if (nb > 0) commit(stage, stage + KP * KPL);
    if (nb > 1) prefetch(offset(1));
    __syncthreads();
    for (int b = 0; b < nb; ++b) {
      compute(b, stage + (b & 1) * STAGE);
      // the other stage was read by batch b - 1, which every wave finished before the last barrier
      if (b + 1 < nb) commit(stage + ((b + 1) & 1) * STAGE, stage + ((b + 1) & 1) * STAGE + KP * KPL);
      if (b + 2 < nb) prefetch(offset(b + 2));
      __syncthreads();
    }
  } else {
    for (int b = 0; b < nb; ++b) {
      __syncthreads();  // every wave is done with the stage of the previous batch
      commit(stage, stage + KP * KPL);
      __syncthreads();  // staged batch visible
      if (b + 1 < nb) prefetch(offset(b + 1));
      compute(b, stage);
    }
  }

  // Planes hold neither infinities nor fp32 values that round to one (above 3.396e38, the type's lowest among
  // them: a key switched off by a dimension of -inf or the lowest value), and lose the last bits of values whose
  // lower planes are subnormal.  Either shows in the sums: the first as an infinity or a NaN (inf - inf in the
  // second plane), the second as values below 2^-95.  A wave with such a row takes its rows again in fp32 matrix
  // instructions, a strip at a time, the next 16 keys' operands in flight from memory (no barrier: the other
  // waves are not needed).  Few registers, so that the products above keep theirs: wide values repeat the logits
  // for each 64 columns.
  if constexpr (FP32_ROWS) {
    bool bad = false;
#pragma unroll
    for (int rs = 0; rs < RS; ++rs) {
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int ct = 0; ct < DVT; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r & 1] += fabsf(num[rs][ct][r]);
      float ds = DENM ? dacc[rs][0] : den[rs];
      if constexpr (!DENM) {
        ds += __shfl_xor(ds, 16);
        ds += __shfl_xor(ds, 32);
      }
      const float all = sum[0] + sum[1];
      const bool b = !(all + fabsf(ds) < __builtin_huge_valf()) || (IN == F32 && all < ds * 0x1p-95f && all > 0.f);
      bad = bad || (b && rvalid[rs]);
    }
    if (__builtin_expect(a.direct != 0 || __any(bad), false)) {
      constexpr int CT = DVT < 4 ? DVT : 4, DU = DP / 16;
      const bool softmax = W == FLASH_SOFTMAX || (IN != F32 && a.direct == 2);
#pragma unroll 1
      for (int job = 0; job < RS * (DVT / CT); ++job) {
        const int ct0 = job / RS * CT, rbase = r0 + (wave * RS + job % RS) * 16, row = rbase + li;
        const int lrow = limit(row), jend = min(kend, limit(rbase + 15));
        // 4 dimensions a lane group and step: columns 16 m + 4 lg of a row
        auto row_units = [&](floatx4 (&f)[DU], const void* p, int64_t at, bool on, float scale) {
#pragma unroll
          for (int m = 0; m < DU; ++m) {
            const int col = 16 * m + 4 * lg;
            f[m] = unit_to_f4<ES>(unit_clip<ES>(load_unit<ES>(p, at + min(col, a.ldqk - 4)), on ? a.d - col : 0), IN, scale);
          }
        };
        floatx4 qf[DU], kf[DU], acc[CT];
        float vf[4][CT], ds = 0.f, top = -1e30f;
        // keys j0 + li and values of keys j0 + 4 lg + s; those behind jend are zero
        auto load_keys = [&](int j0) {
          row_units(kf, a.k, qkbase + static_cast<int64_t>(min(j0 + li, jend - 1)) * a.ldqk, j0 + li < jend, 1.f);
        };
        auto load_values = [&](int j0) {
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const int j = j0 + 4 * lg + s;
            const int64_t vrow = vbase + static_cast<int64_t>(min(j, jend - 1)) * a.ldv;
#pragma unroll
            for (int c = 0; c < CT; ++c) {
              const int col = 16 * (ct0 + c) + li;
              const float x = load_elem(a.v, vrow + min(col, a.dv - 1), IN);
              vf[s][c] = j < jend && col < a.dv ? x : 0.f;
            }
          }
        };
        row_units(qf, a.q, qkbase + static_cast<int64_t>(row < n ? row : 0) * a.ldqk, row < n, a.scale2);
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        int b = 0, j0 = offset(0);
        if (nb_own > 0 && j0 < jend) {
          load_keys(j0);
          load_values(j0);
        }
#pragma unroll 1
        while (b < nb_own && j0 < jend) {
          int next = j0 + 16;  // the batch's next 16 keys, or the next batch
          if (next >= offset(b) + KB) next = offset(++b);
          const int j = j0;
          j0 = next;
          floatx4 x = {0.f, 0.f, 0.f, 0.f};  // keys j + 4 lg + r of the row
#pragma unroll
          for (int m = 0; m < DU; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) x = mfma4(kf[m][e], qf[m][e], x);
          const bool more = b < nb_own && j0 < jend;
          if (more) load_keys(j0);
          float m0 = 0.f;
          if (softmax) {
            m0 = top;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (j + 4 * lg + r < lrow) m0 = fmaxf(m0, x[r]);
            m0 = fmaxf(m0, __shfl_xor(m0, 16));
            m0 = fmaxf(m0, __shfl_xor(m0, 32));
            const float alpha = __builtin_amdgcn_exp2f(top - m0);
            top = m0;
            ds *= alpha;
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[c] *= alpha;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            x[r] = j + 4 * lg + r < lrow ? __builtin_amdgcn_exp2f(x[r] - m0) : 0.f;
            ds += x[r];
          }
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[c] = mfma4(vf[s][c], x[s], acc[c]);
          if (more) load_values(j0);
        }
        ds += __shfl_xor(ds, 16);
        ds += __shfl_xor(ds, 32);
        if (row >= n) continue;
        const int64_t part = (split * a.bh + bh) * a.n + row, obase = (bh * a.n + row) * a.dv;
        if (a.nsplit > 1 && lg == 0 && ct0 == 0)
          *reinterpret_cast<floatx2*>(a.low_den + 2 * part) = floatx2{ds, softmax ? top : 0.f};
        const float dn = fmaxf(ds, a.floor);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          const int c0 = 16 * (ct0 + c) + 4 * lg;
          if (a.nsplit > 1) {
            if (c0 < a.low_ld) *reinterpret_cast<floatx4*>(a.low_num + part * a.low_ld + c0) = acc[c];
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (c0 + r < a.dv) store_elem(a.out, obase + c0 + r, a.out_dtype, acc[c][r] / dn);
          }
        }
      }
      return;
    }
  }
  // ---- epilogue: row sums (over the four lane groups), normalise, store ----
#pragma unroll
  for (int rs = 0; rs < RS; ++rs) {
    float dsum;
    if constexpr (DENM) {
      dsum = dacc[rs][0];  // every element of the column is the row's sum
    } else {
      dsum = den[rs];
      dsum += __shfl_xor(dsum, 16);
      dsum += __shfl_xor(dsum, 32);
    }
    if (!rvalid[rs]) continue;
    if constexpr (TAYLOR) {
      const int64_t row = (bh * a.nsplit + split) * a.low_rows + a.low_off + myrow[rs];
      if (lg == 0) a.low_den[row] = dsum;
#pragma unroll
      for (int ct = 0; ct < DVT; ++ct) {
        const int c0 = 16 * ct + 4 * lg;  // low_ld is whole 32-column groups
        if (c0 < a.dv) *reinterpret_cast<floatx4*>(a.low_num + row * a.low_ld + c0) = num[rs][ct];
      }
      continue;
    }
    if (a.nsplit > 1) {
      const int64_t row = (split * a.bh + bh) * a.n + myrow[rs];
      if (lg == 0) *reinterpret_cast<floatx2*>(a.low_den + 2 * row) = floatx2{dsum, W == FLASH_SOFTMAX ? mrow[rs] : 0.f};
#pragma unroll
      for (int ct = 0; ct < DVT; ++ct) {
        const int c0 = 16 * ct + 4 * lg;
        if (c0 < a.low_ld) *reinterpret_cast<floatx4*>(a.low_num + row * a.low_ld + c0) = num[rs][ct];
      }
      continue;
    }
    const float dn = fmaxf(dsum, a.floor);
    const int64_t obase = (bh * a.n + myrow[rs]) * a.dv;
#pragma unroll
    for (int ct = 0; ct < DVT; ++ct) {
      const int c0 = 16 * ct + 4 * lg;
      if (c0 >= a.dv) continue;
      floatx4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = num[rs][ct][r] / dn;
      if (a.vec_out) {
        *reinterpret_cast<floatx4*>(static_cast<float*>(a.out) + obase + c0) = o;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (c0 + r < a.dv) store_elem(a.out, obase + c0 + r, a.out_dtype, o[r]);
      }
    }
  }
}

// out = the nsplit raw sums relative to their largest maximum, added in order, over their denominator; four columns
// a thread.
static __global__ __launch_bounds__(256) void flash_combine_kernel(const FlashArgs a) {
  const int cu = a.low_ld >> 2;
  const int64_t rows = a.bh * a.n;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t row = e / cu;
  if (row >= rows) return;
  const int c0 = static_cast<int>(e - row * cu) * 4;
  const floatx2* const dm = reinterpret_cast<const floatx2*>(a.low_den);
  float top = dm[row][1];
  for (int s = 1; s < a.nsplit; ++s) top = fmaxf(top, dm[s * rows + row][1]);
  floatx4 o = {0.f, 0.f, 0.f, 0.f};
  float den = 0.f;
  for (int s = 0; s < a.nsplit; ++s) {
    const int64_t r = s * rows + row;
    const floatx2 d = dm[r];
    const float f = __builtin_amdgcn_exp2f(d[1] - top);
    o += f * *reinterpret_cast<const floatx4*>(a.low_num + r * a.low_ld + c0);
    den = fmaf(f, d[0], den);
  }
  const float dn = fmaxf(den, a.floor);
#pragma unroll
  for (int m = 0; m < 4; ++m)
    if (c0 + m < a.dv) store_elem(a.out, row * a.dv + c0 + m, a.out_dtype, o[m] / dn);
}

}  // namespace sta
