// Paged attention that emits the softmax log-sum-exp (the lse producer ActKV
// Algorithm 3 consumes) for gfx950.
//
// Reference: actkv/kernels/lse_attn.py:42-60 (paged_decode_attention_ref, the
// stand-in for "the paged FlashAttention backend whose LSE by-product
// Algorithm 3 consumes") and actkv/paged.py:115-118 (decode_attention).  For
// every query row (query n of request r, query head hq) and the tokens t it
// sees (t < seq_used[r], and t < kv_len[r, n] when causal limits are given):
//   s_t = scale * q . k_t,  lse = logsumexp_t s_t,  out = sum_t softmax(s)_t v_t
// out and lse are float32.  A row that sees no token gets lse = -inf, out = 0
// (torch's logsumexp and softmax-einsum over an empty set).
//
// MFMA path (bf16/fp16, head_dim 256, 128 or 64, any GQA group, more than one 32-row tile
// of query rows per pair; any number at head dim 256): FlashAttention-style,
// one workgroup per (layer, request, KV head, group of NW row tiles), NW waves,
// each owning one 32-row tile of the pair's query rows (n, g) and streaming all
// of the request's tokens.  The transposed products keep every per-query
// quantity inside one lane:
//   S^T = K . Q^T   (v_mfma_f32_32x32x16: A = K rows from LDS, B = Q in registers)
//   lane (lcol, lh) holds s for query row lcol and 16 of the slice's 32 tokens,
//   so the running max / sum of a row are lane-local plus one v_permlane32_swap;
//   O^T += V^T . P^T (A = V^T from LDS, B = P^T: the lane's own 16 probabilities,
//   taken in the token order tau(kb, lh, j) = 16kb + 8(j/4) + 4lh + j%4 that
//   matches the S^T register layout, so no shuffle is needed).  P is split into
//   hi = P rounded to the cache dtype and lo = (P - hi) rounded again, and both
//   terms go through the matrix core: P then carries about 16 significant bits
//   (bf16) instead of 8, so out is within ~1e-5 of the float32 softmax @ v.
// K and V stages go straight from HBM into an LDS ring (buffer loads with the LDS
// bit, several stages ahead), rows XOR-swizzled; V is read back transposed
// (ds_read_b64_tr_b16).  Described at attn_ring_kernel.
//
// Decode path (head dims 128 and 64, the same dtypes, when a pair's query rows fit one 32-row
// tile, N*G <= 32): four waves per (pair, token chunk), each streaming its own
// slices through a private LDS region without workgroup barriers; V comes back
// transposed from LDS (ds_read_b64_tr_b16).  Described at attn_decode_kernel.
//
// Head dim 64 runs the same kernels with half-length token rows: a 16-byte load
// instruction then moves eight rows instead of four, the rows' eight 16-byte chunks are
// swizzled with their own pattern (dswz), and two 32-dim output tiles replace four.
//
// Head dim 256 runs the ring kernel for every row count, one wave per SIMD (a wave's O tile is 128
// registers, its query rows 64), with P as three terms in bf16.  16 query heads over 8 KV heads
// in bf16, against the float32 path these shapes took before: 24 causal queries over 12000 and
// 5003 tokens, attention and scoring together, 742 -> 91 us; a decode step over 8 x 8k tokens
// 318 -> 115 us; 700 causal queries over 3000 and 2003 tokens 2567 -> 225 us.  out is 5.5e-7 to
// 6.9e-7 from 64 bits on them, against 7.7e-7 to 9.9e-7.
//
// Generic path (any other dtype / head_dim up to 512 / block size): float32, up to 8
// query rows of one KV head per workgroup (a decode step's GQA group of up to 8 heads
// reads K and V once), one pass with an online max and sum, token chunks merged by the
// same combine launch.  Described at attn_generic_kernel.
#include "common.h"

#include <algorithm>
#include <cmath>

namespace actkv {

struct AttnArgs {
  const void *q;
  int64_t q_sl, q_sr, q_sn, q_sh;
  const void *kv;  // K plane of layer 0; the V plane is kv + kv_sv elements
  int64_t kv_sl, kv_sv, kv_sb, kv_ss, kv_sh;
  int64_t num_blocks;
  const int32_t *bt;
  int64_t bt_sr;
  int max_blocks;
  const int32_t *seq_used, *n_valid, *kv_len;
  float *out;
  int64_t o_sl, o_sr, o_sn, o_sh;
  float *lse;
  int64_t lse_sl, lse_sr, lse_sn;
  int L, R, N, Hq, Hkv, D, G, BS;
  float scale;
  // token-range split (flash-decoding): chunks per sequence, tokens per chunk, and
  // the partial results of each chunk (row-major [pair][row][chunk])
  // dyn: the decode kernel's interleaved split (attn_dec_chunks); tpc is then unused
  int nchunk, tpc, rows_pad, dyn;
  float *ws_o;   // [pairs][rows_pad][nchunk][D]: unnormalised sum p v
  float *ws_ml;  // [pairs][rows_pad][nchunk][2]: running max (log2 units), sum p
};

__device__ __forceinline__ int attn_seq_len(const AttnArgs &a, int r) {
  const int s = a.seq_used[r];
  const int span = a.max_blocks * a.BS;
  return s < 0 ? 0 : (s > span ? span : s);
}

__device__ __forceinline__ int attn_nq(const AttnArgs &a, int r) {
  return a.n_valid ? min(max(a.n_valid[r], 0), a.N) : a.N;
}

// tokens query n of request r sees: [0, lim)
__device__ __forceinline__ int attn_lim(const AttnArgs &a, int r, int n, int S) {
  return a.kv_len ? min(max(a.kv_len[(int64_t)r * a.N + n], 0), S) : S;
}

// physical block of logical block `b` of request r, or -1 (past the table, or an
// id outside the pool)
__device__ __forceinline__ int attn_phys(const AttnArgs &a, int r, int b) {
  if (b < 0 || b >= a.max_blocks) return -1;
  const int64_t p = a.bt[(int64_t)r * a.bt_sr + b];
  return (p >= 0 && p < a.num_blocks) ? (int)p : -1;
}

// ------------------------------------------------------------------ chunk merge
// One wave merges the nc token chunks of query row `id` (pair * rows_pad + row) and writes
// out and lse, DH / 64 dims per lane:
//   M = max_c m_c, w_c = 2^(m_c - M), out = sum_c w_c O_c / sum_c w_c l_c,
//   lse = ln 2 * (M + log2 sum_c w_c l_c)
// Lane c reads chunk c's (max, sum) for up to 64 chunks at a time (a butterfly max and sum);
// the O rows of the first 16 chunks are loaded in the same round trip (rows past nc are
// never written: their terms are selected away, not multiplied by zero), later ones after.
template <int DH>
__device__ __forceinline__ void attn_merge_row(const AttnArgs &a, int64_t id, int nc, int64_t o_off,
                                               int64_t lse_off, int lane) {
  static_assert(DH == 64 || DH == 128 || DH == 256, "head dims");
  constexpr int PRE = 16, DL = DH / 64;
  const float *ml = a.ws_ml + id * a.nchunk * 2;
  const float *wo = a.ws_o + id * a.nchunk * DH;
  float pre[DL][PRE];
#pragma unroll
  for (int j = 0; j < PRE; ++j) {
    const int jc = max(0, min(j, nc - 1));  // an in-bounds row: the workspace holds nchunk >= max(nc, 1)
#pragma unroll
    for (int k = 0; k < DL; ++k) pre[k][j] = wo[(int64_t)jc * DH + 64 * k + lane];
  }
  float M = -INFINITY;
  for (int c = lane; c < nc; c += 64) M = fmaxf(M, ml[2 * c]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
  const float Ms = M == -INFINITY ? 0.f : M;
  float Lsum = 0.f, ov[DL];
#pragma unroll
  for (int k = 0; k < DL; ++k) ov[k] = 0.f;
  for (int c0 = 0; c0 < nc; c0 += 64) {
    const int c = c0 + lane;
    const float w = c < nc ? __builtin_amdgcn_exp2f(ml[2 * c] - Ms) : 0.f;
    float lw = c < nc ? w * ml[2 * c + 1] : 0.f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lw += __shfl_xor(lw, o, 64);
    Lsum += lw;
    if (c0 == 0) {
#pragma unroll
      for (int j = 0; j < PRE; ++j) {
        const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), j));
#pragma unroll
        for (int k = 0; k < DL; ++k) ov[k] += j < nc ? wj * pre[k][j] : 0.f;
      }
    }
    // the next chunks' rows, PRE at a time and all in flight together (one by one, 64 chunks of a
    // head-dim-256 row cost 48 round trips)
    for (int j0 = c0 == 0 ? PRE : 0; j0 < min(64, nc - c0); j0 += PRE) {
#pragma unroll
      for (int j = 0; j < PRE; ++j) {
        const int jc = min(c0 + j0 + j, nc - 1);
#pragma unroll
        for (int k = 0; k < DL; ++k) pre[k][j] = wo[(int64_t)jc * DH + 64 * k + lane];
      }
#pragma unroll
      for (int j = 0; j < PRE; ++j) {
        const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), j0 + j));   // 0 past nc
#pragma unroll
        for (int k = 0; k < DL; ++k) ov[k] += c0 + j0 + j < nc ? wj * pre[k][j] : 0.f;
      }
    }
  }
  const float inv = Lsum > 0.f ? 1.0f / Lsum : 0.f;
  float *op = a.out + o_off;
#pragma unroll
  for (int k = 0; k < DL; ++k) op[64 * k + lane] = ov[k] * inv;
  if (lane == 0) a.lse[lse_off] = Lsum > 0.f ? (M + __log2f(Lsum)) * 0.6931471805599453f : -INFINITY;
}

// The same merge for any head dim (the float32 path's chunks): the chunk weights are
// recomputed for each 64-dim slice of the row.
__device__ __forceinline__ void attn_merge_row_any(const AttnArgs &a, int64_t id, int nc, int64_t o_off,
                                                   int64_t lse_off, int lane) {
  const int D = a.D;
  const float *ml = a.ws_ml + id * a.nchunk * 2;
  const float *wo = a.ws_o + id * a.nchunk * D;
  float M = -INFINITY;
  for (int c = lane; c < nc; c += 64) M = fmaxf(M, ml[2 * c]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
  const float Ms = M == -INFINITY ? 0.f : M;
  float Lsum = 0.f;
  for (int c0 = 0; c0 < nc; c0 += 64) {
    const int c = c0 + lane;
    float lw = c < nc ? exp2f(ml[2 * c] - Ms) * ml[2 * c + 1] : 0.f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lw += __shfl_xor(lw, o, 64);
    Lsum += lw;
  }
  const float inv = Lsum > 0.f ? 1.0f / Lsum : 0.f;
  float *op = a.out + o_off;
  for (int d0 = 0; d0 < D; d0 += 64) {
    const int d = d0 + lane;
    float o = 0.f;
    if (d < D)
      for (int c = 0; c < nc; ++c) o += exp2f(ml[2 * c] - Ms) * wo[(int64_t)c * D + d];
    if (d < D) op[d] = o * inv;
  }
  if (lane == 0) a.lse[lse_off] = Lsum > 0.f ? (M + __log2f(Lsum)) * 0.6931471805599453f : -INFINITY;
}

// ------------------------------------------------------------------ MFMA path
// ------------------------------------------------------------------ decode path
// A pair whose query rows fit one 32-row tile (N*G <= 32: decode steps and short
// action regions) gets a workgroup of DW waves per token chunk, each wave streaming
// the chunk's 32-token slices w, w + DW, ... on its own.  The next slice's K and V
// rows are loaded into registers (coalesced 16-byte loads, four token rows per
// instruction) while the current slice is multiplied out of the wave's private LDS
// region, so the loop has no workgroup barrier.  K rows sit in LDS with their 16-byte
// chunks XOR-swizzled by token (conflict-free A-operand reads); V rows are stored the
// same way and read back with ds_read_b64_tr_b16, which hands each lane four
// consecutive tokens of one dim: the V^T operand with no register transpose.  The
// waves' (max, sum, O) merge through LDS at the end.  The pairs are split into chunks
// (1.5 * CUs / pairs, at least 8, or 12 at head dim 64; slices interleaved over their waves: attn_split), merged by the
// combine launch; a sequence whose slices fit one chunk is written here directly.
constexpr int DW = 4;                         // waves per decode workgroup

// Token-row geometry at head dim DH (2-byte elements): one KV head's row of a token is PB
// bytes, NC 16-byte chunks (NC = 2^NCS); a 64-lane 16-byte load moves RPI = 2^RPS rows;
// the S^T product takes KS 16-dim steps and O^T has DT 32-dim tiles.
template <int DH> struct RowShape {
  static_assert(DH == 64 || DH == 128 || DH == 256, "head dims");
  static constexpr int PB = 2 * DH, NC = PB / 16, NCS = NC == 32 ? 5 : NC == 16 ? 4 : 3;
  static constexpr int RPI = 64 / NC, RPS = 6 - NCS;
  static constexpr int KS = DH / 16, DT = DH / 32;
  static constexpr int DREG = 2 * 32 * PB;    // decode LDS bytes per wave: K rows, then V rows
};

// The decode split (a.dyn): slice s of a pair (tokens 32s .. 32s + 31) goes to wave
// s mod (nchunk * DW), that is wave s mod DW of chunk (s / DW) mod nchunk.  A wave's slices
// depend on the chunk count only (no other request's length is read); every request spreads
// over the chunks in proportion to its length; and nothing depends on the block table's
// width.  Chunks holding slices of a sequence of S tokens:
__device__ __forceinline__ int attn_dec_chunks(const AttnArgs &a, int S) {
  return min(a.nchunk, (((S + 31) >> 5) + DW - 1) / DW);
}

// 16-byte chunk slot of chunk c of token t is c ^ dswz(t).  Distinct bank groups (the
// address's 16-byte unit mod 16), so no LDS bank conflicts, for: 16 consecutive tokens at
// one chunk (K A-operand reads); four consecutive tokens at four consecutive chunks (a
// 32-lane transposed V read: 16 slots); the chunks of one row (row writes).
//   Head dim 128 (16 chunks, a row is 16 units; head dim 256, 32 chunks, the same modulo 16): 4 (t mod 4) + (t / 4 mod 4).  2 (t mod 8)
//   + (t / 8 mod 2) left the transposed V reads 2-way conflicted.
//   Head dim 64 (8 chunks, a row is 8 units, so rows of odd t use units 8-15): 4 (t / 2 mod 2)
//   + (t / 4 mod 4).  Among 16 tokens each parity takes all 8 values; tokens 4m and 4m + 2
//   (and 4m + 1, 4m + 3) differ in bit 2, so four consecutive chunks of them fall in
//   disjoint halves.
template <int DH>
__device__ __forceinline__ int dswz(int t) {
  if constexpr (DH >= 128) return 4 * (t & 3) + ((t >> 2) & 3);
  else return 4 * ((t >> 1) & 1) + ((t >> 2) & 3);
}

typedef short dv4s __attribute__((ext_vector_type(4)));

// Two floats rounded to T in one dword (one v_cvt_pk on gfx950; element-wise conversions take one
// each).
template <typename T>
__device__ __forceinline__ uint32_t pack2(float x, float y) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef T t2 __attribute__((ext_vector_type(2)));
  const f2 v = {x, y};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, t2));
}

// x - (low half of u) and x - (high half of u), both halves of type T: one dot product each in
// bf16 (the difference is exact where u is x rounded).  The constants (-1, 0) and (0, -1) come in
// registers: as a literal, 0x0000bf80 is assembled to the inline constant -1.0, which the dot
// product reads as 0xbf800000.
struct MinusOne { uint32_t lo, hi; };
__device__ __forceinline__ MinusOne minus_one() {
  MinusOne m;
  asm("s_mov_b32 %0, 0xbf80" : "=s"(m.lo));
  asm("s_mov_b32 %0, 0xbf800000" : "=s"(m.hi));
  return m;
}
__device__ __forceinline__ float minus_half(float x, uint32_t u, uint32_t m, int, __bf16) {
  typedef __bf16 t2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(t2, u), __builtin_bit_cast(t2, m), x, false);
}
__device__ __forceinline__ float minus_half(float x, uint32_t u, uint32_t, int half, _Float16) {
  typedef _Float16 t2 __attribute__((ext_vector_type(2)));
  return x - (float)__builtin_bit_cast(t2, u)[half];
}

// The probabilities of a 32-token slice, p[16] per lane, as TERMS operands of the cache dtype
// (eight values in four registers) for each 16-token k step: p = term 0 + term 1 (+ term 2),
// each the rest rounded.
template <typename T, int TERMS>
__device__ __forceinline__ void split_p(const float (&p)[16], uint4 (&out)[TERMS][2], MinusOne m1) {
  uint32_t w[TERMS][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float x = p[2 * i], y = p[2 * i + 1];
#pragma unroll
    for (int k = 0; k < TERMS; ++k) {
      w[k][i] = pack2<T>(x, y);
      if (k + 1 < TERMS) {
        x = minus_half(x, w[k][i], m1.lo, 0, T{});
        y = minus_half(y, w[k][i], m1.hi, 1, T{});
      }
    }
  }
#pragma unroll
  for (int k = 0; k < TERMS; ++k)
#pragma unroll
    for (int b = 0; b < 2; ++b)
      out[k][b] = make_uint4(w[k][4 * b], w[k][4 * b + 1], w[k][4 * b + 2], w[k][4 * b + 3]);
}

template <typename T, typename V8, int DH, bool CAUSAL>
__global__ void __launch_bounds__(DW * 64) __attribute__((amdgpu_waves_per_eu(DH == 64 ? 3 : 2, DH == 64 ? 3 : 2)))
attn_decode_kernel(AttnArgs a, int pairs, int bs_shift) {
  using RS = RowShape<DH>;
  constexpr int PB = RS::PB, NC = RS::NC, NCS = RS::NCS, RPI = RS::RPI, KS = RS::KS, DT = RS::DT;
  const int G = a.G;   // query heads per KV head: rows (n, g) of a tile are independent
  __shared__ __attribute__((aligned(16))) unsigned char reg_lds[DW][RS::DREG];
  __shared__ float mrg_ml[DW][32][2];
  __shared__ int wg_lim;
  const int p = blockIdx.x / a.nchunk, chunk = blockIdx.x % a.nchunk;
  if (p >= pairs) return;
  const int h = p % a.Hkv;
  const int r = (p / a.Hkv) % a.R;
  const int l = p / (a.Hkv * a.R);
  const int nq = attn_nq(a, r);
  if (nq * G <= 0) return;
  const int S_all = attn_seq_len(a, r);
  // chunks holding slices; with one (or none: chunk 0 then writes the empty result) the
  // workgroup writes the result itself, with more the combine launch merges them
  const int nact = a.nchunk > 1 ? max(attn_dec_chunks(a, S_all), 1) : 1;
  if (chunk >= nact) return;
  const int S = S_all;
  const int BS = a.BS;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lcol = lane & 31, lh = lane >> 5;
  const int row = lcol;
  const int n = row / G, g = row % G;
  const bool valid = n < nq;
  const int lim = valid ? min(max(attn_lim(a, r, n, S_all), 0), S) : 0;
  const int lim_m = valid ? lim : 0x7fffffff;
  int s_end = S;
  if constexpr (CAUSAL) {
    if (tid == 0) wg_lim = 0;
    __syncthreads();
    if (valid && lim > 0) atomicMax(&wg_lim, lim);
    __syncthreads();
    s_end = wg_lim;
  }
  const int nsl = (s_end + 31) / 32;  // slices of the pair anyone needs

  V8 qf[KS];
  {
    const T *qp = (const T *)a.q + (int64_t)l * a.q_sl + (int64_t)r * a.q_sr +
                  (int64_t)(valid ? n : 0) * a.q_sn + (int64_t)(h * G + g) * a.q_sh + lh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const V8 *)(qp + ks * 16);
    if (!valid) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = V8{};
    }
  }
  const T *kplane = (const T *)a.kv + (int64_t)l * a.kv_sl + (int64_t)h * a.kv_sh;
  const T *vplane = kplane + a.kv_sv;
  unsigned char *kl = reg_lds[wave];
  unsigned char *vl = kl + 32 * PB;

  // block-table entry of token group i (tokens 4i..4i+3) of slice s: lane i < 8 holds it.
  // Entries past the sequence are read too (bounds-checked by attn_phys): load_slice skips
  // their tokens.
  auto slice_phys = [&](int s) { return attn_phys(a, r, (s * 32 + 4 * (lane & 7)) >> bs_shift); };
  // lane: token rows RPI i + lane/NC (i < 32/RPI), 16-byte chunk lane%NC, of K and V.  The
  // RPI (4 or 8) rows of one load lie in one block (blocks hold at least 16 tokens), the
  // block of token group RPI i / 4.
  constexpr int NI = 32 / RPI;
  uint4 kr[NI], vr[NI];
  auto load_slice = [&](int s, int ph) {
    const int c = lane & (NC - 1);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int pb = __builtin_amdgcn_readlane(ph, i * RPI / 4);
      const int t = s * 32 + RPI * i + (lane >> NCS);
      const bool ok = pb >= 0 && t < S;
      const int64_t off = ok ? (int64_t)pb * a.kv_sb + (int64_t)(t & (BS - 1)) * a.kv_ss + c * 8 : 0;
      kr[i] = *(const uint4 *)(kplane + off);
      vr[i] = *(const uint4 *)(vplane + off);
      if (!ok) { kr[i] = make_uint4(0, 0, 0, 0); vr[i] = make_uint4(0, 0, 0, 0); }
    }
  };
  auto store_slice = [&]() {
    const int c = lane & (NC - 1);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int t = RPI * i + (lane >> NCS);
      const int o = t * PB + ((c ^ dswz<DH>(t)) << 4);
      *(uint4 *)(kl + o) = kr[i];
      *(uint4 *)(vl + o) = vr[i];
    }
  };

  const float c2 = a.scale * 1.4426950408889634f;
  const MinusOne m1 = minus_one();
  float m2 = -INFINITY, lsum = 0.f;
  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[dt][e] = 0.f;

  auto compute = [&](int s) {
    // S^T = K . Q^T for the slice's 32 tokens (A: token lcol, dims 16ks + 8lh .. +7)
    f32x16 st = {};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int c = 2 * ks + lh;
      const V8 kf = *(const V8 *)(kl + lcol * PB + ((c ^ dswz<DH>(lcol)) << 4));
      if constexpr (__is_same(T, __bf16))
        st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], st, 0, 0, 0);
      else
        st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[ks], st, 0, 0, 0);
    }
    const int t0 = s * 32;
    if (__builtin_amdgcn_ballot_w64(lim_m < t0 + 32) != 0ull) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int t = t0 + 8 * (e >> 2) + 4 * lh + (e & 3);
        st[e] = t < lim_m ? st[e] : -INFINITY;
      }
    }
    float mx = st[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, st[e]);
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const float m_new = fmaxf(m2, mx * c2);
    const float msafe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m2 - msafe);
    float ps = 0.f;
    float pe[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      pe[e] = __builtin_amdgcn_exp2f(fmaf(st[e], c2, -msafe));
      ps += pe[e];
    }
    uint4 pt[2][2];  // P = hi + lo, both in the cache dtype
    split_p<T, 2>(pe, pt, m1);
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(ps), __float_as_uint(ps), false, false);
      ps = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    lsum = lsum * alpha + ps;
    m2 = m_new;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0ull) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[dt][e] *= alpha;
    }
    // O^T += V^T . P^T.  A = V^T[dim][tau(kb, lh, j)]: two transposed reads give tokens
    // 16kb + 4lh + 0..3 and + 8..11 of dim 32dt + 16((lane/16)&1) + lane%16; lane
    // 4j' + q' of each 16-lane group points at token j', dims 4q' .. 4q'+3
    const int jj = (lane & 15) >> 2, qq = lane & 3;
    const int dgrp = 16 * ((lane >> 4) & 1) + 4 * qq;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int d = 32 * dt + dgrp;
        const int cc = d >> 3, half = (d >> 2) & 1;
        const int t_lo = 16 * kb + 4 * lh + jj, t_hi = t_lo + 8;
        const dv4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (dv4s __attribute__((address_space(3))) *)(vl + t_lo * PB + ((cc ^ dswz<DH>(t_lo)) << 4) + half * 8));
        const dv4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (dv4s __attribute__((address_space(3))) *)(vl + t_hi * PB + ((cc ^ dswz<DH>(t_hi)) << 4) + half * 8));
        // whole-register casts: the 64-bit results become the operand's two halves
        // (inserting the 16-bit elements one by one compiled to a wrong operand)
        const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
        const V8 va = __builtin_bit_cast(V8, make_uint4(l2.x, l2.y, h2.x, h2.y));
        if constexpr (__is_same(T, __bf16)) {
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(V8, pt[0][kb]), oacc[dt], 0, 0, 0);
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(V8, pt[1][kb]), oacc[dt], 0, 0, 0);
        } else {
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, __builtin_bit_cast(V8, pt[0][kb]), oacc[dt], 0, 0, 0);
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, __builtin_bit_cast(V8, pt[1][kb]), oacc[dt], 0, 0, 0);
        }
      }
    }
  };

  // ---- the wave's slices: wave, wave + DW, ...; table entries two slices ahead
  const int step = a.nchunk * DW;
  int s = chunk * DW + wave;
  int ph_next = slice_phys(s + step);
  if (s < nsl) load_slice(s, slice_phys(s));
  for (; s < nsl; s += step) {
    store_slice();
    if (s + step < nsl) load_slice(s + step, ph_next);
    ph_next = slice_phys(s + 2 * step);
    compute(s);
  }

  // ---- merge the waves' (max, sum, O) through LDS
  __syncthreads();
  {
    float *om = (float *)reg_lds[wave];   // DT x 4 KiB: the wave's DREG bytes
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) om[(dt * 16 + e) * 64 + lane] = oacc[dt][e];
    if (lh == 0) { mrg_ml[wave][lcol][0] = m2; mrg_ml[wave][lcol][1] = lsum; }
  }
  __syncthreads();
  if (wave == 0) {
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < DW; ++w) M = fmaxf(M, mrg_ml[w][lcol][0]);
    const float Ms = M == -INFINITY ? 0.f : M;
    float Lsum = 0.f, wgt[DW];
#pragma unroll
    for (int w = 0; w < DW; ++w) {
      wgt[w] = __builtin_amdgcn_exp2f(mrg_ml[w][lcol][0] - Ms);
      Lsum += wgt[w] * mrg_ml[w][lcol][1];
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float o = 0.f;
#pragma unroll
        for (int w = 0; w < DW; ++w) o += wgt[w] * ((const float *)reg_lds[w])[(dt * 16 + e) * 64 + lane];
        oacc[dt][e] = o;
      }
    if (valid && nact > 1) {  // this chunk's partial result
      const int64_t pr = ((int64_t)p * a.rows_pad + row) * a.nchunk + chunk;
      float *wo = a.ws_o + pr * DH;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4 v;
          v[0] = oacc[dt][4 * i]; v[1] = oacc[dt][4 * i + 1]; v[2] = oacc[dt][4 * i + 2]; v[3] = oacc[dt][4 * i + 3];
          *(f32x4 *)(wo + 32 * dt + 8 * i + 4 * lh) = v;
        }
      if (lh == 0) { a.ws_ml[pr * 2] = M; a.ws_ml[pr * 2 + 1] = Lsum; }
    } else if (valid) {       // the whole sequence: the result
      const float inv = Lsum > 0.f ? 1.0f / Lsum : 0.f;
      float *op = a.out + (int64_t)l * a.o_sl + (int64_t)r * a.o_sr + (int64_t)n * a.o_sn + (int64_t)(h * G + g) * a.o_sh;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d0 = 32 * dt + 8 * i + 4 * lh;
          f32x4 v;
          v[0] = oacc[dt][4 * i] * inv; v[1] = oacc[dt][4 * i + 1] * inv;
          v[2] = oacc[dt][4 * i + 2] * inv; v[3] = oacc[dt][4 * i + 3] * inv;
          *(f32x4 *)(op + d0) = v;
        }
      if (lh == 0)
        a.lse[(int64_t)l * a.lse_sl + (int64_t)r * a.lse_sr + (int64_t)n * a.lse_sn + h * G + g] =
            Lsum > 0.f ? (M + __log2f(Lsum)) * 0.6931471805599453f : -INFINITY;
    }
  }
}

// ------------------------------------------------------------------ ring path
// Pairs with more than one 32-row tile.  A workgroup of NW waves (one row tile each)
// shares ST-token stages of K and V held in an NSTG-deep LDS ring.  The stages are
// loaded straight into LDS with buffer_load_dwordx4 ... lds, NSTG - 1 stages ahead of
// the one being multiplied: no register staging, one LDS barrier per stage, and the
// wait for a stage is counted by hand (wait_stages).  Each load instruction moves
// four token rows (eight at head dim 64; 1 KB) of one block, so the buffer resource is that
// block (wave-uniform); its lanes pick the global 16-byte chunk that lands in their LDS
// slot, which lays rows out with the decode path's XOR swizzle, and tokens past the
// chunk (or in blocks the table marks invalid) are out of the resource's range, so the
// hardware writes zeros.  V is read back transposed (ds_read_b64_tr_b16).  The block
// table of the workgroup's token range sits in an LDS window, refilled (after a drain)
// when the loads reach its end.

// s_waitcnt with vmcnt <= N and the other counters unconstrained
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// workgroup barrier ordering LDS only (no drain of the loads in flight)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Stage size and ring depth, from a sweep on 36 layers x 32k tokens x 128 queries and on
// 4 requests x 8k tokens x 48 causal queries: with the loads issued ahead, depth matters
// little (3 or 4 stages of 64 tokens and 2 of 128 are within 8%) and fewer, larger stages
// (fewer barriers) win; 4- and 2-wave workgroups keep 64-token stages so that two fit
// per CU.  Head dim 256: what fits twice per CU (32 tokens of K and V are 32 KB) for one and two
// waves, 64 tokens for four.
constexpr int ring_stage(int tiles, int dh) {
  return dh == 256 ? (tiles >= 4 ? 64 : 32) : tiles >= 8 ? 128 : 64;
}
template <int TILES, int DH> struct RingShape {             // TILES: row tiles per workgroup
  static constexpr int ST = ring_stage(TILES, DH);            // tokens per stage
  static constexpr int NSTG = 2;                              // ring depth
  static constexpr int TBLW = TILES >= 8 ? 4096 : 2048;       // block-table window (entries)
  static constexpr int SBYTES = 2 * ST * RowShape<DH>::PB;    // K then V rows of a stage
  static constexpr int IPP = ST / RowShape<DH>::RPI;          // load instructions per plane
  static_assert(ST % 32 == 0, "whole slices per stage");
};

// wait until at most `rem` stages' loads (PER instructions each) are outstanding
template <int PER, int MAXR>
__device__ __forceinline__ void wait_stages(int rem) {
  if constexpr (MAXR >= 3) { if (rem >= 3) { wait_vmcnt<3 * PER>(); return; } }
  if constexpr (MAXR >= 2) { if (rem >= 2) { wait_vmcnt<2 * PER>(); return; } }
  if constexpr (MAXR >= 1) { if (rem >= 1) { wait_vmcnt<PER>(); return; } }
  wait_vmcnt<0>();
}

typedef int ri32x4 __attribute__((ext_vector_type(4)));

// N loads of 16 bytes per lane from buffer `rsrc`, at byte offsets voff[i], into LDS at
// lds_base + 1024 i + 16 * lane.  Inline assembly: the compiler's wait counting would otherwise
// drain every load in flight before each LDS read of the ring; the kernel counts them itself.
// M0 carries the LDS base and is restored.
template <int N>
__device__ __forceinline__ void buf_lds16(ri32x4 rsrc, const unsigned *voff, unsigned lds_base) {
  static_assert(N % 2 == 0, "pairs of loads");
  unsigned saved;
  if constexpr (N == 2) {
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(voff[0]), "v"(voff[1]), "s"(rsrc), "s"(lds_base)
                 : "memory", "scc");
  } else if constexpr (N == 4) {
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %6\n\tbuffer_load_dwordx4 %1, %5, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\tbuffer_load_dwordx4 %2, %5, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\tbuffer_load_dwordx4 %3, %5, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\tbuffer_load_dwordx4 %4, %5, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(rsrc), "s"(lds_base)
                 : "memory", "scc");
  } else {
    buf_lds16<4>(rsrc, voff, lds_base);
    buf_lds16<N - 4>(rsrc, voff + 4, lds_base + 4096);
  }
}

// Issue order of a slice: MF matrix products and RD LDS reads among its VALU work (about 130
// operations).
template <int MF, int RD>
__device__ __forceinline__ void slice_schedule() {
    constexpr int PRE = RD < 4 ? RD : 4, VPM = MF >= 128 ? 1 : 128 / MF;
  __builtin_amdgcn_sched_group_barrier(0x100, PRE, 0);     // DS read
#pragma unroll
  for (int i = 0; i < MF; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // MFMA
    if (i < RD - PRE) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);   // VALU
  }
}

// A row's probabilities are 2^(s - m2).  With P as three terms (24 bits) the reference m2 follows
// the running max only when the max of some row of the tile is more than REF_SLACK ahead, and then
// all of the tile's sums and O are rescaled: p stays below 2^8, with the same relative precision.
// With two terms m2 is the running max itself: its token then has p = 1, which two terms hold
// exactly, and where attention is peaked that token dominates (bf16 causal prefill 1.5e-6 from 64
// bits, 2.4e-6 with the slack).
constexpr float REF_SLACK = 8.0f;

template <typename T, typename V8, int DH, int NW, bool CAUSAL>
__global__ void __launch_bounds__(NW * 64)
__attribute__((amdgpu_waves_per_eu(DH == 256 ? 1 : (NW >= 4 ? 2 : 1), DH == 256 ? 1 : 2)))
attn_ring_kernel(AttnArgs a, int pairs, int ngroups, int bs_shift) {
  const int G = a.G;   // query heads per KV head: rows (n, g) of a tile are independent
  using SH = RingShape<NW, DH>;
  using RS = RowShape<DH>;
  constexpr int PB = RS::PB, NC = RS::NC, NCS = RS::NCS, RPI = RS::RPI, KS = RS::KS, DT = RS::DT;
  constexpr int ST = SH::ST, NSTG = SH::NSTG, TBLW = SH::TBLW;
  constexpr int PER = 2 * SH::IPP / NW;  // load instructions per wave per stage
  // bf16 at head dim 256: a third term gives P 24 significant bits, as many as the float32 path
  // that serves the other dtypes there (with hi + lo alone out was 1.3e-6 from 64 bits on
  // causal prefill against that path's 7.7e-7)
  constexpr int PT = DH == 256 && __is_same(T, __bf16) ? 3 : 2;
  static_assert(NSTG == 2, "the fragment addresses alternate between two ring slots");
  static_assert((2 * SH::IPP) % NW == 0, "whole load instructions per wave");
  __shared__ __attribute__((aligned(1024))) unsigned char ring[NSTG][SH::SBYTES];
  __shared__ int tbl[TBLW];
  __shared__ int wg_lim;

  // XCD-aware mapping: the row groups and chunks of one pair share an XCD
  const int bid = blockIdx.x;
  const int xcd = bid & 7, jj = bid >> 3;
  const int per_pair = ngroups * a.nchunk;
  const int seq = (jj / per_pair) * 8 + xcd;
  // causal: the last groups see the most tokens and go first, so that the launch ends on short ones
  const int gpos = (jj % per_pair) / a.nchunk, chunk = jj % a.nchunk;
  const int grp = CAUSAL ? ngroups - 1 - gpos : gpos;
  if (seq >= pairs) return;
  const int h = seq % a.Hkv;
  const int l = seq / (a.Hkv * a.R);
  // requests rotated by the layer: an XCD's workgroups go to its shader engines in turn, and with
  // as many requests as engines the longest would always meet the same one
  const int r = (seq / a.Hkv + l) % a.R;
  const int p = (l * a.R + r) * a.Hkv + h;   // the pair, as the merge counts them
  const int nq = attn_nq(a, r);
  if (grp * NW * 32 >= nq * G) return;
  const int S_all = attn_seq_len(a, r);
  if (a.nchunk > 1 && chunk * a.tpc >= S_all) return;
  const int c_begin = min(chunk * a.tpc, S_all);
  const int S = min(S_all - c_begin, a.tpc);
  const int BS = a.BS;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lcol = lane & 31, lh = lane >> 5;
  const int row = (grp * NW + wave) * 32 + lcol;
  const int n = row / G, g = row % G;
  const bool valid = n < nq;
  const bool active = (grp * NW + wave) * 32 < nq * G;   // a wave of padding rows only loads
  const int my_lim = valid ? min(max(attn_lim(a, r, n, S_all) - c_begin, 0), S) : 0;
  // the masking limit: padding rows (never written) see everything, so they never force it
  const int lim_m = valid ? my_lim : 0x7fffffff;
  int s_end = S;
  if constexpr (CAUSAL) {
    if (tid == 0) wg_lim = 0;
    __syncthreads();
    if (my_lim > 0) atomicMax(&wg_lim, my_lim);
    __syncthreads();
    s_end = wg_lim;
  }
  const int nst = (s_end + ST - 1) / ST;

  V8 qf[KS];
  {
    const T *qp = (const T *)a.q + (int64_t)l * a.q_sl + (int64_t)r * a.q_sr +
                  (int64_t)(valid ? n : 0) * a.q_sn + (int64_t)(h * G + g) * a.q_sh + lh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const V8 *)(qp + ks * 16);
    if (!valid) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = V8{};
    }
  }
  // the query loads complete here, before the first ring load: otherwise the compiler's
  // wait for them lands inside the loop, where the hardware counter also holds the
  // ring's loads and the wait would drain them every stage
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(qf[ks]));

  // ---- block table window: logical blocks [blk0 + wbase, blk0 + wbase + TBLW)
  const int blk0 = c_begin >> bs_shift;
  int wbase = 0;
  auto load_window = [&]() {
    for (int i = tid; i < TBLW; i += NW * 64) tbl[i] = attn_phys(a, r, blk0 + wbase + i);
  };
  load_window();
  __syncthreads();
  // before issuing stage gi: move the window when the stage's last block is past it (the
  // workgroup calls this uniformly; a stage spans at most ST / BS + 1 blocks)
  auto ensure_window = [&](int gi) {
    const int lb = ((c_begin + gi * ST + ST - 1) >> bs_shift) - blk0;
    if (lb - wbase >= TBLW) {
      __syncthreads();
      wbase = ((c_begin + gi * ST) >> bs_shift) - blk0;
      load_window();
      __syncthreads();
    }
  };

  // ---- stage loads: instruction k of a stage: plane k / IPP, tokens RPI(k % IPP) .. +RPI-1.
  // The V instructions of 16 consecutive tokens lie in one block (blocks hold at least 16 tokens,
  // stages start at a multiple of 32): they share a buffer resource that starts at the group's
  // first row, their offsets are the same for every group, and a stage's table entries come in
  // one LDS read (lane j holds the wave's group j).  A resource per instruction took 110 scalar
  // and 64 vector operations a stage; this takes 45 and 5.
  constexpr int V = 16 / RPI, GPW = PER / V, GPP = SH::IPP / V;
  static_assert(PER % V == 0 && SH::IPP % V == 0, "whole 16-token groups per wave and plane");
  const uint64_t kbase = (uint64_t)(uintptr_t)((const T *)a.kv + (int64_t)l * a.kv_sl + (int64_t)h * a.kv_sh);
  const uint64_t vbase = kbase + (uint64_t)a.kv_sv * sizeof(T);
  const unsigned ring_base = (unsigned)(uintptr_t)&ring[0][0];
  const int lrow = lane >> NCS;
  const unsigned ss_bytes = (unsigned)(a.kv_ss * (int64_t)sizeof(T));   // a block spans less than 4 GiB
  const unsigned grp_bytes = 15 * ss_bytes + PB;
  const uint64_t sb_bytes = (uint64_t)a.kv_sb * sizeof(T);
  unsigned vo[V];   // the global chunk landing in slot lane % NC of row RPI v + lrow
#pragma unroll
  for (int v = 0; v < V; ++v)
    vo[v] = (unsigned)(RPI * v + lrow) * ss_bytes + (unsigned)(((lane & (NC - 1)) ^ dswz<DH>(RPI * v + lrow)) << 4);
  const int g_lane = (wave * GPW + min(lane, GPW - 1)) % GPP;
  auto issue = [&](int gi) {
    const int phv = tbl[((c_begin + gi * ST + 16 * g_lane) >> bs_shift) - blk0 - wbase];
    const bool whole = gi * ST + ST <= S;                    // every token of the stage exists
    const unsigned slot = ring_base + (unsigned)((gi % NSTG) * SH::SBYTES);
#pragma unroll
    for (int j = 0; j < GPW; ++j) {
      const int k = wave * GPW + j;
      const int plane = k / GPP, tg = k % GPP;
      const int t0 = gi * ST + 16 * tg;                      // chunk-relative first token
      const int ph = __builtin_amdgcn_readlane(phv, j);
      const unsigned s_row = (unsigned)((c_begin + t0) & (BS - 1)) * ss_bytes;
      const uint64_t bb = (plane ? vbase : kbase) + (uint64_t)(ph < 0 ? 0 : ph) * sb_bytes + s_row;
      ri32x4 rs;
      rs[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)bb);
      rs[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(bb >> 32) & 0xffffu));
      rs[2] = __builtin_amdgcn_readfirstlane(ph < 0 ? 0 : (int)grp_bytes);
      rs[3] = 0x00020000;
      const unsigned dst = __builtin_amdgcn_readfirstlane(slot + (unsigned)(plane * ST * PB + tg * V * 1024));
      if (whole) {
        buf_lds16<V>(rs, vo, dst);
      } else {
        unsigned vt[V];
#pragma unroll
        for (int v = 0; v < V; ++v) vt[v] = t0 + RPI * v + lrow < S ? vo[v] : 0xfffffff0u;
        buf_lds16<V>(rs, vt, dst);
      }
    }
  };

  const float c2 = a.scale * 1.4426950408889634f;
  const MinusOne m1 = minus_one();
  float m2 = -INFINITY, lsum = 0.f;
  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[dt][e] = 0.f;

  const int jq = (lane & 15) >> 2, qq = lane & 3;
  const int dgrp = 16 * ((lane >> 4) & 1) + 4 * qq;
  // LDS addresses of this lane's fragments in the stage being multiplied: one per k step (K rows)
  // and two per output tile (V rows, tokens of j and j + 8); slices and k steps of 16 tokens are
  // constant offsets from them (computed per slice they took 27 VALU operations each)
  typedef const __attribute__((address_space(3))) unsigned char *lds_ptr;
  lds_ptr ka[KS], va_lo[DT], va_hi[DT];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    ka[ks] = (lds_ptr)&ring[0][0] + (lcol * PB + (((2 * ks + lh) ^ dswz<DH>(lcol)) << 4));
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int d = 32 * dt + dgrp, cc = d >> 3, half = (d >> 2) & 1;
    const int t_lo = 4 * lh + jq, t_hi = t_lo + 8;
    va_lo[dt] = (lds_ptr)&ring[0][0] + (ST * PB + t_lo * PB + ((cc ^ dswz<DH>(t_lo)) << 4) + half * 8);
    va_hi[dt] = (lds_ptr)&ring[0][0] + (ST * PB + t_hi * PB + ((cc ^ dswz<DH>(t_hi)) << 4) + half * 8);
  }
  // S^T = K . Q^T of the stage's 32-token slice b
  auto qk = [&](int b) {
    f32x16 st = {};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const V8 kf = *(const __attribute__((address_space(3))) V8 *)(ka[ks] + b * 32 * PB);
      if constexpr (__is_same(T, __bf16))
        st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], st, 0, 0, 0);
      else
        st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[ks], st, 0, 0, 0);
    }
    return st;
  };
  // tokens past a row's limit (slice at token t0): their logits become -inf
  auto mask = [&](f32x16 &x, int t0) {
    if (__builtin_amdgcn_ballot_w64(lim_m < t0 + 32) != 0ull) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int t = t0 + 8 * (e >> 2) + 4 * lh + (e & 3);
        x[e] = t < lim_m ? x[e] : -INFINITY;
      }
    }
  };
  // The probabilities of a slice against the rows' reference m2, as PT terms, and their sum ps.
  // Returns whether the reference moved (for the whole wave; m_old then holds the one before).
  auto softmax = [&](const f32x16 &x, uint4 (&pt)[PT][2], float &ps, float &m_old) {
    float mx = x[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, x[e]);
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const float m_new = fmaxf(m2, mx * c2);
    const bool grow = __builtin_amdgcn_ballot_w64(m_new > m2 + (PT == 3 ? REF_SLACK : 0.f)) != 0ull;
    m_old = m2;
    m2 = grow ? m_new : m2;
    const float msafe = m2 == -INFINITY ? 0.f : m2;
    float pe[16];
    ps = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      pe[e] = __builtin_amdgcn_exp2f(fmaf(x[e], c2, -msafe));
      ps += pe[e];
    }
    split_p<T, PT>(pe, pt, m1);
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(ps), __float_as_uint(ps), false, false);
    ps = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    // the terms are formed here, beside this slice's products, and not sunk to their use
#pragma unroll
    for (int k = 0; k < PT; ++k)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        asm volatile("" : "+v"(pt[k][kb].x), "+v"(pt[k][kb].y), "+v"(pt[k][kb].z), "+v"(pt[k][kb].w));
    return grow;
  };
  // O^T += V^T . P^T of slice b
  auto pv = [&](const uint4 (&pt)[PT][2], int b) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      V8 va[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const dv4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (dv4s __attribute__((address_space(3))) *)(va_lo[dt] + (b * 32 + 16 * kb) * PB));
        const dv4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (dv4s __attribute__((address_space(3))) *)(va_hi[dt] + (b * 32 + 16 * kb) * PB));
        const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
        va[dt] = __builtin_bit_cast(V8, make_uint4(l2.x, l2.y, h2.x, h2.y));
      }
      // one term over all output tiles before the next: consecutive products go to
      // different accumulators
#pragma unroll
      for (int k = 0; k < PT; ++k) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          if constexpr (__is_same(T, __bf16))
            oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[dt], __builtin_bit_cast(V8, pt[k][kb]), oacc[dt], 0, 0, 0);
          else
            oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[dt], __builtin_bit_cast(V8, pt[k][kb]), oacc[dt], 0, 0, 0);
        }
      }
    }
  };

  // ---- pipeline: stage g in ring slot g % NSTG, loads NSTG - 1 stages ahead
#pragma unroll
  for (int i = 0; i < NSTG - 1; ++i)
    if (i < nst) {
      ensure_window(i);
      issue(i);
    }
  for (int gs = 0; gs < nst; ++gs) {
    // stage gs has landed once at most rem younger stages' loads are outstanding
    wait_stages<PER, NSTG - 2>(min(NSTG - 2, nst - 1 - gs));
    lds_barrier();  // stage gs visible to all waves; stage gs - 1 is no longer read
    const int gi = gs + NSTG - 1;
    if (gi < nst) {
      ensure_window(gi);
      issue(gi);
    }
    // Slice b's softmax runs beside the products that do not need it: S^T of slice b + 1 and
    // P . V of slice b - 1 (one MFMA, its LDS reads and its share of the VALU work at a time:
    // left to the compiler, the exponentials had no MFMA beside them).  One wave can issue a VALU
    // operation every 5 cycles and an MFMA of this shape every 32, both at once; two waves share
    // a SIMD, oldest first, so a wave's own order decides how much of that is reached.  With
    // padding-only waves idle, the products of one term over all output tiles in a row, the lo
    // terms by dot products and one buffer resource per 16 tokens: 48 causal queries over 4 x 8k
    // tokens, 36 layers, 2022 -> 1873 us; 700 over 3000 and 2003 at head dim 256 259 -> 224;
    // decode at head dim 256 over 8 x 8k 151 -> 121.
    constexpr int NS = ST / 32;
    if (active) {
      f32x16 st_cur = qk(0);
      uint4 pt[PT][2];
#pragma unroll
      for (int b = 0; b < NS; ++b) {
        mask(st_cur, gs * ST + 32 * b);
        f32x16 st_next;
        uint4 pt_next[PT][2];
        float ps, m_old;
        if (b + 1 < NS) st_next = qk(b + 1);
        if (b > 0) pv(pt, b - 1);
        const bool grow = softmax(st_cur, pt_next, ps, m_old);
        if (b == 0 && NS > 1) slice_schedule<KS, KS>();
        else if (b + 1 < NS) slice_schedule<KS + 2 * DT * PT, KS + 4 * DT>();
        else if (NS > 1) slice_schedule<2 * DT * PT, 4 * DT>();
        if (grow) {
          const float alpha = __builtin_amdgcn_exp2f(m_old - (m2 == -INFINITY ? 0.f : m2));
          lsum *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) oacc[dt][e] *= alpha;
        }
        lsum += ps;
        st_cur = st_next;
#pragma unroll
        for (int k = 0; k < PT; ++k) { pt[k][0] = pt_next[k][0]; pt[k][1] = pt_next[k][1]; }
      }
      pv(pt, NS - 1);
    }
    // the lane's addresses move to the other ring slot
    const int hop = gs & 1 ? -SH::SBYTES : SH::SBYTES;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ka[ks] += hop;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) { va_lo[dt] += hop; va_hi[dt] += hop; }
  }

  if (!valid) return;
  // ---- split: the chunk's partial (unnormalised O, reference, sum) for the combine kernel
  if (a.nchunk > 1) {
    const int64_t pr = ((int64_t)p * a.rows_pad + row) * a.nchunk + chunk;
    float *wo = a.ws_o + pr * DH;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 v;
        v[0] = oacc[dt][4 * i]; v[1] = oacc[dt][4 * i + 1]; v[2] = oacc[dt][4 * i + 2]; v[3] = oacc[dt][4 * i + 3];
        *(f32x4 *)(wo + 32 * dt + 8 * i + 4 * lh) = v;
      }
    if (lh == 0) { a.ws_ml[pr * 2] = m2; a.ws_ml[pr * 2 + 1] = lsum; }
    return;
  }
  const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
  float *op = a.out + (int64_t)l * a.o_sl + (int64_t)r * a.o_sr + (int64_t)n * a.o_sn + (int64_t)(h * G + g) * a.o_sh;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d0 = 32 * dt + 8 * i + 4 * lh;
      f32x4 v;
      v[0] = oacc[dt][4 * i] * inv; v[1] = oacc[dt][4 * i + 1] * inv;
      v[2] = oacc[dt][4 * i + 2] * inv; v[3] = oacc[dt][4 * i + 3] * inv;
      *(f32x4 *)(op + d0) = v;
    }
  if (lh == 0)
    a.lse[(int64_t)l * a.lse_sl + (int64_t)r * a.lse_sr + (int64_t)n * a.lse_sn + h * G + g] =
        lsum > 0.f ? (m2 + __log2f(lsum)) * 0.6931471805599453f : -INFINITY;
}

// ------------------------------------------------------------------ split combine
// grid ceil(pairs*rows_pad/4), 256 threads: one wave per (pair, row) merging with
// attn_merge_row (DH = 0: attn_merge_row_any, the float32 path's head dims).  The decode
// kernel (a.dyn) wrote a sequence of at most one chunk's tokens itself: those rows are skipped.
template <int DH>
__global__ void __launch_bounds__(256) attn_combine_kernel(AttnArgs a, int pairs) {
  const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= (int64_t)pairs * a.rows_pad) return;
  const int lane = threadIdx.x & 63;
  const int p = (int)(id / a.rows_pad), row = (int)(id % a.rows_pad);
  const int h = p % a.Hkv;
  const int r = (p / a.Hkv) % a.R;
  const int l = p / (a.Hkv * a.R);
  const int n = row / a.G, g = row % a.G;
  if (n >= attn_nq(a, r)) return;
  // chunks past the sequence were never written: they hold no token of this row
  const int S_all = attn_seq_len(a, r);
  const int nc = a.dyn ? attn_dec_chunks(a, S_all) : min(a.nchunk, (S_all + a.tpc - 1) / a.tpc);
  if (a.dyn && nc <= 1) return;
  const int64_t o_off = (int64_t)l * a.o_sl + (int64_t)r * a.o_sr + (int64_t)n * a.o_sn + (int64_t)(h * a.G + g) * a.o_sh;
  const int64_t lse_off = (int64_t)l * a.lse_sl + (int64_t)r * a.lse_sr + (int64_t)n * a.lse_sn + h * a.G + g;
  if constexpr (DH == 0)
    attn_merge_row_any(a, id, nc, o_off, lse_off, lane);
  else
    attn_merge_row<DH>(a, id, nc, o_off, lse_off, lane);
}

// ------------------------------------------------------------------ generic path
// Any dtype pairing, head dims up to 512, any block size.  grid pairs * ngroups * nchunk,
// 256 threads: a workgroup takes up to NR query rows (n, g) of one (layer, request, KV
// head) pair -- a decode step's whole GQA group of up to 8 heads, so K and V are read once
// for all of its rows -- over one token chunk, 256 tokens at a time:
//   thread j: s_i = q_i . k_(t0+j) for each row i (the rows from LDS, the dot products in
//   registers as independent FMA chains), the tile's max and sum of p per row through wave
//   reductions and LDS, p_i,j into LDS; then O_i += sum_j p_i,j v_(t0+j) by token groups
//   (ceil(D/8) threads per token, 8 dims each; the groups' partial O summed in order at the
//   chunk's end).
// Online softmax in log2 units, as the matrix-core kernels; a split sequence's chunks go
// through the same workspace layout ([pair][row][chunk][D] and (max, sum)) and the combine
// launch.  Tokens in blocks the table marks invalid, and tokens a row does not see, get
// probability 0 (the V rows of invalid blocks are not read).
// NR rows per workgroup (a power of two up to AG_ROWS, the fewest that hold a pair's rows):
// the row loops are unrolled over NR, and rows past the pair's last are padding that sees
// no token.  With the row loops bounded at run time instead, the compiler walked the rows
// one at a time and re-read K and V per row; a cap of 16 rows cost a wave per SIMD (133
// registers) and measured slower than 8 on 32 and 512 rows per pair.
constexpr int AG_ROWS = 8;  // the launch switch instantiates 1, 2, 4 and 8
template <typename QT, typename KT, int NR>
__global__ void __launch_bounds__(256) attn_generic_kernel(AttnArgs a, int pairs, int ngroups) {
  extern __shared__ __attribute__((aligned(16))) float sm[];  // q rows [NR][DP], then p [NR][256]
  __shared__ float red[NR][4], redsum[NR][4];
  __shared__ int lims[NR];
  __shared__ int64_t offs[256];
  __shared__ float vred[2048];  // the token groups' partial O of one row: tp * D <= 2048
  const int D = a.D, DP = (D + 3) & ~3;
  float *qs = sm, *ps = sm + NR * DP;
  const int bid = blockIdx.x;
  const int chunk = bid % a.nchunk;
  const int grp = (bid / a.nchunk) % ngroups;
  const int p = bid / (a.nchunk * ngroups);
  if (p >= pairs) return;
  const int h = p % a.Hkv;
  const int r = (p / a.Hkv) % a.R;
  const int l = p / (a.Hkv * a.R);
  const int G = a.G;
  const int nq = attn_nq(a, r);
  const int row0 = grp * NR;
  if (row0 >= nq * G) return;
  const int nrows = min(NR, nq * G - row0);
  const int S_all = attn_seq_len(a, r);
  if (a.nchunk > 1 && chunk * a.tpc >= S_all) return;   // the combine reads only chunks with tokens
  const int c_begin = min(chunk * a.tpc, S_all);
  const int c_end = a.nchunk > 1 ? min(S_all, c_begin + a.tpc) : S_all;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  for (int i = tid; i < NR * DP; i += 256) {
    const int ri = i / DP, d = i % DP, row = row0 + ri;
    float v = 0.f;
    if (ri < nrows && d < D)
      v = (float)((const QT *)a.q)[(int64_t)l * a.q_sl + (int64_t)r * a.q_sr + (int64_t)(row / G) * a.q_sn +
                                   (int64_t)(h * G + row % G) * a.q_sh + d];
    qs[i] = v;
  }
  if (tid < NR) lims[tid] = tid < nrows ? min(attn_lim(a, r, (row0 + tid) / G, S_all), c_end) : c_begin;
  __syncthreads();
  int t_end = c_begin;  // the last token any row of the workgroup sees, plus one
  for (int i = 0; i < nrows; ++i) t_end = max(t_end, lims[i]);

  const KT *kplane = (const KT *)a.kv + (int64_t)l * a.kv_sl + (int64_t)h * a.kv_sh;
  const KT *vplane = kplane + a.kv_sv;
  const float c2 = a.scale * 1.4426950408889634f;
  // P.V mapping: tpt threads per token, each with DPT consecutive dims of its V row; tp tokens
  // in flight at a time, token j of a tile on thread group j mod tp
  constexpr int DPT = 8;
  const int tpt = (D + DPT - 1) / DPT, tp = 256 / tpt;
  const int vgrp = tid / tpt, dbase = (tid - vgrp * tpt) * DPT;
  const bool vact = vgrp < tp;
  float m2[NR], lsum[NR], acc[NR][DPT];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    m2[i] = -INFINITY;
    lsum[i] = 0.f;
#pragma unroll
    for (int e = 0; e < DPT; ++e) acc[i][e] = 0.f;
  }

  for (int t0 = c_begin; t0 < t_end; t0 += 256) {
    const int t = t0 + tid;
    int64_t off = -1;
    if (t < t_end) {
      const int ph = attn_phys(a, r, t / a.BS);
      if (ph >= 0) off = (int64_t)ph * a.kv_sb + (int64_t)(t % a.BS) * a.kv_ss;
    }
    offs[tid] = off;
    float x[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) x[i] = 0.f;
    if (off >= 0) {
      const KT *kr = kplane + off;
      int d = 0;
      // unrolled: several loads of the K row in flight per thread (bit-identical results;
      // 16 and 64 queries per pair 809 -> 549 and 907 -> 684 us, decode unchanged)
#pragma unroll 8
      for (; d + 4 <= D; d += 4) {
        const float k0 = (float)kr[d], k1 = (float)kr[d + 1], k2 = (float)kr[d + 2], k3 = (float)kr[d + 3];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const float4 qv = *(const float4 *)&qs[i * DP + d];
          x[i] = fmaf(k0, qv.x, x[i]);
          x[i] = fmaf(k1, qv.y, x[i]);
          x[i] = fmaf(k2, qv.z, x[i]);
          x[i] = fmaf(k3, qv.w, x[i]);
        }
      }
      for (; d < D; ++d) {
        const float k0 = (float)kr[d];
#pragma unroll
        for (int i = 0; i < NR; ++i) x[i] = fmaf(k0, qs[i * DP + d], x[i]);
      }
    }
    // scaled logits (log2 units), -inf where the row does not see the token; tile max per row
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      x[i] = off >= 0 && t < lims[i] ? x[i] * c2 : -INFINITY;   // padding rows see no token
      float mx = x[i];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      if (lane == 0) red[i][wave] = mx;
    }
    __syncthreads();
    float alpha[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const float tm = fmaxf(fmaxf(red[i][0], red[i][1]), fmaxf(red[i][2], red[i][3]));
      const float m_new = fmaxf(m2[i], tm);
      const float msafe = m_new == -INFINITY ? 0.f : m_new;
      alpha[i] = exp2f(m2[i] - msafe);
      m2[i] = m_new;
      const float pv = x[i] == -INFINITY ? 0.f : exp2f(x[i] - msafe);
      ps[i * 256 + tid] = pv;
      float sum = pv;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      if (lane == 0) redsum[i][wave] = sum;
    }
    __syncthreads();
    // l_i += the tile's sum of p (the same four wave sums, in order, in every thread);
    // O_i[d] += sum_j p_i,j v_j[d] over the thread's tokens j = vgrp, vgrp + tp, ...
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      lsum[i] = lsum[i] * alpha[i] + ((redsum[i][0] + redsum[i][1]) + (redsum[i][2] + redsum[i][3]));
#pragma unroll
      for (int e = 0; e < DPT; ++e) acc[i][e] *= alpha[i];
    }
    const int cnt = min(256, t_end - t0);
    if (vact) {
      for (int j = vgrp; j < cnt; j += tp) {
        const int64_t oj = offs[j];
        if (oj < 0) continue;  // a token of an invalid block: p = 0 in every row
        const KT *vr = vplane + oj + dbase;
        float v[DPT];
#pragma unroll
        for (int e = 0; e < DPT; ++e) v[e] = dbase + e < D ? (float)vr[e] : 0.f;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const float pj = ps[i * 256 + j];
#pragma unroll
          for (int e = 0; e < DPT; ++e) acc[i][e] = fmaf(pj, v[e], acc[i][e]);
        }
      }
    }
    __syncthreads();  // ps, offs and red are rewritten by the next tile
  }

  // each row: the token groups' partial O summed in group order through LDS, then written
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    if (i >= nrows) break;  // uniform
    __syncthreads();
    if (vact) {
#pragma unroll
      for (int e = 0; e < DPT; ++e)
        if (dbase + e < D) vred[vgrp * D + dbase + e] = acc[i][e];
    }
    __syncthreads();
    const int row = row0 + i, n = row / G, g = row % G;
    if (a.nchunk > 1) {
      const int64_t pr = ((int64_t)p * a.rows_pad + row) * a.nchunk + chunk;
      float *wo = a.ws_o + pr * D;
      for (int d = tid; d < D; d += 256) {
        float o = 0.f;
        for (int gi = 0; gi < tp; ++gi) o += vred[gi * D + d];
        wo[d] = o;
      }
      if (tid == 0) { a.ws_ml[pr * 2] = m2[i]; a.ws_ml[pr * 2 + 1] = lsum[i]; }
    } else {
      float *op = a.out + (int64_t)l * a.o_sl + (int64_t)r * a.o_sr + (int64_t)n * a.o_sn + (int64_t)(h * G + g) * a.o_sh;
      const float inv = lsum[i] > 0.f ? 1.0f / lsum[i] : 0.f;
      for (int d = tid; d < D; d += 256) {
        float o = 0.f;
        for (int gi = 0; gi < tp; ++gi) o += vred[gi * D + d];
        op[d] = o * inv;
      }
      if (tid == 0)
        a.lse[(int64_t)l * a.lse_sl + (int64_t)r * a.lse_sr + (int64_t)n * a.lse_sn + h * G + g] =
            lsum[i] > 0.f ? (m2[i] + __log2f(lsum[i])) * 0.6931471805599453f : -INFINITY;
    }
  }
}

// Waves of a ring workgroup for a pair with rtiles 32-row tiles of query rows.  (Two tiles per
// wave, each K and V^T fragment read once for 64 rows, need about 500 registers, one wave per
// SIMD, and measured 4.86 ms against 3.40 ms on 36 layers x 32k x 128 queries.)
static int ring_waves(int rtiles, int D) {
  if (rtiles == 1) return 1;   // head dim 256 only
  if (rtiles <= 2) return 2;
  if (rtiles <= 4 || D == 256) return 4;
  return 8;
}

struct AttnSplit { int nchunk, tpc, rows_pad, ngroups; };
// compute units of the current device (256 on MI355X), queried once per device
static int device_cus() {
  static int cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// Token chunks per pair of the ring path: the count with the least estimated time, from
//   rounds of resident workgroups x (a chunk's tokens + set-up)
//     + writing the chunks' partial results and merging them (4 TB/s, and a launch).
// Chunks hold at least 256 tokens.  Per-token times are a workgroup's, measured at the residency
// that the LDS stages and registers allow (one workgroup per CU at 8 waves and at 4 of head dim
// 256, else two).  Past three rounds the launch levels out and half a round is added instead of
// rounding up.  Against four rounds of workgroups whatever the shape, as before: 2048 causal
// queries over 6144 and 5003 tokens 677 -> 499 us (one chunk instead of two: 134 MB of partial
// results less, and the longest groups first), 1000 queries of a head-dim-64 model 568 -> 388,
// 300 queries over 20000 tokens 236 -> 180 (6 chunks instead of 26), 16 over 4 x 8k, 8 layers,
// 275 -> 240.
static int ring_chunks(int64_t items, int64_t rows, int tiles, int D, int span, int cus) {
  const int64_t slots = (int64_t)cus * (tiles >= 8 || (D == 256 && tiles >= 4) ? 1 : 2);
  const double us_token = D == 256 ? (tiles >= 4 ? 0.110 : 0.045) : D == 128 ? 0.048 : 0.038;
  const double us_setup = 4.0, us_merge = 4.0, us_per_row_chunk = 2.0 * (D + 2) * sizeof(float) / 4.0e6;
  const int most = std::max(1, span / 256);
  int best = 1;
  double best_us = 0.0;
  for (int c = 1; c <= most; ++c) {
    const double x = (double)items * c / (double)slots;
    const double rounds = x <= 3.0 ? std::ceil(x) : x + 0.5;
    double us = rounds * ((double)span / c * us_token + us_setup);
    if (c > 1) us += us_merge + (double)rows * c * us_per_row_chunk;
    if (c == 1 || us < best_us) { best_us = us; best = c; }
    if (x > 8.0) break;   // more chunks only add set-ups and partial results
  }
  return best;
}

static AttnSplit attn_split(int pairs, int N, int G, int D, int span, int cus) {
  AttnSplit sp;
  const int rtiles = (N * G + 31) / 32;
  if (rtiles == 1 && D != 256) {
    // decode kernel: DW waves per (pair, chunk), two resident workgroups per CU.  With few
    // pairs the chunks stop at about 1.5 workgroups per CU, within one round: a served decode
    // step's per-layer call (32 pairs x 4400 tokens) took 27.7 / 28.1 / 26.1 / 28.3 / 31.7 /
    // 33.7 us with 8 / 10 / 12 / 16 / 20 / 24 chunks, and 37 us with a second round (32).  With many pairs there are several rounds anyway, and at least 8 chunks per
    // pair keep the workgroups of the longest requests in a ragged batch from forming the
    // tail (a chunk holds at least one slice per wave: attn_dec_chunks).  From 16 rounds of
    // pairs on, the tail is a small part of the call and one pass per pair keeps the
    // workspace from growing with the batch (8 chunks of 256k pairs would want gigabytes).
    // The slices are interleaved over the chunks, so nothing depends on the block table's
    // width: the same sequences give the same bits however wide the table is.  Partial
    // results are kept for the N * G rows that exist.
    sp.ngroups = 1;
    sp.rows_pad = N * G;
    // Head dim 64: three workgroups per CU (152 registers; 169 allowed two) and at least 12
    // chunks: a decode step of 16 requests, 64 query heads, 74.9 -> 71.0 us (8 chunks 73.9, 6
    // 76.0), 8 layers of it 398 -> 388, 36 layers of 30000 tokens 429 -> 418.
    sp.nchunk = pairs >= 32 * cus ? 1 : std::max(D == 64 ? 12 : 8, 3 * cus / 2 / std::max(pairs, 1));
    sp.tpc = sp.nchunk > 1 ? 0 : std::max(span, 1);
    return sp;
  }
  const int tiles = ring_waves(rtiles, D);
  const int st = ring_stage(tiles, D);
  sp.ngroups = (rtiles + tiles - 1) / tiles;
  sp.rows_pad = N * G;   // only rows that exist are written and merged
  const int nchunk = ring_chunks((int64_t)pairs * sp.ngroups, (int64_t)pairs * sp.rows_pad, tiles, D, span, cus);
  int tpc = ((span + nchunk - 1) / nchunk + st - 1) / st * st;
  tpc = std::max(tpc, st);
  sp.nchunk = (span + tpc - 1) / tpc;
  sp.tpc = tpc;
  if (sp.nchunk <= 1) { sp.nchunk = 1; sp.tpc = std::max(span, 1); }
  return sp;
}

static size_t attn_ws_bytes(int pairs, const AttnSplit &sp, int D) {
  if (sp.nchunk <= 1) return 0;
  return (size_t)pairs * sp.rows_pad * sp.nchunk * (D + 2) * sizeof(float);
}

template <typename T, typename V8, int DH>
static int launch_attn_mfma(AttnArgs a, int bs_shift, void *ws, size_t ws_bytes, hipStream_t st) {
  const int pairs = a.L * a.R * a.Hkv;
  const int rtiles = (a.N * a.G + 31) / 32;
  const bool causal = a.kv_len != nullptr;
  AttnSplit sp = attn_split(pairs, a.N, a.G, DH, a.max_blocks * a.BS, device_cus());
  const size_t need = attn_ws_bytes(pairs, sp, DH);
  if (sp.nchunk > 1 && (!ws || ws_bytes < need)) {  // no (large enough) workspace: no split
    sp.nchunk = 1;
    sp.tpc = std::max(a.max_blocks * a.BS, 1);
  }
  a.nchunk = sp.nchunk; a.tpc = sp.tpc; a.rows_pad = sp.rows_pad;
  const bool decode = rtiles == 1 && DH != 256;
  a.dyn = decode && sp.nchunk > 1;
  a.ws_o = sp.nchunk > 1 ? (float *)ws : nullptr;
  a.ws_ml = sp.nchunk > 1 ? (float *)((char *)ws + (size_t)pairs * sp.rows_pad * sp.nchunk * DH * sizeof(float)) : nullptr;
  if (decode) {
    if constexpr (DH != 256) {
      const int grid = pairs * sp.nchunk;
      if (causal)
        hipLaunchKernelGGL((attn_decode_kernel<T, V8, DH, true>), dim3(grid), dim3(DW * 64), 0, st, a, pairs, bs_shift);
      else
        hipLaunchKernelGGL((attn_decode_kernel<T, V8, DH, false>), dim3(grid), dim3(DW * 64), 0, st, a, pairs, bs_shift);
    }
  } else {
#define ACTKV_ATTN(NWV)                                                                            \
  do {                                                                                             \
    const int grid = ((pairs + 7) / 8) * 8 * sp.ngroups * sp.nchunk;                               \
    if (causal)                                                                                    \
      hipLaunchKernelGGL((attn_ring_kernel<T, V8, DH, NWV, true>), dim3(grid), dim3(NWV * 64), \
                         0, st, a, pairs, sp.ngroups, bs_shift);                                   \
    else                                                                                           \
      hipLaunchKernelGGL((attn_ring_kernel<T, V8, DH, NWV, false>), dim3(grid), dim3(NWV * 64),\
                         0, st, a, pairs, sp.ngroups, bs_shift);                                   \
  } while (0)
  const int nw = ring_waves(rtiles, DH);
  if (nw == 2) {
    ACTKV_ATTN(2);
  } else if constexpr (DH == 256) {
    if (nw == 1) ACTKV_ATTN(1);
    else ACTKV_ATTN(4);
  } else {
    if (nw == 4) ACTKV_ATTN(4);
    else ACTKV_ATTN(8);
  }
#undef ACTKV_ATTN
  }
  int rc = actkv_check_launch();
  if (rc || sp.nchunk <= 1) return rc;
  const int64_t waves = (int64_t)pairs * sp.rows_pad;
  hipLaunchKernelGGL(attn_combine_kernel<DH>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a, pairs);
  return actkv_check_launch();
}

// Token split of the float32 path: about four workgroups per CU over the (pair, row group)
// items, chunks of a whole number of 256-token tiles.
// rows per workgroup of the float32 path: the fewest (a power of two, at most AG_ROWS) that
// hold a pair's N * G rows
static int attn_generic_rows(int N, int G) {
  const int64_t rows = (int64_t)N * G;
  int nr = 1;
  while (nr < AG_ROWS && nr < rows) nr *= 2;
  return nr;
}

static AttnSplit attn_split_generic(int pairs, int N, int G, int span, int cus) {
  AttnSplit sp;
  const int nr = attn_generic_rows(N, G);
  sp.ngroups = (int)(((int64_t)N * G + nr - 1) / nr);
  sp.rows_pad = sp.ngroups * nr;
  const int64_t items = (int64_t)pairs * sp.ngroups;
  const int64_t want = 4LL * cus;
  int nchunk = (int)std::min<int64_t>(std::max<int64_t>(1, (want + items - 1) / items), std::max(1, span / 256));
  int tpc = ((span + nchunk - 1) / nchunk + 255) / 256 * 256;
  tpc = std::max(tpc, 256);
  sp.nchunk = (span + tpc - 1) / tpc;
  sp.tpc = tpc;
  if (sp.nchunk <= 1) { sp.nchunk = 1; sp.tpc = std::max(span, 1); }
  return sp;
}

template <typename QT, typename KT>
static int launch_attn_generic(AttnArgs a, void *ws, size_t ws_bytes, hipStream_t st) {
  const int64_t pairs64 = (int64_t)a.L * a.R * a.Hkv;
  const int nr = attn_generic_rows(a.N, a.G);
  const int64_t groups = ((int64_t)a.N * a.G + nr - 1) / nr;
  if (pairs64 * groups > 0x7fffffffLL) return ACTKV_ERR_UNSUPPORTED;
  const int pairs = (int)pairs64;
  AttnSplit sp = attn_split_generic(pairs, a.N, a.G, a.max_blocks * a.BS, device_cus());
  const size_t need = attn_ws_bytes(pairs, sp, a.D);
  if (sp.nchunk > 1 && (!ws || ws_bytes < need || (int64_t)pairs * sp.ngroups * sp.nchunk > 0x7fffffffLL)) {
    sp.nchunk = 1;
    sp.tpc = std::max(a.max_blocks * a.BS, 1);
  }
  a.nchunk = sp.nchunk; a.tpc = sp.tpc; a.rows_pad = sp.rows_pad; a.dyn = 0;
  a.ws_o = sp.nchunk > 1 ? (float *)ws : nullptr;
  a.ws_ml = sp.nchunk > 1 ? (float *)((char *)ws + (size_t)pairs * sp.rows_pad * sp.nchunk * a.D * sizeof(float)) : nullptr;
  const size_t shm = (size_t)nr * (((a.D + 3) & ~3) + 256) * sizeof(float);
  const dim3 grid((unsigned)((int64_t)pairs * sp.ngroups * sp.nchunk));
#define ACTKV_AG(NRV) hipLaunchKernelGGL((attn_generic_kernel<QT, KT, NRV>), grid, dim3(256), shm, st, a, pairs, sp.ngroups)
  switch (nr) {
    case 1: ACTKV_AG(1); break;
    case 2: ACTKV_AG(2); break;
    case 4: ACTKV_AG(4); break;
    default: ACTKV_AG(8); break;   // AG_ROWS
  }
#undef ACTKV_AG
  int rc = actkv_check_launch();
  if (rc || sp.nchunk <= 1) return rc;
  const int64_t waves = (int64_t)pairs * sp.rows_pad;
  hipLaunchKernelGGL(attn_combine_kernel<0>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a, pairs);
  return actkv_check_launch();
}

template <typename QT>
static int dispatch_attn_generic(const AttnArgs &a, int kv_dtype, void *ws, size_t wb, hipStream_t st) {
  switch (kv_dtype) {
    case ACTKV_F32: return launch_attn_generic<QT, float>(a, ws, wb, st);
    case ACTKV_F16: return launch_attn_generic<QT, _Float16>(a, ws, wb, st);
    case ACTKV_BF16: return launch_attn_generic<QT, __bf16>(a, ws, wb, st);
  }
  return ACTKV_ERR_INVALID_ARG;
}

static bool attn_aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace actkv

using namespace actkv;

extern "C" int actkv_paged_attention(
    const void *q, int q_dtype, int64_t q_sl, int64_t q_sr, int64_t q_sn, int64_t q_sh,
    const void *kv, int kv_dtype, int64_t kv_sl, int64_t kv_sv, int64_t kv_sb, int64_t kv_ss,
    int64_t kv_sh, int64_t num_blocks, const int32_t *block_table, int64_t bt_sr, int max_blocks,
    const int32_t *seq_used, const int32_t *n_valid, const int32_t *kv_len, float *out,
    int64_t o_sl, int64_t o_sr, int64_t o_sn, int64_t o_sh, float *lse, int64_t lse_sl,
    int64_t lse_sr, int64_t lse_sn, int L, int R, int N, int Hq, int Hkv, int D, int block_size,
    float scale, void *workspace, size_t workspace_bytes, void *stream) {
  if (!q || !kv || !block_table || !seq_used || !out || !lse) return ACTKV_ERR_INVALID_ARG;
  if (L < 1 || R < 1 || N < 0 || Hq < 1 || Hkv < 1 || D < 1 || block_size < 1 || max_blocks < 1 ||
      num_blocks < 1)
    return ACTKV_ERR_INVALID_ARG;
  if (Hq % Hkv != 0 || !(scale > 0.f)) return ACTKV_ERR_INVALID_ARG;
  if (dtype_size(q_dtype) == 0 || dtype_size(kv_dtype) == 0) return ACTKV_ERR_INVALID_ARG;
  if ((int64_t)max_blocks * block_size > 0x7fffffffLL || D > 512) return ACTKV_ERR_UNSUPPORTED;
  if (N == 0) return ACTKV_OK;
  hipStream_t st = (hipStream_t)stream;
  AttnArgs a;
  a.q = q; a.q_sl = q_sl; a.q_sr = q_sr; a.q_sn = q_sn; a.q_sh = q_sh;
  a.kv = kv; a.kv_sl = kv_sl; a.kv_sv = kv_sv; a.kv_sb = kv_sb; a.kv_ss = kv_ss; a.kv_sh = kv_sh;
  a.num_blocks = num_blocks;
  a.bt = block_table; a.bt_sr = bt_sr; a.max_blocks = max_blocks;
  a.seq_used = seq_used; a.n_valid = n_valid; a.kv_len = kv_len;
  a.out = out; a.o_sl = o_sl; a.o_sr = o_sr; a.o_sn = o_sn; a.o_sh = o_sh;
  a.lse = lse; a.lse_sl = lse_sl; a.lse_sr = lse_sr; a.lse_sn = lse_sn;
  a.L = L; a.R = R; a.N = N; a.Hq = Hq; a.Hkv = Hkv; a.D = D; a.G = Hq / Hkv; a.BS = block_size;
  a.scale = scale;
  a.nchunk = 1; a.tpc = max_blocks * block_size; a.rows_pad = 0; a.dyn = 0;
  a.ws_o = nullptr; a.ws_ml = nullptr;
  const int G = a.G;
  int bs_shift = -1;
  for (int sh = 4; sh < 31; ++sh)
    if (block_size == (1 << sh)) bs_shift = sh;
  const bool vec_ok = attn_aligned16(q) && attn_aligned16(kv) && attn_aligned16(out) &&
                      q_sl % 8 == 0 && q_sr % 8 == 0 && q_sn % 8 == 0 && q_sh % 8 == 0 &&
                      kv_sl % 8 == 0 && kv_sv % 8 == 0 && kv_sb % 8 == 0 && kv_ss % 8 == 0 &&
                      kv_sh % 8 == 0 && o_sl % 4 == 0 && o_sr % 4 == 0 && o_sn % 4 == 0 && o_sh % 4 == 0;
  const bool mfma_ok = q_dtype == kv_dtype && (kv_dtype == ACTKV_BF16 || kv_dtype == ACTKV_F16) &&
                       (D == 256 || D == 128 || D == 64) && G >= 1 && vec_ok && bs_shift >= 0 &&
                       (int64_t)block_size * kv_ss <= 0x7fffffffLL;   // byte offsets in a block: 32 bits
  if (mfma_ok) {
    void *ws = workspace;
    const size_t wb = workspace_bytes;
    if (kv_dtype == ACTKV_BF16)
      return D == 64    ? launch_attn_mfma<__bf16, bf16x8, 64>(a, bs_shift, ws, wb, st)
             : D == 128 ? launch_attn_mfma<__bf16, bf16x8, 128>(a, bs_shift, ws, wb, st)
                        : launch_attn_mfma<__bf16, bf16x8, 256>(a, bs_shift, ws, wb, st);
    return D == 64    ? launch_attn_mfma<_Float16, f16x8, 64>(a, bs_shift, ws, wb, st)
           : D == 128 ? launch_attn_mfma<_Float16, f16x8, 128>(a, bs_shift, ws, wb, st)
                      : launch_attn_mfma<_Float16, f16x8, 256>(a, bs_shift, ws, wb, st);
  }
  switch (q_dtype) {
    case ACTKV_F32: return dispatch_attn_generic<float>(a, kv_dtype, workspace, workspace_bytes, st);
    case ACTKV_F16: return dispatch_attn_generic<_Float16>(a, kv_dtype, workspace, workspace_bytes, st);
    default: return dispatch_attn_generic<__bf16>(a, kv_dtype, workspace, workspace_bytes, st);
  }
}

extern "C" size_t actkv_paged_attention_workspace_size(int L, int R, int N, int Hq, int Hkv, int D,
                                                       int max_blocks, int block_size) {
  if (L < 1 || R < 1 || N < 1 || Hkv < 1 || Hq % Hkv != 0 || max_blocks < 1 || block_size < 1) return 0;
  const int G = Hq / Hkv;
  if (G < 1 || D > 512) return 0;
  if ((int64_t)max_blocks * block_size > 0x7fffffffLL) return 0;
  const int pairs = L * R * Hkv;
  // head dims 256, 128 and 64 take the matrix-core split or, with a dtype or block size off that
  // path, the float32 path's: room for either
  const size_t gen = attn_ws_bytes(pairs, attn_split_generic(pairs, N, G, max_blocks * block_size, device_cus()), D);
  if (D != 256 && D != 128 && D != 64) return gen;
  return std::max(gen, attn_ws_bytes(pairs, attn_split(pairs, N, G, D, max_blocks * block_size, device_cus()), D));
}
