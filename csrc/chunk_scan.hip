// Chunk-parallel form of the recurrences: whole chunks of 16 tokens (32 in ssd
// and mlstm of bf16 rows, at the wide kernels below) go through matrix products
// instead of one token at a time. Per head the state S is a D x DV fp32 matrix and every token does
//
//   general delta  w = exp(-scale sigmoid(zw + w0)), a = sigmoid(za + ab),
//                  u = k / sqrt(sum k^2 + 1e-6)
//                  S <- diag(w) S - (a u)(u^T S) + k v^T,   o = S^T r
//   channel delta  w = exp(-exp(a_log) softplus(z + dt_bias)), k^, q^ unit
//                  vectors (q^ times qscale), b = sigmoid(beta)
//                  S <- diag(w) S;  S <- S + b k^ (v - S^T k^)^T, o = S^T q^
//   gla            w = sigmoid(z + p0)^c0
//                  S <- diag(w) S + k v^T,                  o = S^T (q qscale)
//   ssd, mlstm     one decay a and write scale w per head and token
//                  S <- a S + w k v^T,                      o = S^T (q qscale)
//
// Let W_t be the product of the decays of a chunk's tokens up to t, per key
// channel, and Z_t = (what token t reads of the state before its own write).
// Then for the chunk, S0 being the state before it,
//
//   general  (I - Bm) Z = U S0 + Km V,   Bm_ts = u_t W_{t-1}/W_s b_s  (s < t)
//            with b = -a u, U_t = u_t W_{t-1}, Km likewise with k_s
//            O = R S0 + Mb Z + Mk V,     R_t = r_t W_t, Mb_ts = r_t W_t/W_s b_s
//            S = diag(W_C) S0 + B^T Z + K^T V,  B_s = b_s W_C/W_s, K_s likewise
//   channel  (I + A) Y = V - U S0,       Y = V - Z, U_t = k_t W_t,
//            A_ts = k_t W_t/W_s b_s k_s  (s < t);  O = R S0 + M Y,
//            S = diag(W_C) S0 + K^T Y
//   gla      O = R S0 + M V,  S = diag(W_C) S0 + K^T V
//   scalar   O = diag(W) Q S0 + M V,  M_ts = q_t k_s W_t/W_s w_s (s <= t)
//            S = W_C S0 + K^T diag(w W_C/W) V, Q and K as they are, shared by
//            the heads of a group; every ratio is a product of its own
//
// Everything but the state is known ahead, so it is laid down by one fully
// parallel kernel (one workgroup per chunk and head: the decays' products,
// the 16 x 16 matrices, the triangular solve), and a second kernel walks the
// chunks with the state in registers: a wave owns 16 columns of S as D / 16
// accumulator tiles of v_mfma_f32_16x16x4_f32 (or shares its rows with others).
// The tiles' register layout (row 4 g + i of a tile in lane group g, register i)
// is at once the layout of the right operand of the products that read S when
// the left operand's columns are taken in the order 4 g + i, so the state never
// leaves its registers; Z and Y pass from one product into the next the same
// way.
//
// Arithmetic is fp32 throughout (the matrix unit's fp32 products: fp32 inputs,
// fp32 accumulation; the chunks of 32 multiply bf16 rows as they are by fp32
// numbers cut without loss into three bf16 terms). Ratios W_t / W_s are formed from products counted from
// the middle of the chunk, so both factors stay in range while either half's
// product is above 1e-30; chunks beyond that (or with decays that are no
// numbers) form every ratio on its own.
//
// One token at a time is a chain of two dot products and two lane reductions
// per token on D x DV lanes; measured at 32 heads of 128 x 128, 8011 tokens in
// two prompts: 12.3 ms, 1.5 us a token. Figures of this form stand at the
// launcher.
#include "scan_common.h"

// Float4 slots of a chunk's operands. Left operands whose rows are tokens:
// lane (g, m) of tile t reads channels 16 t + 4 g .. + 3 of token m. The
// token index is twisted so that writing one token's channels spreads over
// all LDS banks.
PS_DEV int ck_row_slot(int t, int g, int m) {
  return t * 64 + g * 16 + (m ^ ((t * 4 + g) & 15));
}
// Left operands whose rows are channels: lane (g, m) reads tokens 4 g .. + 3
// of channel 16 t + m.
PS_DEV int ck_col_slot(int t, int g, int m) { return t * 64 + g * 16 + m; }

// Floats of one chunk's operands and where each lies.
template <int MODE, int DP>
struct CkItem {
  static constexpr int ROW = 16 * DP;  // one 16 x DP operand
  static constexpr int R = 0;
  static constexpr int K = ROW;
  static constexpr int U = 2 * ROW;                        // delta forms
  static constexpr int B = 3 * ROW;                        // general delta
  static constexpr int NROW = MODE == CK_GD ? 4 : (MODE == CK_CD ? 3 : 2);
  static constexpr int M = NROW * ROW;                     // on V (Y)
  static constexpr int C = M + 256;                        // solve on V
  static constexpr int MB = C + 256;                       // on Z
  static constexpr int NSQ = MODE == CK_GD ? 3 : (MODE == CK_CD ? 2 : 1);
  static constexpr int GAM = M + NSQ * 256;                // [DP]
  static constexpr int FLAG = GAM + DP;  // not 0: an input is no finite number
  static constexpr int TOTAL = FLAG + 4;
};

// Chunks of a segment of n rows (segments shorter than 16 rows are not this
// kernel's). The chunks of all segments, one segment after the other, are the
// items; a pass takes `cap` of them from `base` on.
template <int L = 16>
PS_DEV int ck_count(int n) {
  return n < 16 ? 0 : (n + L - 1) / L;
}

// Which chunk of which segment an item is; false past the last one. Every wave
// of a block finds the same.
template <int L = 16>
PS_DEV bool ck_find(const int* seq_rows, int S_, int item, int lane, int* seg,
                    int* chunk) {
  int base = 0;
  for (int s0 = 0; s0 < S_; s0 += 64) {
    const int s = s0 + lane;
    const int cnt = s < S_ ? ck_count<L>(seq_rows[4 * s + 1]) : 0;
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off, 64);
      if (lane >= off) incl += up;
    }
    const int first = base + incl - cnt;
    const unsigned long long hit =
        __ballot(cnt > 0 && item >= first && item < first + cnt);
    if (hit) {
      const int l = __ffsll((long long)hit) - 1;
      *seg = s0 + l;
      *chunk = item - __builtin_amdgcn_readlane(first, l);
      return true;
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  return false;
}

// A segment's row of seq_rows and its first chunk among those of all.
struct CkSeg {
  int seg, t0, n, p0, slot, first;
};

// The segment that `rank` others are longer than (of equal ones the first), seg
// -1 where there is none or it has no chunks. Workgroups start in the order of
// their numbers, so the longest walks start first, and the CU of one takes a
// shorter one beside it: general delta, 32 heads, prompts of 336 and 166 chunks,
// 0.60 -> 0.47 ms. Up to 64 segments every lane asks for one's row: one trip to
// memory before the walk's own. Segments too short for a chunk (single tokens
// beside prompts) cost no turn: channel delta, 32 heads, 6007 rows in 3 prompts
// beside 37 tokens, 549 us ordered, 565 as they come. Past 32 with chunks, or 64
// in all, they go as they come: a turn a segment in each of many short workgroups
// is more than the order gives. us, ordered / as they come: general delta, 32 fp32
// heads of 96 x 96, 1200 rows in 40 prompts 188 / 161, 3000 in 40 333 / 307, of
// 64 x 64, 6000 in 60 364 / 343; 8 heads of 64 x 64, 8000 in 40 114 / 120.
template <int L = 16>
PS_DEV CkSeg ck_by_length(const int* seq_rows, int S_, int rank) {
  const int lane = threadIdx.x & 63;
  CkSeg at;
  int before = 0;
  at.seg = rank;
  if (S_ == 1 || S_ > 64) {
    at.t0 = seq_rows[4 * rank], at.n = seq_rows[4 * rank + 1];
    if (ck_count<L>(at.n) == 0) {
      at.seg = -1;
      return at;
    }
    at.p0 = seq_rows[4 * rank + 2], at.slot = seq_rows[4 * rank + 3];
    for (int s = lane; s < rank; s += 64)
      before += ck_count<L>(seq_rows[4 * s + 1]);
  } else {
    const int* own = seq_rows + 4 * min(lane, S_ - 1);
    const int t0 = own[0], n = lane < S_ ? own[1] : 0, p0 = own[2],
              slot = own[3];
    const unsigned long long live = __ballot(ck_count<L>(n) > 0);
    const int count = __popcll(live);
    if (count <= 32) {
      if (rank >= count) {
        at.seg = -1;
        return at;
      }
      int longer = 0;
      for (unsigned long long left = live; left; left &= left - 1) {
        const int s = __ffsll(left) - 1;
        const int other = __builtin_amdgcn_readlane(n, s);
        longer += other > n || (other == n && s < lane);
      }
      at.seg = __ffsll((unsigned long long)__ballot(longer == rank) & live) - 1;
    } else if ((live >> rank & 1) == 0) {
      at.seg = -1;
      return at;
    }
    at.t0 = __builtin_amdgcn_readlane(t0, at.seg);
    at.n = __builtin_amdgcn_readlane(n, at.seg);
    at.p0 = __builtin_amdgcn_readlane(p0, at.seg);
    at.slot = __builtin_amdgcn_readlane(slot, at.seg);
    before = lane < at.seg ? ck_count<L>(n) : 0;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  at.first = __builtin_amdgcn_readfirstlane(before);
  return at;
}

// Sums of eight values over the wave: lanes 8 e .. 8 e + 7 return that of x[e].
// Every step of the first three adds two halves of the lanes and keeps half of the
// values in each, so that ten exchanges take the place of 48 one after the other.
PS_DEV float ck_wave_sums(const float (&x)[8]) {
  const int lane = threadIdx.x & 63;
  float a[4], b[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool up = lane & 32;
    a[i] = (up ? x[4 + i] : x[i]) + __shfl_xor(up ? x[i] : x[4 + i], 32, 64);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool up = lane & 16;
    b[i] = (up ? a[2 + i] : a[i]) + __shfl_xor(up ? a[i] : a[2 + i], 16, 64);
  }
  const bool up = lane & 8;
  float s = (up ? b[1] : b[0]) + __shfl_xor(up ? b[0] : b[1], 8, 64);
#pragma unroll
  for (int d = 4; d > 0; d >>= 1) s += __shfl_xor(s, d, 64);
  return s;
}

// Lays down a chunk's operands: a workgroup per (chunk, head), a lane per channel
// of eight rows. Bound by its vector instructions (1100 a wave for the general
// delta, three waves a SIMD: registers), beside a write of 32 KB. Four workgroups a
// CU spill for the channel delta (480 -> 500 us of its whole operation).
template <typename T, int MODE, int DP>
__global__ __launch_bounds__(256, MODE == CK_GLA ? 4 : 3) void ck_prep_kernel(
    float* __restrict__ items, CkIn in, const int* __restrict__ seq_rows,
    int S_, int H, int G, int D, float scale, float c0f, int base) {
  typedef CkItem<MODE, DP> It;
  constexpr int LD = DP + 4;
  // operand rows in channel order; reused for the fragments that are not stored
  // from registers (rows R and U, then what lies behind the rows) once the
  // 16 x 16 products are done
  constexpr int ROWS = MODE == CK_GD ? 4 : (MODE == CK_CD ? 3 : 2);
  constexpr int SU = It::ROW, SO = (MODE == CK_GLA ? 1 : 2) * It::ROW - It::M;
  __shared__ __align__(16) float stage[
      It::TOTAL + SO > ROWS * 16 * LD ? It::TOTAL + SO : ROWS * 16 * LD];
  __shared__ __align__(16) float su[MODE == CK_GLA ? 4 : 16 * LD];
  __shared__ __align__(16) float sm[4][16][20];
  __shared__ float red[2][16][2];
  __shared__ float half_prod[2][128];
  float* X1 = stage;              // rows that read the state for the output
  float* Y1 = X1 + 16 * LD;       // columns written with V
  float* X0 = Y1 + 16 * LD;       // rows that read it for Z
  float* Y0 = X0 + 16 * LD;       // columns written with Z

  // which chunk of which segment
  const int item = blockIdx.x, hd = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int seg, chunk;
  if (!ck_find(seq_rows, S_, base + item, lane, &seg, &chunk)) return;
  // the same in all lanes: rows' addresses are a scalar and one offset per lane,
  // and what depends on the half a branch
  seg = __builtin_amdgcn_readfirstlane(seg);
  chunk = __builtin_amdgcn_readfirstlane(chunk);
  const int n = seq_rows[4 * seg + 1];
  const int row0 = seq_rows[4 * seg] + 16 * chunk;
  const int nv = min(16, n - 16 * chunk);

  const int half = wave >> 1, d = threadIdx.x & 127;
  const bool on = d < DP, real = d < D;
  const int grp = hd / (H / G);

  // all loads ahead of any use, from a row and a channel that exist
  const int dc = real ? d : 0;
  const unsigned at_c = dc * sizeof(T);
  const size_t h0 = (size_t)hd * D;
  const size_t k0 = MODE == CK_GD ? h0 : (size_t)grp * D;
  auto get = [&](const void* p, size_t row, int ld, size_t c, unsigned at) {
    return MxElem<T>::ld(
        (const T*)((const char*)((const T*)p + row * ld + c) + at));
  };
  float kv[8], rv[8], wv[8], av[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const size_t row = (size_t)(row0 + min(half * 8 + e, nv - 1));
    kv[e] = get(in.k, row, in.ldk, k0, at_c);
    rv[e] = get(in.q, row, in.ldq, k0, at_c);
    wv[e] = get(in.dec, row, in.lddec, h0, at_c);
    av[e] = 0.f;
    if (MODE == CK_GD) av[e] = get(in.a, row, in.lda, h0, at_c);
  }
  // one number per row: each of eight lanes has one, and all take it from there
  float ar = 0.f;
  if (MODE == CK_CD)
    ar = get(in.a, row0 + min(half * 8 + (lane & 7), nv - 1), in.lda, hd, 0);
  const float c0z = in.p0[h0 + dc];
  float c1 = 0.f;
  if (MODE == CK_GD) c1 = in.p1[h0 + dc];
  if (MODE == CK_CD) c1 = expf(in.p1[hd]);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (MODE == CK_GD) {
      wv[e] = ck_exp(-scale * ck_sigmoid(wv[e] + c0z));
      av[e] = ck_sigmoid(av[e] + c1);
    } else if (MODE == CK_CD) {
      wv[e] = ck_exp(-c1 * ck_softplus(wv[e] + c0z));
    } else {
      wv[e] = ck_exp(ck_log_sigmoid(wv[e] + c0z) * c0f);
    }
  }
  if (MODE == CK_CD) {
    ar = half * 8 + (lane & 7) < nv ? ck_sigmoid(ar) : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      av[e] = __uint_as_float(
          __builtin_amdgcn_readlane(__float_as_uint(ar), e));
  }
  // rows past the segment's end and channels past the head's change nothing
  if (DP != 128 || D != DP || nv != 16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool live = real && half * 8 + e < nv;
      wv[e] = live ? wv[e] : 1.f;
      if (!live) kv[e] = rv[e] = 0.f;
      if (MODE == CK_GD && !live) av[e] = 0.f;
    }
  }

  // unit vectors
  if (MODE != CK_GLA) {
    float sq[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sq[e] = kv[e] * kv[e];
    const float k2 = ck_wave_sums(sq);
    float r2 = 0.f;
    if (MODE == CK_CD) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sq[e] = rv[e] * rv[e];
      r2 = ck_wave_sums(sq);
    }
    if ((lane & 7) == 0) {
      red[0][half * 8 + (lane >> 3)][wave & 1] = k2;
      red[1][half * 8 + (lane >> 3)][wave & 1] = r2;
    }
  }
  // products of the decays within the half
  float pin[8];   // up to and with token e, from the half's first
  float suf[8];   // of the tokens behind e, to the half's last
  {
    float p = 1.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p *= wv[e];
      pin[e] = p;
    }
    float s = 1.f;
#pragma unroll
    for (int e = 7; e >= 0; --e) {
      suf[e] = s;
      s *= wv[e];
    }
  }
  half_prod[half][d] = pin[7];
  float mag = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    mag += fabsf(kv[e]) + fabsf(rv[e]) + fabsf(wv[e]) + fabsf(av[e]);
  const bool odd = __syncthreads_or(!(mag < INFINITY));
  // out of range (or no number): ratios are formed one by one
  const bool slow = __builtin_amdgcn_readfirstlane(
      __syncthreads_or(on && !(pin[7] > 1e-30f && pin[7] < 1e30f)));
  const float other = half_prod[half ^ 1][d];

  float uv[8], bv[8];  // u (GD) / k^ (CD); b
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int tt = half * 8 + e;
    uv[e] = bv[e] = 0.f;
    if (MODE == CK_GD) {
      const float ik = ck_rsqrt(red[0][tt][0] + red[0][tt][1] + 1e-6f);
      uv[e] = kv[e] * ik;
      bv[e] = -av[e] * uv[e];
    } else if (MODE == CK_CD) {
      const float ik = ck_rsqrt(red[0][tt][0] + red[0][tt][1] + 1e-6f);
      const float iq = scale * ck_rsqrt(red[1][tt][0] + red[1][tt][1] + 1e-6f);
      uv[e] = kv[e] * ik;
      kv[e] = av[e] * uv[e];
      rv[e] *= iq;
    } else {
      rv[e] *= scale;
    }
  }

  if (on) {
    // operand rows of token e: wt, iw W_t counted from the middle (W_7 = 1) and
    // its inverse; general delta's reading rows take W_{t-1} (wp)
    auto put = [&](int e, float wt, float iw, float wp) {
      const int at = (half * 8 + e) * LD + d;
      if (MODE == CK_GD) X0[at] = uv[e] * wp;
      if (MODE == CK_CD) X0[at] = uv[e] * wt;
      X1[at] = rv[e] * wt;
      if (MODE == CK_GD) Y0[at] = bv[e] * iw;
      Y1[at] = kv[e] * iw;
    };
    // what reads the state before the chunk: products from its start
    auto reads = [&](int e, float before, float to) {
      if (MODE == CK_GD) su[(half * 8 + e) * LD + d] = uv[e] * before;
      if (MODE == CK_CD) su[(half * 8 + e) * LD + d] = uv[e] * to;
    };
    if (half == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        reads(e, e > 0 ? pin[e > 0 ? e - 1 : 0] : 1.f, pin[e]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        reads(e, e > 0 ? other * pin[e > 0 ? e - 1 : 0] : other,
              other * pin[e]);
    }
    if (slow) {
#pragma unroll
      for (int e = 0; e < 8; ++e) put(e, 1.f, 1.f, 1.f);
    } else if (half == 0) {
      float before = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float inv = ck_rcp(suf[e]);
        put(e, inv, suf[e], before);
        before = inv;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        put(e, pin[e], ck_rcp(pin[e]), e > 0 ? pin[e > 0 ? e - 1 : 0] : 1.f);
    }
  }
  __syncthreads();

  // the 16 x 16 products, one per wave: C[t][s], t in rows
  const int g = lane >> 4, m16 = lane & 15;
  if (!slow) {
    const float* xa = nullptr;
    const float* yb = nullptr;
    if (MODE == CK_GD) {
      xa = wave < 2 ? X0 : X1;
      yb = (wave & 1) ? Y1 : Y0;
    } else if (MODE == CK_CD) {
      if (wave < 2) {
        xa = wave == 0 ? X0 : X1;
        yb = Y1;
      }
    } else if (wave == 0) {
      xa = X1;
      yb = Y1;
    }
    if (xa != nullptr) {
      ck_f32x4 c = {0.f, 0.f, 0.f, 0.f}, c2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < DP / 16; ++t) {
        const ck_f32x4 x = *(const ck_f32x4*)(xa + m16 * LD + t * 16 + g * 4);
        const ck_f32x4 y = *(const ck_f32x4*)(yb + m16 * LD + t * 16 + g * 4);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[0], y[0], c, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[1], y[1], c2, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[2], y[2], c, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[3], y[3], c2, 0, 0, 0);
      }
      const bool strict = xa == X0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 4 * g + i;
        const bool seen = strict ? t > m16 : t >= m16;
        sm[wave][t][m16] = seen ? c[i] + c2[i] : 0.f;
      }
    }
    __syncthreads();
  } else {
    // every ratio on its own: thread (t, s) multiplies the decays between
    // its two tokens, channel by channel
    float* sw = &sm[0][0][0];  // 16 x 16 decays of one channel tile
    const int t = threadIdx.x >> 4, s = threadIdx.x & 15;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int d0 = 0; d0 < DP; d0 += 16) {
      __syncthreads();
      if (on && d >= d0 && d < d0 + 16) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          sw[(half * 8 + e) * 17 + d - d0] = wv[e];
      }
      __syncthreads();
      for (int i = 0; i < 16; ++i) {
        float ez = 1.f;  // behind s, up to t - 1
        for (int jj = s + 1; jj < t; ++jj) ez *= sw[jj * 17 + i];
        const float er = t > s ? ez * sw[t * 17 + i] : 1.f;
        const float y1 = Y1[s * LD + d0 + i];
        if (MODE == CK_GD) {
          const float y0 = Y0[s * LD + d0 + i], x0 = X0[t * LD + d0 + i];
          acc[0] += x0 * ez * y0;
          acc[1] += x0 * ez * y1;
          acc[2] += X1[t * LD + d0 + i] * er * y0;
          acc[3] += X1[t * LD + d0 + i] * er * y1;
        } else {
          if (MODE == CK_CD) acc[0] += X0[t * LD + d0 + i] * er * y1;
          acc[MODE == CK_CD ? 1 : 0] += X1[t * LD + d0 + i] * er * y1;
        }
      }
    }
    __syncthreads();
    constexpr int STRICT = MODE == CK_GD ? 2 : (MODE == CK_CD ? 1 : 0);
#pragma unroll
    for (int w = 0; w < 4; ++w)
      sm[w][t][s] = (w < STRICT ? t > s : t >= s) ? acc[w] : 0.f;
    __syncthreads();
  }

  // Fragments over the operand rows, which nothing reads any more; those of 16
  // bytes go to memory at once, on their way during the substitution.
  float* dst = items + ((size_t)item * H + hd) * It::TOTAL;
  constexpr int LAST = MODE == CK_GD ? 3 : (MODE == CK_CD ? 1 : 0);
  if (on) {
    const int t = d >> 4, dg = (d & 15) >> 2, di = d & 3;
    float kf[8], bf[8];
    auto scaled = [&](int e, float from, float to) {
      stage[ck_row_slot(t, dg, half * 8 + e) * 4 + di] = rv[e] * from;
      kf[e] = kv[e] * to;
      bf[e] = bv[e] * to;
    };
    if (half == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) scaled(e, pin[e], suf[e] * other);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) scaled(e, other * pin[e], suf[e]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = ck_col_slot(t, half * 2 + h, d & 15) * 4;
      *(ck_f32x4*)(dst + It::K + at) =
          ck_f32x4{kf[4 * h], kf[4 * h + 1], kf[4 * h + 2], kf[4 * h + 3]};
      if (MODE == CK_GD)
        *(ck_f32x4*)(dst + It::B + at) =
            ck_f32x4{bf[4 * h], bf[4 * h + 1], bf[4 * h + 2], bf[4 * h + 3]};
    }
    if (half == 0) stage[SO + It::GAM + d] = pin[7] * other;
    if (threadIdx.x < 4) stage[SO + It::FLAG + threadIdx.x] = odd ? 1.f : 0.f;
  }
  if (wave == 3)
    *(ck_f32x4*)(stage + SO + It::M + lane * 4) =
        *(const ck_f32x4*)(&sm[LAST][m16][g * 4]);
  if (MODE == CK_GD && wave == 2)
    *(ck_f32x4*)(stage + SO + It::MB + lane * 4) =
        *(const ck_f32x4*)(&sm[2][m16][g * 4]);
  if (MODE != CK_GLA) {
    // forward substitution, one thread per column of [U | Km] (general) or
    // [U | I] (channel)
    const int col = threadIdx.x;
    if (col < DP + 16) {
      float x[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        float b;
        if (col < DP)
          b = su[t * LD + col];
        else if (MODE == CK_GD)
          b = sm[1][t][col - DP];
        else
          b = t == col - DP ? 1.f : 0.f;
#pragma unroll
        for (int s4 = 0; s4 < (t + 3) / 4; ++s4) {
          const ck_f32x4 r4 = *(const ck_f32x4*)(&sm[0][t][s4 * 4]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int s = s4 * 4 + i;
            if (s < t) b += (MODE == CK_GD ? r4[i] : -r4[i]) * x[s];
          }
        }
        x[t] = b;
      }
      if (col < DP) {
        const int t = col >> 4, dg = (col & 15) >> 2, di = col & 3;
#pragma unroll
        for (int tt = 0; tt < 16; ++tt)
          stage[SU + ck_row_slot(t, dg, tt) * 4 + di] = x[tt];
      } else {
        const int s = col - DP;
#pragma unroll
        for (int tt = 0; tt < 16; ++tt)
          stage[SO + It::C + ((s >> 2) * 16 + tt) * 4 + (s & 3)] = x[tt];
      }
    }
  }
  __syncthreads();
  auto copy = [&](int from, int to, int shift) {
#pragma unroll
    for (int i = from / 4; i < to / 4; i += 256) {
      const int at = i + threadIdx.x;
      if (at < to / 4)
        *(ck_f32x4*)(dst + at * 4) =
            *(const ck_f32x4*)(stage + shift + at * 4);
    }
  };
  copy(It::R, It::R + It::ROW, 0);
  if (MODE != CK_GLA) copy(It::U, It::U + It::ROW, SU - It::U);
  copy(It::M, It::TOTAL, SO);
}

PS_DEV bool ck_finite(ck_f32x4 a) {
  // the sum of the magnitudes is a number below infinity only if all are
  return fabsf(a[0]) + fabsf(a[1]) + fabsf(a[2]) + fabsf(a[3]) < INFINITY;
}

// acc + (16 x 16 matrix) x term by term, x in the accumulators' layout, `frag`
// the matrix in fragment order. The matrix's zeros above its diagonal are left
// out: an entry of x that is no finite number would turn them into NaN and
// reach earlier tokens. tmp: 256 floats of this wave's.
PS_DEV ck_f32x4 ck_square_terms(const float* frag, ck_f32x4 x, ck_f32x4 acc,
                                int lane, float* tmp) {
  const int g = lane >> 4, n = lane & 15;
#pragma unroll
  for (int i = 0; i < 4; ++i) tmp[(4 * g + i) * 16 + n] = x[i];
  __builtin_amdgcn_wave_barrier();
#pragma unroll 1
  for (int s = 0; s < 16; ++s) {
    const float xs = tmp[s * 16 + n];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = frag[((s >> 2) * 16 + 4 * g + i) * 4 + (s & 3)];
      if (a != 0.f) acc[i] += a * xs;
    }
  }
  __builtin_amdgcn_wave_barrier();
  return acc;
}

// The same for one product's tokens 4 k + i (k: lane group): f the matrix's
// entries as that product takes them, x the lane's value, sums in its order.
PS_DEV ck_f32x4 ck_token_terms(float f, float x, ck_f32x4 acc, int lane,
                               float* tmp) {
  const int g = lane >> 4, n = lane & 15;
  tmp[lane] = f;
  tmp[64 + lane] = x;
  __builtin_amdgcn_wave_barrier();
#pragma unroll 1
  for (int k = 0; k < 4; ++k) {
    const float xs = tmp[64 + k * 16 + n];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = tmp[k * 16 + 4 * g + i];
      if (a != 0.f) acc[i] = fmaf(a, xs, acc[i]);
    }
  }
  __builtin_amdgcn_wave_barrier();
  return acc;
}

// Row tiles of 16 that a wave has: one up to 64 rows. us, one / two: general
// delta, 8 heads of 64 x 64, 8000 rows in 2 prompts 296 / 386, 32 heads, 5000 in
// 4 252 / 290, of 32 x 32 201 / 235; of 96 x 96 452 / 414, of 128 x 128 581 / 462
// (twice the waves for as many instructions beside the products).
static constexpr int ck_row_tiles(int dp) { return dp <= 64 ? 1 : 2; }

// Waves that a SIMD has registers for: three, since many short segments are
// more workgroups than two a SIMD hold; two where three would spill more than
// one register (fp32 rows of 128, either delta: 78 and 25). us, two / three:
// general delta, 32 fp32 heads of 96 x 96, 1200 rows in 40 prompts 161 / 139,
// 3000 in 40 307 / 285, 4000 in 8 330 / 327.
static constexpr int ck_sweep_waves(int mode, int dp, bool wide) {
  return !wide || dp <= 96 || mode == CK_GLA ? 3 : 2;
}

// Walks the chunks of one (segment, head) for 16 columns of its state: a wave
// per 32 rows of it (16 of up to 64), two to four waves. raw [T, H * DV]: S^T r
// before the read-out's norm.
//
// The chain from one chunk to the next is what bounds this kernel: a prompt
// has a few hundred chunks, and heads x DV / 16 workgroups are one or two a
// CU, so that a SIMD issues for one or two waves and every instruction counts.
// Rows are split over the waves: no two of them read the same operands, which
// come from memory straight into registers about a chunk and a half ahead, and
// only the waves' shares of Z and O pass through LDS. There are two sets of
// both, so a chunk has one barrier: a set is written again behind the barrier
// of the next chunk, which no wave reaches before it has read it. O's shares
// are added one chunk later, behind that chunk's barrier. Products with the
// 16 x 16 matrices are shared out by tokens, one of each group of four a wave.
// Loads of values and stores of rows go through buffers that end with the
// segment: no branches in a chunk, and what lies outside reads as zero.
// Measured (general delta, 128 x 128, one prompt of 336 chunks): 2.13 us a
// chunk with operands through LDS and 32 columns a workgroup, 1.05 now, of
// which the products take 0.5; 8 heads, 8000 rows in 2 prompts 698 -> 410 us, 32
// heads 935 -> 723.
// Workgroups of one head are H apart, so that they share an XCD's L2 where
// that is a multiple of 8.
//
// PART 1 and 2 (gla, whose state only decays between writes): a segment's
// chunks in `parts` runs that are walked at once. The first launch walks all
// runs but the last from an empty state and leaves what each adds to the state
// and its decays' product in `part` ([S_, H, parts] records of D x DV and DP;
// the last run's record takes the state before the segment). The second starts
// each run from what the runs before it leave and writes the outputs.
template <typename T, int MODE, int DP, int PART>
__global__ __launch_bounds__(DP * 4 / ck_row_tiles(DP),
                             ck_sweep_waves(MODE, DP, sizeof(T) == 4))
    void ck_sweep_kernel(
    float* __restrict__ raw, const float* __restrict__ items, int cap,
    const T* __restrict__ v, int ldv, float* __restrict__ state,
    const int* __restrict__ seq_rows, int S_, int H, int D, int DV, int base,
    float* __restrict__ part, int parts) {
  typedef CkItem<MODE, DP> It;
  constexpr int RT = ck_row_tiles(DP);   // row tiles of a wave
  constexpr int NW = DP / 16 / RT;       // waves
  constexpr int NQ = (4 + NW - 1) / NW;  // tokens of four a wave takes
  // three waves have two tokens' matrix entries each, and three a SIMD would
  // spill with the written rows on their own and the last chunk's shares early.
  // Added behind the removed ones (general delta, widths 65 to 96): the state is
  // 6.9e-8 from 64-bit results, its rows 1.81e-7
  constexpr bool LEAN = NW == 3;
  constexpr int SET = NW * 64;         // shares of one chunk, float4
  __shared__ ck_f32x4 zx[2 * SET], ox[2 * SET];
  __shared__ float tmps[NW * 128];

  const int ncb = (DV + 15) / 16;
  const int run = PART ? blockIdx.x / (S_ * H) / ncb : 0;
  const int rest = blockIdx.x - run * S_ * H * ncb;
  const int hd = rest % H, cb = rest / H % ncb;
  const CkSeg at = ck_by_length(seq_rows, S_, rest / (H * ncb));
  if (at.seg < 0) return;
  // the same in all lanes, which is not seen through the cases of ck_by_length: in
  // scalar registers for the loads' addresses (channel delta, 32 fp32 heads, 6007
  // rows in 3 prompts beside 37 tokens 610 -> 585 us). The three-term walk has none
  // left for them and keeps them as they are (32 heads of 96 x 40, 2000 rows in 20
  // prompts 49 us, 53 so)
  const int sh = __builtin_amdgcn_readfirstlane(at.seg) * H + hd;
  int t0 = __builtin_amdgcn_readfirstlane(at.t0);
  int n = __builtin_amdgcn_readfirstlane(at.n);
  const int p0 = __builtin_amdgcn_readfirstlane(at.p0);
  const int slot = __builtin_amdgcn_readfirstlane(at.slot);
  const int all = ck_count(n);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int first = at.first - base;  // its first chunk of this pass
  int c0 = max(0, -first);
  int count =
      __builtin_amdgcn_readfirstlane(min(all, cap - first) - c0);
  if (count <= 0) return;
  first += c0;
  const bool old = p0 != 0 || c0 != 0;  // there is a state to start from
  bool last = true;  // this run ends the segment's chunks of the pass
  if constexpr (PART != 0) {
    const int per = (count + parts - 1) / parts;
    last = (run + 1) * per >= count;
    // a first run is always there; the others may be empty
    if (run * per >= count) return;
    first += run * per;
    c0 += run * per;
    count = min(per, count - run * per);
  }
  // the rows from the first chunk on
  t0 = __builtin_amdgcn_readfirstlane(t0 + 16 * c0);
  n = __builtin_amdgcn_readfirstlane(n - 16 * c0);

  const int g = lane >> 4, m16 = lane & 15;
  const int j = cb * 16 + m16;  // this lane's column
  const bool col = j < DV;
  // row i of row tile t of the state
  auto row = [&](int t, int i) {
    return 16 * (RT * wave + t) + 4 * g + i;
  };
  float* Sg = state + ((size_t)slot * H + hd) * (size_t)D * DV;
  ck_f32x4 S[RT];
  const size_t rec = (size_t)D * DV + DP;  // of one run
  float* pt = PART ? part + (size_t)sh * parts * rec : nullptr;
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = row(t, i);
      const bool in = col && d < D;
      const size_t at = (size_t)d * DV + j;
      float x = 0.f;
      if (PART != 2 && in && old) x = Sg[at];
      if constexpr (PART == 1) {
        if (run == 0 && in) pt[(parts - 1) * rec + at] = x;
        x = 0.f;
      }
      if constexpr (PART == 2) {
        if (in) x = pt[(parts - 1) * rec + at];
      }
      S[t][i] = x;
    }
  if constexpr (PART == 2) {
#pragma unroll 2
    for (int q = 0; q < run; ++q)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = row(t, i);
          const float add =
              col && d < D ? pt[q * rec + (size_t)d * DV + j] : 0.f;
          S[t][i] = S[t][i] * pt[q * rec + (size_t)D * DV + d] + add;
        }
  }
  // product of the decays over the run, this wave's rows
  ck_f32x4 decay[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) decay[t] = {1.f, 1.f, 1.f, 1.f};

  // Operands through buffers, too: a uniform base, a uniform offset and a
  // 32-bit one per lane, so that a load is one instruction. `next` is the chunk
  // to fetch (the last one again behind it).
  const char* next = (const char*)(items + ((size_t)first * H + hd) * It::TOTAL);
  const size_t step = (size_t)H * It::TOTAL * sizeof(float);
  unsigned at_row[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
    at_row[t] = ck_row_slot(RT * wave + t, g, m16) * 16;
  const unsigned at_col = ck_col_slot(RT * wave, g, m16) * 16;
  const unsigned at_gam = (16 * RT * wave + 4 * g) * 4;
  const unsigned at_sq = (lane * 4 + wave) * 4;
  auto operands = [&] {
    return __builtin_amdgcn_make_buffer_rsrc((void*)next, 0, It::TOTAL * 4,
                                             0x00020000);
  };
  auto load4 = [&](__amdgpu_buffer_rsrc_t r, unsigned at, int op) {
    return __builtin_bit_cast(
        ck_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, op * 4, 0));
  };
  auto load1 = [&](__amdgpu_buffer_rsrc_t r, unsigned at, int op) {
    return __uint_as_float(
        __builtin_amdgcn_raw_buffer_load_b32(r, at, op * 4, 0));
  };
  // columns past the last one: beyond any buffer
  const unsigned off = 0x80000000u;
  unsigned at_v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    at_v[i] = col ? ((4 * g + i) * (unsigned)ldv + j) * sizeof(T) : off;
  const unsigned rs = H * DV;
  const unsigned at_out = col ? (g * rs + j) * 4 : off;
  const T* vseg = v + (size_t)t0 * ldv + hd * DV;
  float* oseg = raw + (size_t)t0 * rs + hd * DV;
  // chunk c's rows (and more, up to the segment's end) of `p`, rows of `ld`
  // elements of `e` bytes
  auto rows_from = [&](const void* p, int c, unsigned ld, unsigned e) {
    const unsigned more = min(n - 16 * c - 1, 16);
    return __builtin_amdgcn_make_buffer_rsrc(
        (char*)p + (size_t)c * (16u * e) * ld, 0, (more * ld + DV) * e,
        0x00020000);
  };

  // operands of a chunk: what meets the state before it, and what is written
  struct Reads {
    ck_f32x4 r[RT], u[RT];
    float cx[NQ], mx[NQ];  // this wave's tokens of the matrices on V
    T v[4];                // as loaded: a conversion here would wait for them
    float flag;
  };
  struct Writes {
    ck_f32x4 k[RT], b[RT], gam[RT];
    float zx[NQ];  // this wave's tokens of the matrix on Z (Y)
  };
  constexpr int LASTSQ = MODE == CK_GD ? It::MB : It::M;
  auto fetch_reads = [&](int c, Reads& x) {
    const auto p = operands();
    if constexpr (MODE != CK_GLA) {
#pragma unroll
      for (int t = 0; t < RT; ++t) x.u[t] = load4(p, at_row[t], It::U);
    }
    if constexpr (PART != 1) {
#pragma unroll
      for (int t = 0; t < RT; ++t) x.r[t] = load4(p, at_row[t], It::R);
      x.flag = ((const float*)next)[It::FLAG];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int at = wave + q * NW < 4 ? q * NW * 4 : 0;
      if constexpr (MODE != CK_GLA) x.cx[q] = load1(p, at_sq + at, It::C);
      if constexpr (MODE != CK_CD && PART != 1)
        x.mx[q] = load1(p, at_sq + at, It::M);
    }
    const auto vr = rows_from(vseg, min(c, count - 1), ldv, sizeof(T));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (sizeof(T) == 2)
        x.v[i].x = __builtin_amdgcn_raw_buffer_load_b16(vr, at_v[i], 0, 0);
      else
        x.v[i] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(vr, at_v[i], 0, 0));
    }
  };
  auto fetch_writes = [&](int c, Writes& x) {
    const auto p = operands();
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      x.gam[t] = load4(p, at_gam, It::GAM + t * 16);
      x.k[t] = load4(p, at_col, It::K + t * 256);
      if constexpr (MODE == CK_GD) x.b[t] = load4(p, at_col, It::B + t * 256);
    }
    if constexpr (MODE != CK_GLA) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        x.zx[q] = load1(p, at_sq + (wave + q * NW < 4 ? q * NW * 4 : 0),
                        LASTSQ);
    }
    if (c + 1 < count) next += step;
  };

  // the waves' shares of chunk c's rows: every wave takes groups of four,
  // reads them early and adds them later
  struct Shares {
    float o[NQ][NW];
  };
  auto shares_of = [&](int c, Shares& x) {
    const ck_f32x4* from = ox + (c & 1) * SET;
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int w = 0; w < NW; ++w)
        x.o[q][w] = ((const float*)(from + w * 64 +
                                    min(wave + q * NW, 3) * 16 + m16))[g];
  };
  auto emit = [&](int c, const Shares& x) {
    const auto out = rows_from(oseg, max(c, 0), rs, 4);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int tg = wave + q * NW;
      float o = x.o[q][0];
#pragma unroll
      for (int w = 1; w < NW; ++w) o += x.o[q][w];
      __builtin_amdgcn_raw_buffer_store_b32(
          __float_as_uint(o), out,
          (c < 0 || tg > 3 ? off : at_out) + 16 * tg * rs, 0, 0);
    }
  };

  const ck_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // Chunk c from `rd` and `wr`; those of chunk c + 2 take their places as
  // soon as they are used.
  auto walk = [&](int c, Reads& rd, Writes& wr) {
    // what comes of the state, and what of the chunk's own rows: apart, and
    // the written rows (L) too, so that the larger sums are added last (the
    // state's error against 64 bits is 5.6e-8 so, 7.7e-8 with K V on the state
    // before B Z)
    ck_f32x4 V, Z[2] = {zero, zero}, O[2] = {zero, zero}, L[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) L[t] = zero;
#pragma unroll
    for (int i = 0; i < 4; ++i) V[i] = MxElem<T>::ld(&rd.v[i]);
    // the same in every wave: all have all of V
    const bool fin =
        PART == 1 || __all(rd.flag == 0.f && ck_finite(V));
    // this wave's token of each group of four
    auto pick = [&](const ck_f32x4& x, int q) {
      const int i = wave + q * NW;
      float y = i == 1 ? x[1] : x[0];
      y = i == 2 ? x[2] : y;
      return i == 3 ? x[3] : y;
    };
    // a product with a 16 x 16 matrix; where a number is not finite its terms
    // come from `terms` below instead
    const unsigned mask = __builtin_amdgcn_readfirstlane(fin ? ~0u : 0u);
    auto on_tokens = [&](const float (&f)[NQ], const ck_f32x4& x,
                         ck_f32x4& acc) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        // three waves: the fourth token is the first wave's; no branch
        const unsigned mq = 4 % NW == 0 || wave + q * NW < 4 ? mask : 0;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(
            __uint_as_float(__float_as_uint(f[q]) & mq),
            __uint_as_float(__float_as_uint(pick(x, q)) & mq), acc, 0, 0, 0);
      }
    };
    // The same term by term, zeros above the diagonal left out: beside a value
    // that is no finite number they would reach earlier tokens. No loads here:
    // where ways meet, waits are for the latest load of either.
    auto terms = [&](const float (&f)[NQ], const ck_f32x4& x, ck_f32x4& acc) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if (4 % NW == 0 || wave + q * NW < 4)
          acc = ck_token_terms(f[q], pick(x, q), acc, lane,
                               tmps + wave * 128);
    };
    if (!fin) {
      if constexpr (MODE != CK_GLA) terms(rd.cx, V, Z[1]);
      if constexpr (MODE != CK_CD && PART != 1) terms(rd.mx, V, O[1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MODE != CK_GLA) {
      on_tokens(rd.cx, V, Z[1]);
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          // channel: Y = C V - U S
          Z[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              MODE == CK_CD ? -rd.u[t][i] : rd.u[t][i], S[t][i], Z[0], 0, 0,
              0);
    }
    if constexpr (PART != 1) {
      if constexpr (MODE != CK_CD) on_tokens(rd.mx, V, O[1]);
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          O[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(rd.r[t][i], S[t][i],
                                                      O[0], 0, 0, 0);
    }
    ck_f32x4* zs = zx + (c & 1) * SET;
    if constexpr (MODE != CK_GLA && NW > 1) zs[wave * 64 + lane] = Z[0] + Z[1];
    fetch_reads(c + 2, rd);
#pragma unroll
    for (int u = 0; u < 18; ++u) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x004, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // a load
    }
    if constexpr (PART != 1) __syncthreads();
    ck_f32x4 zr[NW];
    Shares so;
    if constexpr (MODE != CK_GLA && NW > 1) {
#pragma unroll
      for (int w = 0; w < NW; ++w) zr[w] = zs[w * 64 + lane];
    }
    if constexpr (PART != 1 && !LEAN) shares_of(c - 1, so);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      S[t] *= wr.gam[t];
      if constexpr (PART == 1) decay[t] *= wr.gam[t];
    }
    auto written = [&](ck_f32x4(&acc)[RT]) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr.k[t][i], V[i],
                                                        acc[t], 0, 0, 0);
    };
    if constexpr (MODE == CK_GD && !LEAN) written(L);
    ck_f32x4 Y = V;
    if constexpr (MODE != CK_GLA) {
      Y = NW > 1 ? zr[0] : Z[0] + Z[1];
      // in one order, so that every wave has the same sum
#pragma unroll
      for (int w = 1; w < NW; ++w) Y += zr[w];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < RT; ++t)
        S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
            MODE == CK_GD ? wr.b[t][i] : wr.k[t][i], Y[i], S[t], 0, 0, 0);
    if constexpr (MODE == CK_GD && !LEAN) {
#pragma unroll
      for (int t = 0; t < RT; ++t) S[t] += L[t];
    }
    if constexpr (MODE == CK_GD && LEAN) written(S);
    if constexpr (MODE != CK_GLA) {
      on_tokens(wr.zx, Y, O[1]);
      __builtin_amdgcn_sched_barrier(0);
      if (!fin) terms(wr.zx, Y, O[1]);
    }
    fetch_writes(c + 2, wr);
    if constexpr (PART != 1) {
      if constexpr (LEAN) shares_of(c - 1, so);
      emit(c - 1, so);
      ox[(c & 1) * SET + wave * 64 + lane] = O[0] + O[1];
    }
  };

  Reads ra, rb;
  Writes wa, wb;
  fetch_reads(0, ra);
  __builtin_amdgcn_sched_barrier(0);  // landing in this order, as below
  fetch_writes(0, wa);
  __builtin_amdgcn_sched_barrier(0);
  fetch_reads(1, rb);
  __builtin_amdgcn_sched_barrier(0);
  fetch_writes(1, wb);
  __builtin_amdgcn_sched_barrier(0);
  // one way out: where ways meet, waits are for the latest load of either
  int c = 0;
#pragma unroll 1
  for (; c + 1 < count; c += 2) {
    walk(c, ra, wa);
    walk(c + 1, rb, wb);
  }
  if (c < count) walk(c, ra, wa);
  if constexpr (PART != 1) {
    __syncthreads();
    Shares so;
    shares_of(count - 1, so);
    emit(count - 1, so);
  }
  float* Se = Sg;
  if constexpr (PART == 1) {
    Se = pt + run * rec;
    if (cb == 0 && m16 == 0) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          Se[(size_t)D * DV + row(t, i)] = decay[t][i];
    }
  }
  if (col && (PART != 2 || last)) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (row(t, i) < D) Se[(size_t)row(t, i) * DV + j] = S[t][i];
  }
}

// ---------------------------------------------------------------------------
// one decay per head and token
// ---------------------------------------------------------------------------
template <int DP>
struct CkGroup {  // per chunk and group: fragments of Q and K
  static constexpr int R = 0;
  static constexpr int K = 16 * DP;
  static constexpr int TOTAL = 32 * DP;
};
// Floats of a head in a row of the matrix LSTM's outputs before their read-out: its
// columns, n.q behind them, up to a border of 16 bytes.
__host__ __device__ constexpr int ck_pitch(int DV) { return (DV + 4) & ~3; }

struct CkHead {  // per chunk and head
  static constexpr int M = 0;     // 16 x 16 on V, fragment order
  static constexpr int DR = 256;  // [16] decay from the chunk's start
  static constexpr int DK = 272;  // [16] write scale and decay to its end
  static constexpr int GAM = 288; // decay over the chunk
  static constexpr int TOTAL = 292;
};

// Gates of the matrix LSTM: i = cap(wr + p0), f = logsigmoid(cap(dec + p1)),
// m' = max(f + m, i); ga / gw / ge [T, H] = exp(f + m - m'), exp(i - m'),
// exp(-m'). The running maximum over 64 tokens is a scan over a wave's lanes of the
// maps m -> max(m + A, B). A workgroup per (segment, head), whose waves scan 64
// tokens each at a time; the maps of whole waves go through LDS, where every wave
// follows m through those before it, so that it is what one wave after another would
// find. A turn takes 0.8 us whatever its waves (one wave a segment: 16 heads, 4950 rows
// in 2 prompts 44 us, 9 with 16).
template <typename T>
__global__ __launch_bounds__(1024) void ck_gates_kernel(
    float* __restrict__ ga, float* __restrict__ gw, float* __restrict__ ge,
    const T* __restrict__ wr, int ldwr, const T* __restrict__ dec, int lddec,
    const float* __restrict__ p0, const float* __restrict__ p1,
    float* __restrict__ aux, const int* __restrict__ seq_rows, int H, int D,
    float cap) {
  __shared__ float2 s_map[2][16];
  const int seg = blockIdx.x / H, hd = blockIdx.x % H;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int t0 = seq_rows[4 * seg], n = seq_rows[4 * seg + 1];
  const int pos0 = seq_rows[4 * seg + 2], slot = seq_rows[4 * seg + 3];
  if (n < 16) return;
  float* mp = aux + ((size_t)slot * H + hd) * (D + 1) + D;
  float m = pos0 != 0 ? *mp : 0.f;  // before the turn's first token
  const float bi = p0[hd], bf = p1[hd];
  // the next turn's inputs are asked for before these are used: few waves have
  // nothing else to wait beside
  auto fetch = [&](int t, float* zi, float* zf) {
    const size_t row = (size_t)(t0 + min(t, n - 1));
    *zi = MxElem<T>::ld(wr + row * ldwr + hd);
    *zf = MxElem<T>::ld(dec + row * lddec + hd);
  };
  float zi, zf, ni, nf;
  fetch(wave * 64 + lane, &ni, &nf);
  int turn = 0;
  for (int tb = 0; tb < n; tb += 64 * waves) {
    const int t = tb + wave * 64 + lane;
    const size_t row = (size_t)(t0 + min(t, n - 1));
    zi = ni + bi;
    zf = nf + bf;
    fetch(t + 64 * waves, &ni, &nf);
    const float ig = cap * tanhf(zi / cap);
    const float fg = ck_log_sigmoid(cap * tanhf(zf / cap));
    float A = fg, B = ig;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float a1 = __shfl_up(A, off, 64), b1 = __shfl_up(B, off, 64);
      if (lane >= off) {
        B = fmaxf(b1 + A, B);
        A += a1;
      }
    }
    if (lane == 63) s_map[turn][wave] = make_float2(A, B);
    __syncthreads();
    float mw = m;  // before this wave's first token
    for (int w = 0; w < waves; ++w) {
      const float2 ab = s_map[turn][w];
      if (w == wave) mw = m;
      m = fmaxf(m + ab.x, ab.y);
    }
    turn ^= 1;
    const float mn = fmaxf(mw + A, B);
    float mo = __shfl_up(mn, 1, 64);
    if (lane == 0) mo = mw;
    if (t < n) {
      ga[row * H + hd] = expf(fg + mo - mn);
      gw[row * H + hd] = expf(ig - mn);
      ge[row * H + hd] = expf(-mn);
    }
    if (t == n - 1) *mp = mn;
  }
}

// Waves of a workgroup of the gates: as many as a segment of all rows has 64s of,
// fewer where the segments' heads are many (a workgroup of a segment of a few rows has
// nothing to do, whatever its size).
static int ck_gate_waves(int T_, int S_, int H) {
  const long most = 8192l / ((long)S_ * H);
  const int want = (T_ + 63) / 64 < 16 ? (T_ + 63) / 64 : 16;
  return most < 1 ? 1 : most < want ? (int)most : want;
}

template <typename T, int MODE, int DP>
__global__ __launch_bounds__(256) void ck_prep_scalar_kernel(
    float* __restrict__ gitems, float* __restrict__ hitems, CkIn in,
    const float* __restrict__ ga, const float* __restrict__ gw,
    const int* __restrict__ seq_rows, int S_, int H, int G, int D,
    float qscale, int base) {
  typedef CkGroup<DP> Gi;
  constexpr int LD = DP + 4;
  __shared__ __align__(16) float Q[16 * LD];
  __shared__ __align__(16) float K[16 * LD];
  __shared__ __align__(16) float qk[256];
  __shared__ __align__(16) float sa[16][16];
  __shared__ float sw[16][16];

  const int item = blockIdx.x, grp = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int seg, chunk;
  if (!ck_find(seq_rows, S_, base + item, lane, &seg, &chunk)) return;
  const int n = seq_rows[4 * seg + 1];
  const int row0 = seq_rows[4 * seg] + 16 * chunk;
  const int nv = min(16, n - 16 * chunk);
  const T* qp = (const T*)in.q + grp * D;
  const T* kp = (const T*)in.k + grp * D;
  for (int i = threadIdx.x; i < 16 * DP; i += 256) {
    const int t = i / DP, d = i % DP;
    const size_t row = (size_t)(row0 + min(t, nv - 1));
    const int dc = min(d, D - 1);
    const float q = MxElem<T>::ld(qp + row * in.ldq + dc);
    const float k = MxElem<T>::ld(kp + row * in.ldk + dc);
    const bool live = t < nv && d < D;
    Q[t * LD + d] = live ? q * qscale : 0.f;
    K[t * LD + d] = live ? k : 0.f;
  }
  __syncthreads();
  const int g = lane >> 4, m16 = lane & 15;
  if (wave == 0) {
    ck_f32x4 c = {0.f, 0.f, 0.f, 0.f}, c2 = c;
#pragma unroll
    for (int t = 0; t < DP / 16; ++t) {
      const ck_f32x4 x = *(const ck_f32x4*)(Q + m16 * LD + t * 16 + g * 4);
      const ck_f32x4 y = *(const ck_f32x4*)(K + m16 * LD + t * 16 + g * 4);
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[0], y[0], c, 0, 0, 0);
      c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[1], y[1], c2, 0, 0, 0);
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[2], y[2], c, 0, 0, 0);
      c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[3], y[3], c2, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      qk[((m16 >> 2) * 16 + 4 * g + i) * 4 + (m16 & 3)] = c[i] + c2[i];
  }
  if (blockIdx.z == 0) {
    float* dst = gitems + ((size_t)item * G + grp) * Gi::TOTAL;
    for (int f = threadIdx.x; f < DP * 4; f += 256) {  // float4 slots
      const int t = f >> 6, fg = (f >> 4) & 3, fm = f & 15;
      *(ck_f32x4*)(dst + Gi::R + ck_row_slot(t, fg, fm) * 4) =
          *(const ck_f32x4*)(Q + fm * LD + t * 16 + fg * 4);
      ck_f32x4 kk;
#pragma unroll
      for (int i = 0; i < 4; ++i) kk[i] = K[(4 * fg + i) * LD + t * 16 + fm];
      *(ck_f32x4*)(dst + Gi::K + f * 4) = kk;
    }
  }
  // this slice's heads, 16 at a time: their scalars, then the matrices
  const int per = H / G;
  const int slice = (per + gridDim.z - 1) / gridDim.z;
  const int h1 = min(per, (int)(blockIdx.z + 1) * slice);
  for (int hb = blockIdx.z * slice; hb < h1; hb += 16) {
    __syncthreads();
    {
      const int hl = threadIdx.x & 15, t = threadIdx.x >> 4;
      const int hd = grp * per + min(hb + hl, h1 - 1);
      const size_t row = (size_t)(row0 + min(t, nv - 1));
      float a, w;
      if (MODE == CK_SSD) {
        w = ck_softplus(
            MxElem<T>::ld((const T*)in.dec + row * in.lddec + hd) +
            in.p0[hd]);
        a = expf(-expf(in.p1[hd]) * w);
      } else {
        a = ga[row * H + hd];
        w = gw[row * H + hd];
      }
      sa[hl][t] = t < nv ? a : 1.f;
      sw[hl][t] = t < nv ? w : 0.f;
    }
    __syncthreads();
    // thread = entry of the matrix in fragment order
    const int s = wave * 4 + (threadIdx.x & 3), t = (threadIdx.x >> 2) & 15;
    const float dot = qk[threadIdx.x];
    for (int hl = 0; hl < 16 && hb + hl < h1; ++hl) {
      float e = 1.f;
#pragma unroll
      for (int j4 = 0; j4 < 4; ++j4) {
        const ck_f32x4 a4 = *(const ck_f32x4*)(&sa[hl][j4 * 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = j4 * 4 + i;
          e *= (j > s && j <= t) ? a4[i] : 1.f;
        }
      }
      float* dst = hitems +
                   ((size_t)item * H + grp * per + hb + hl) * CkHead::TOTAL;
      dst[CkHead::M + threadIdx.x] = t >= s ? dot * e * sw[hl][s] : 0.f;
      if (s == 0) dst[CkHead::DR + t] = e * sa[hl][0];
      if (t == 15) dst[CkHead::DK + s] = e * sw[hl][s];
      if (s == 0 && t == 15) dst[CkHead::GAM] = e * sa[hl][0];
    }
  }
}

// The walk of ck_sweep_kernel for one decay per head and token. out: the
// finished fp32 rows of ssd, (o + skip v) silu(gate), or the raw read-outs
// [T, H * ck_pitch(DV)] of mlstm, whose column DV is the normaliser's (its values
// are 1, its state lies in aux). PART, part and parts as there; a record is the
// D x (DV, with the normaliser DV + 1) state and one decay.
template <typename T, int MODE, int DP, int PART>
__global__ __launch_bounds__(256, 2) void ck_sweep_scalar_kernel(
    float* __restrict__ out, int ldo, const float* __restrict__ gitems,
    const float* __restrict__ hitems, int cap, CkIn in,
    const float* __restrict__ p2, float* __restrict__ state,
    float* __restrict__ aux, const int* __restrict__ seq_rows, int S_, int H,
    int G, int D, int DV, int base, float* __restrict__ part,
    int parts) {
  typedef CkGroup<DP> Gi;
  constexpr int NT = DP / 32;
  constexpr int PG = Gi::TOTAL / 1024;  // DP is a multiple of 32
  constexpr int BUF = Gi::TOTAL + 512;  // fragments, then the head's
  __shared__ __align__(16) float lds[2 * BUF];
  __shared__ __align__(16) float xch[4 * 256];
  __shared__ __align__(16) float tmps[4 * 256];
  float* tmp = tmps + (threadIdx.x >> 6) * 256;

  const int cols = DV + (MODE == CK_MLSTM ? 1 : 0), ncb = (cols + 31) / 32;
  const int sh = blockIdx.x % (S_ * H), cb = blockIdx.x / (S_ * H) % ncb;
  const int run = PART ? blockIdx.x / (S_ * H) / ncb : 0;
  const int seg = sh / H, hd = sh % H, grp = hd / (H / G);
  int t0 = seq_rows[4 * seg], n = seq_rows[4 * seg + 1];
  const int p0 = seq_rows[4 * seg + 2], slot = seq_rows[4 * seg + 3];
  const int all = ck_count(n);
  if (all == 0) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int first = 0;
  for (int s = lane; s < seg; s += 64)
    first += ck_count(seq_rows[4 * s + 1]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off, 64);
  first = __builtin_amdgcn_readfirstlane(first) - base;  // of this pass
  int c0 = max(0, -first);
  int count =
      __builtin_amdgcn_readfirstlane(min(all, cap - first) - c0);
  if (count <= 0) return;
  first += c0;
  const bool old = p0 != 0 || c0 != 0;  // there is a state to start from
  bool last = true;  // this run ends the segment's chunks of the pass
  if constexpr (PART != 0) {
    const int per = (count + parts - 1) / parts;
    last = (run + 1) * per >= count;
    if (run * per >= count) return;
    first += run * per;
    c0 += run * per;
    count = min(per, count - run * per);
  }
  // the rows from the first chunk on
  t0 += 16 * c0;
  n -= 16 * c0;

  const int g = lane >> 4, m16 = lane & 15;
  const int ct = wave >> 1, ds = wave & 1, tb = ds * NT;
  const int j = cb * 32 + ct * 16 + m16;
  const bool col = j < DV;
  const bool ncol = MODE == CK_MLSTM && j == DV;
  const int hv = hd * DV + (col ? j : 0);
  float* Sg = state + ((size_t)slot * H + hd) * (size_t)D * DV + j;
  float* Ng = MODE == CK_MLSTM ? aux + ((size_t)slot * H + hd) * (D + 1)
                               : nullptr;
  const size_t rec = (size_t)D * cols + 4;  // of one run
  float* pt = PART ? part + (size_t)sh * parts * rec : nullptr;
  ck_f32x4 S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * (tb + t) + 4 * g + i;
      float x = 0.f;
      if (PART != 2 && d < D && old) {
        if (col) x = Sg[(size_t)d * DV];
        if (ncol) x = Ng[d];
      }
      if constexpr (PART == 1) {
        if (run == 0 && d < D && (col || ncol))
          pt[(parts - 1) * rec + (size_t)d * cols + j] = x;
        x = 0.f;
      }
      if constexpr (PART == 2) {
        if (d < D && (col || ncol))
          x = pt[(parts - 1) * rec + (size_t)d * cols + j];
      }
      S[t][i] = x;
    }
  if constexpr (PART == 2) {
#pragma unroll 2
    for (int q = 0; q < run; ++q) {
      const float a = pt[q * rec + (size_t)D * cols];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = 16 * (tb + t) + 4 * g + i;
          const float add = d < D && (col || ncol)
                                ? pt[q * rec + (size_t)d * cols + j]
                                : 0.f;
          S[t][i] = S[t][i] * a + add;
        }
    }
  }
  float decay = 1.f;  // over the run

  const char* gsrc =
      (const char*)(gitems + ((size_t)first * G + grp) * Gi::TOTAL);
  const char* hsrc =
      (const char*)(hitems + ((size_t)first * H + hd) * CkHead::TOTAL);
  const size_t gstep = (size_t)G * Gi::TOTAL * sizeof(float);
  const size_t hstep = (size_t)H * CkHead::TOTAL * sizeof(float);
  const unsigned at16 = threadIdx.x * 16;
  const unsigned ath = min((int)threadIdx.x, CkHead::TOTAL / 4 - 1) * 16;
  const T* vcol = (const T*)in.v + (size_t)t0 * in.ldv + hv;
  const T* gcol = (const T*)in.gate + (size_t)t0 * in.ldg + hv;
  const float skip = MODE == CK_SSD ? p2[hd] : 0.f;
  struct Next {
    ck_f32x4 f[PG], h;
    T v[4], gt[4];
  };
  auto fetch = [&](int c, Next& x) {
    c = min(c, count - 1);
#pragma unroll
    for (int u = 0; u < PG; ++u)
      x.f[u] = *(const ck_f32x4*)(gsrc + c * gstep + u * 4096 + at16);
    x.h = *(const ck_f32x4*)(hsrc + c * hstep + ath);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tt = min(16 * c + 4 * g + i, n - 1);
      x.v[i] = vcol[(size_t)tt * in.ldv];
      if (MODE == CK_SSD) x.gt[i] = gcol[(size_t)tt * in.ldg];
    }
  };
  auto put = [&](float* dst, const Next& x) {
#pragma unroll
    for (int u = 0; u < PG; ++u)
      *(ck_f32x4*)(dst + u * 1024 + threadIdx.x * 4) = x.f[u];
    if (threadIdx.x < 128)
      *(ck_f32x4*)(dst + Gi::TOTAL + threadIdx.x * 4) = x.h;
  };
  auto walk = [&](int c, const float* buf, Next& x, float* nbuf,
                  const Next& nx) {
    const float* hb = buf + Gi::TOTAL;
    const int left = n - 16 * c - 4 * g;
    ck_f32x4 V, gt;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float y = MxElem<T>::ld(&x.v[i]);
      if (MODE == CK_MLSTM) y = col ? y : (ncol ? 1.f : 0.f);
      V[i] = i < left && (MODE == CK_MLSTM || col) ? y : 0.f;
      gt[i] = MODE == CK_SSD ? MxElem<T>::ld(&x.gt[i]) : 0.f;
    }
    ck_f32x4 r4[NT], k4[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      r4[t] = *(const ck_f32x4*)(buf + Gi::R + ck_row_slot(tb + t, g, m16) * 4);
      k4[t] = *(const ck_f32x4*)(buf + Gi::K + ck_col_slot(tb + t, g, m16) * 4);
    }
    const ck_f32x4 q4 = *(const ck_f32x4*)(hb + CkHead::M + lane * 4);
    const ck_f32x4 dr = *(const ck_f32x4*)(hb + CkHead::DR + g * 4);
    const ck_f32x4 dk = *(const ck_f32x4*)(hb + CkHead::DK + g * 4);
    const float gam = hb[CkHead::GAM];
    const bool fin = !__any(!ck_finite(V));
    fetch(c + 2, x);
    put(nbuf, nx);
    const ck_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    ck_f32x4 O = zero, Z = zero, X = zero;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        O = __builtin_amdgcn_mfma_f32_16x16x4f32(r4[t][i], S[t][i], O, 0, 0,
                                                 0);
        Z = __builtin_amdgcn_mfma_f32_16x16x4f32(r4[t][i + 1], S[t][i + 1], Z,
                                                 0, 0, 0);
      }
    if constexpr (PART == 1) decay *= gam;
    const ck_f32x4 W = V * dk;
#pragma unroll
    for (int t = 0; t < NT; ++t) S[t] *= gam;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[t][i], W[i], S[t], 0,
                                                    0, 0);
      X = __builtin_amdgcn_mfma_f32_16x16x4f32(q4[i], V[i], X, 0, 0, 0);
    }
    O += Z;
    if (ds == 1) *(ck_f32x4*)(xch + ct * 256 + lane * 4) = O;
    if (!fin) X = ck_square_terms(hb + CkHead::M, V, zero, lane, tmp);
    // also: this chunk's buffer is read, the next one's is filled
    __syncthreads();
    if (PART != 1 && ds == 0 && (col || ncol)) {
      O = (O + *(const ck_f32x4*)(xch + ct * 256 + lane * 4)) * dr + X;
      const size_t row = (size_t)(t0 + 16 * c + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < left) {
          if (MODE == CK_SSD)
            out[(row + i) * ldo + hv] =
                (O[i] + skip * V[i]) * gt[i] * ck_sigmoid(gt[i]);
          else
            out[(row + i) * ldo + hd * ck_pitch(DV) + j] = O[i];
        }
      }
    }
  };
  Next xa, xb;
  fetch(0, xa);
  fetch(1, xb);
  put(lds, xa);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int c = 0; c < count; c += 2) {
    walk(c, lds, xa, lds + BUF, xb);
    if (c + 1 >= count) break;
    // the exchange of the chunk before is read by then
    __syncthreads();
    walk(c + 1, lds + BUF, xb, lds, xa);
    if (c + 2 >= count) break;
    __syncthreads();
  }
  if (PART == 1 && cb == 0 && threadIdx.x == 0)
    pt[run * rec + (size_t)D * cols] = decay;
  if (PART == 2 && !last) return;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * (tb + t) + 4 * g + i;
      if (d < D) {
        if (PART == 1) {
          if (col || ncol) pt[run * rec + (size_t)d * cols + j] = S[t][i];
        } else {
          if (col) Sg[(size_t)d * DV] = S[t][i];
          if (ncol) Ng[d] = S[t][i];
        }
      }
    }
}

// ---------------------------------------------------------------------------
// one decay per head and token, bf16 rows: chunks of 32 on the bf16 unit
// ---------------------------------------------------------------------------
// The order of a chunk's 32 tokens in the inner index of a product: a lane
// group's eight are 4 g .. + 3 and 16 + 4 g .. + 3, which are also the rows it
// has of two accumulator tiles.
#define CK_WIDE 32

template <int DP>
struct CkWide {  // per chunk and group, bytes
  static constexpr int Q = 0;               // [2 token tiles][DP / 32][64] x 16
  static constexpr int K = 64 * DP;         // [DP / 16][64] x 16, transposed
  static constexpr int QK = 128 * DP;       // [3 blocks][64] x 16: q_t k_s, fp32
  static constexpr int TOTAL = QK + 3072;
};
struct CkWideHead {  // per chunk and head, floats
  static constexpr int A = 0;     // [32] decay of a token
  static constexpr int W = 32;    // [32] its write scale
  static constexpr int DR = 64;   // [32] decay from the start, with it, scaled
  static constexpr int DK = 96;   // [32] write scale and decay to the end
  static constexpr int P = 128;   // [32] decay from the block of four's start
  static constexpr int SUF = 160; // [16] first half: behind it to 15
  static constexpr int PRE = 176; // [16] second half: from 16, with it
  static constexpr int GAM = 192; // decay over the chunk
  static constexpr int FLAG = 193; // not 0: a q, k or write scale is no finite
                                   // number, or so large that q k w might not be
  static constexpr int TOTAL = 196;
};

template <int MODE, int DP>
__global__ __launch_bounds__(256) void ck_prep_wide_kernel(
    char* __restrict__ gitems, float* __restrict__ hitems, CkIn in,
    const float* __restrict__ ga, const float* __restrict__ gw,
    const int* __restrict__ seq_rows, int S_, int H, int G, int D,
    float qscale, int base) {
  typedef CkWide<DP> Gi;
  typedef CkWideHead Hd;
  constexpr int LD = DP + 8;
  __shared__ __align__(16) unsigned short Q[32 * LD], K[32 * LD];
  __shared__ __align__(16) float sa[8][32];
  __shared__ float sw[8][32];

  const int item = blockIdx.x, grp = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int seg, chunk;
  if (!ck_find<CK_WIDE>(seq_rows, S_, base + item, lane, &seg, &chunk)) return;
  const int n = seq_rows[4 * seg + 1];
  const int row0 = seq_rows[4 * seg] + 32 * chunk;
  const int nv = min(32, n - 32 * chunk);
  const int g = lane >> 4, m16 = lane & 15;
  const mx_bf16* qp = (const mx_bf16*)in.q + grp * D;
  const mx_bf16* kp = (const mx_bf16*)in.k + grp * D;
  bool odd = false;
  for (int i = threadIdx.x; i < 32 * DP; i += 256) {
    const int t = i / DP, d = i % DP;
    const size_t row = (size_t)(row0 + min(t, nv - 1));
    const int dc = min(d, D - 1);
    const unsigned short q = qp[row * in.ldq + dc].x;
    const unsigned short k = kp[row * in.ldk + dc].x;
    const bool live = t < nv && d < D;
    Q[t * LD + d] = live ? q : 0;
    K[t * LD + d] = live ? k : 0;
    odd |= live && max(q & 0x7fff, k & 0x7fff) >= 0x4d80;  // 2^28
  }
  odd = __syncthreads_or(odd);
  if (blockIdx.z == 0) {
    char* dst = gitems + ((size_t)item * G + grp) * Gi::TOTAL;
    auto rows8 = [&](const unsigned short* x, int tok, int ks) {
      const unsigned short* p = x + tok * LD + 32 * ks + 4 * g;
      return ck_join(*(const ck_u32x2*)p, *(const ck_u32x2*)(p + 16));
    };
    if (wave < 3) {
      // blocks (tokens t, s): (0, 0), (1, 0), (1, 1), s in rows. Sums of 32
      // channels by pairs: the rows' error against 64 bits is 9.4e-8 so, 1.01e-7
      // with one sum after the other (1.00e-7 by fp32 products)
      ck_f32x4 c[4] = {};
#pragma unroll
      for (int ks = 0; ks < DP / 32; ++ks)
        c[ks] = ck_mfma(rows8(K, (wave == 2 ? 16 : 0) + m16, ks),
                        rows8(Q, (wave == 0 ? 0 : 16) + m16, ks), c[ks]);
      *(ck_f32x4*)(dst + Gi::QK + (wave * 64 + lane) * 16) =
          ((c[0] + c[1]) + (c[2] + c[3])) * qscale;
    }
    for (int f = wave; f < DP / 16; f += 4) {
      // f: token tile and 32 channels of Q, 16 channels of K
      const int mt = f / (DP / 32), ks = f % (DP / 32);
      *(ck_u32x4*)(dst + Gi::Q + (f * 64 + lane) * 16) =
          rows8(Q, 16 * mt + m16, ks);
      unsigned short x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[j] = K[((j >> 2) * 16 + 4 * g + (j & 3)) * LD + 16 * f + m16];
      ck_u32x4 y;
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = x[2 * j] | (unsigned)x[2 * j + 1] << 16;
      *(ck_u32x4*)(dst + Gi::K + (f * 64 + lane) * 16) = y;
    }
  }
  // this slice's heads, 8 at a time: a thread per token
  const int per = H / G;
  const int slice = (per + gridDim.z - 1) / gridDim.z;
  const int h1 = min(per, (int)(blockIdx.z + 1) * slice);
  const int hl = threadIdx.x >> 5, t = threadIdx.x & 31;
  for (int hb = blockIdx.z * slice; hb < h1; hb += 8) {
    const int hd = grp * per + min(hb + hl, h1 - 1);
    const size_t row = (size_t)(row0 + min(t, nv - 1));
    float a, w;
    if (MODE == CK_SSD) {
      w = ck_softplus(
          MxElem<mx_bf16>::ld((const mx_bf16*)in.dec + row * in.lddec + hd) +
          in.p0[hd]);
      a = expf(-expf(in.p1[hd]) * w);
    } else {
      a = ga[row * H + hd];
      w = gw[row * H + hd];
    }
    a = t < nv ? a : 1.f;
    w = t < nv ? w : 0.f;
    const unsigned large = __ballot(!(w < 0x1p60f)) >> (threadIdx.x & 32);
    __syncthreads();
    sa[hl][t] = a;
    sw[hl][t] = w;
    __syncthreads();
    if (hb + hl < h1) {
      // products up to t (of all, of its half, of its four) and behind t; a
      // decay that is not in a product must not touch it: no quotients
      float dr = 1.f, pre = 1.f, p4 = 1.f, to = 1.f, suf = 1.f;
#pragma unroll
      for (int j4 = 0; j4 < 8; ++j4) {
        const ck_f32x4 a4 = *(const ck_f32x4*)(&sa[hl][j4 * 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = j4 * 4 + i;
          const float up = j <= t ? a4[i] : 1.f;
          dr *= up;
          if (j >= 16) pre *= up;
          p4 *= j >= (t & ~3) ? up : 1.f;
          const float down = j > t ? a4[i] : 1.f;
          to *= down;
          if (j < 16) suf *= down;
        }
      }
      float* dst = hitems +
                   ((size_t)item * H + grp * per + hb + hl) * Hd::TOTAL;
      dst[Hd::A + t] = a;
      dst[Hd::W + t] = w;
      dst[Hd::DR + t] = dr * qscale;
      dst[Hd::DK + t] = to * w;
      dst[Hd::P + t] = p4;
      if (t < 16)
        dst[Hd::SUF + t] = suf;
      else
        dst[Hd::PRE + t - 16] = pre;
      if (t == 31) {
        dst[Hd::GAM] = dr;
        *(unsigned*)(dst + Hd::FLAG) = large | odd;
      }
    }
  }
}

// Walks the chunks of one (segment, head): NW tiles of 16 columns of the state a
// workgroup, each in two waves that have half of its rows (one wave where DP is
// no multiple of 64). out, PART, part and parts as in ck_sweep_scalar_kernel,
// whose products these are, for bf16 q, k and v.
//
// Q, K and V go into the products as they are and the state, the weights of the
// chunk's own rows (M) and the scaled values (W) as three bf16 terms: no number
// is rounded, and the matrix unit takes 3 / 16 of the fp32 products' time. What
// bounds the walk is then the issue of instructions, above all cutting the
// state into terms (176 for a tile's rows), once a chunk, which is why a chunk
// has 32 tokens. M, the same for all columns of a head, is made by three waves
// and passes through LDS, a chunk ahead; the two waves of a tile exchange their
// shares of O there, each for the token tile that the other one writes. One
// barrier a chunk does for both.
// Measured (ssd, 128 heads of 128 x 64, 8192 rows in 2 prompts): 605 us by
// fp32 products in chunks of 16, 330 with all rows of a tile in one wave (one
// wave a SIMD: 800 instructions in 5300 cycles), 285 with two; the whole call
// 308, and 297 since infinities take a walk of their own.
// memory that no kernel under way writes: scalar loads
#define CK_CONST __attribute__((address_space(4)))
struct CkWideCall {
  float* out;
  int ldo;
  const char* gitems;
  const float* hitems;
  int cap;
  CkIn in;
  const float* p2;
  float *state, *aux;
  const int* seq_rows;
  int S_, H, G, D, DV, base;
  float* part;
  int parts;
};
template <int DP, int NW>
struct CkWideLds {
  static constexpr int WAVES = NW * (DP % 64 == 0 ? 2 : 1);
  ck_u32x4 mfrag[2][2][3][64];  // set, token tile, term
  float vtmp[WAVES][512];
  ck_f32x4 share[2][DP % 64 == 0 ? WAVES : 1][64];
};

// The walk; false where something in it came to no finite number (to all waves of
// the workgroup, or each on its own where PART is 1): then the state is not
// written. AGAIN: the walk from its start after that, with nothing ahead, for
// infinities as the fp32 products have them. In the loop itself their branches
// took 3 to 10 % of the walk.
template <int MODE, int DP, int PART, int NW, bool AGAIN>
PS_DEV bool ck_walk_wide(const CkWideCall& a, CkWideLds<DP, NW>& lds) {
  typedef CkWide<DP> Gi;
  typedef CkWideHead Hd;
  constexpr int RH = DP % 64 == 0 ? 2 : 1;   // waves that share a column tile
  constexpr int NT = DP / 16, NK = DP / 32;  // tiles of the state
  constexpr int WT = NT / RH, WK = NK / RH;  // and of a wave
  auto& mfrag = lds.mfrag;
  auto& vtmp = lds.vtmp;
  auto& share = lds.share;
  const CkIn& in = a.in;
  const int S_ = a.S_, H = a.H, G = a.G, D = a.D, DV = a.DV, ldo = a.ldo;
  const int cap = a.cap, base = a.base, parts = a.parts;
  const int* seq_rows = a.seq_rows;

  const int cols = DV + (MODE == CK_MLSTM ? 1 : 0);
  const int ncb = ((cols + 15) / 16 + NW - 1) / NW;
  const int run = PART ? blockIdx.x / (S_ * H) / ncb : 0;
  const int rest = blockIdx.x - run * S_ * H * ncb;
  const int hd = rest % H, cb = rest / H % ncb;
  const CkSeg at = ck_by_length<CK_WIDE>(seq_rows, S_, rest / (H * ncb));
  if (at.seg < 0) return true;
  const int sh = at.seg * H + hd, grp = hd / (H / G);
  int t0 = at.t0, n = at.n;
  const int p0 = at.p0, slot = at.slot;
  const int all = ck_count<CK_WIDE>(n);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int first = at.first - base;  // its first chunk of this pass
  int c0 = max(0, -first);
  int count =
      __builtin_amdgcn_readfirstlane(min(all, cap - first) - c0);
  if (count <= 0) return true;
  first += c0;
  const bool old = p0 != 0 || c0 != 0;  // there is a state to start from
  bool last = true;  // this run ends the segment's chunks of the pass
  if constexpr (PART != 0) {
    const int per = (count + parts - 1) / parts;
    last = (run + 1) * per >= count;
    if (run * per >= count) return true;
    first += run * per;
    c0 += run * per;
    count = min(per, count - run * per);
  }
  // the rows from the first chunk on
  t0 = __builtin_amdgcn_readfirstlane(t0 + 32 * c0);
  n = __builtin_amdgcn_readfirstlane(n - 32 * c0);

  const int g = lane >> 4, m16 = lane & 15;
  // which part of the rows; a wave's rows of the output are the token tile of
  // that number where two share them
  const int rh = RH == 2 ? wave & 1 : 0;
  const int j = (cb * NW + wave / RH) * 16 + m16;
  const bool col = j < DV;
  const bool ncol = MODE == CK_MLSTM && j == DV;
  float* Sg = a.state + ((size_t)slot * H + hd) * (size_t)D * DV + j;
  float* Ng = MODE == CK_MLSTM ? a.aux + ((size_t)slot * H + hd) * (D + 1)
                               : nullptr;
  const size_t rec = (size_t)D * cols + 4;  // of one run
  float* pt = PART ? a.part + (size_t)sh * parts * rec : nullptr;
  ck_f32x4 S[WT];
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * (WT * rh + t) + 4 * g + i;
      float x = 0.f;
      if (PART != 2 && d < D && old) {
        if (col) x = Sg[(size_t)d * DV];
        if (ncol) x = Ng[d];
      }
      if constexpr (PART == 1) {
        if (run == 0 && d < D && (col || ncol))
          pt[(parts - 1) * rec + (size_t)d * cols + j] = x;
        x = 0.f;
      }
      if constexpr (PART == 2) {
        if (d < D && (col || ncol))
          x = pt[(parts - 1) * rec + (size_t)d * cols + j];
      }
      S[t][i] = x;
    }
  if constexpr (PART == 2) {
#pragma unroll 2
    for (int q = 0; q < run; ++q) {
      const float a = pt[q * rec + (size_t)D * cols];
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = 16 * (WT * rh + t) + 4 * g + i;
          const float add = d < D && (col || ncol)
                                ? pt[q * rec + (size_t)d * cols + j]
                                : 0.f;
          S[t][i] = S[t][i] * a + add;
        }
    }
  }
  float decay = 1.f;  // over the run

  // Everything comes through buffers: a uniform base, a uniform offset and a
  // 32-bit one per lane; rows behind the segment read as zero and are not
  // written, nor are columns behind the last one (`off` is beyond any buffer).
  const size_t gstep = (size_t)G * Gi::TOTAL;
  const size_t hstep = (size_t)H * Hd::TOTAL * sizeof(float);
  // of the chunk ahead by one, two (the last one again behind it)
  const char* g1 = a.gitems + ((size_t)first * G + grp) * Gi::TOTAL;
  const char* g2 = g1;
  const char* h2 =
      (const char*)(a.hitems + ((size_t)first * H + hd) * Hd::TOTAL);
  const unsigned at16 = lane * 16, off = 0x80000000u;
  const unsigned rsv = in.ldv * 2, rsg = in.ldg * 2, rso = ldo * 4;
  const unsigned at_v = col ? 4 * g * rsv + j * 2 : off;
  const unsigned at_g = col ? 4 * g * rsg + j * 2 : off;
  const unsigned at_o = col || ncol ? 4 * g * rso + j * 4 : off;
  const char* vseg =
      (const char*)((const mx_bf16*)in.v + (size_t)t0 * in.ldv + hd * DV);
  const char* gseg =
      MODE == CK_SSD
          ? (const char*)((const mx_bf16*)in.gate + (size_t)t0 * in.ldg +
                          hd * DV)
          : nullptr;
  char* oseg = (char*)(a.out + (size_t)t0 * ldo +
                       hd * (MODE == CK_SSD ? DV : ck_pitch(DV)));
  // chunk c's rows (and more, up to the segment's end) of `p`, `rb` bytes
  // apart, `width` bytes of each
  auto rows_from = [&](const char* p, int c, unsigned rb, unsigned width) {
    const unsigned more = min(n - 32 * c - 1, 32);
    return __builtin_amdgcn_make_buffer_rsrc((void*)(p + (size_t)c * 32 * rb),
                                             0, more * rb + width, 0x00020000);
  };
  const float skip = MODE == CK_SSD ? a.p2[hd] : 0.f;

  struct Cells {  // of this lane's rows, as loaded
    unsigned short v[8], gt[8 / RH];
  };
  struct Block {  // of M: scores, decays (or what lies behind), scales
    ck_f32x4 qk, x, w;
    float y, u1, u2;
  };
  struct Scales {
    ck_f32x4 dr[2 / RH], dk[2];
    float gam;
    unsigned odd;
  };
  // of Q the wave's own token tile first
  ck_u32x4 Q[PART == 1 ? 1 : 2 * WK], K[WT];
  auto fetch_q = [&] {
    const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)g1, 0, Gi::TOTAL,
                                                     0x00020000);
#pragma unroll
    for (int f = 0; f < 2 * WK; ++f)
      Q[f] = __builtin_bit_cast(
          ck_u32x4,
          __builtin_amdgcn_raw_buffer_load_b128(
              r, at16,
              Gi::Q + (((f / WK) ^ rh) * NK + WK * rh + f % WK) * 1024, 0));
  };
  auto fetch_k = [&] {
    const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)g1, 0, Gi::TOTAL,
                                                     0x00020000);
#pragma unroll
    for (int f = 0; f < WT; ++f)
      K[f] = __builtin_bit_cast(
          ck_u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                        r, at16, Gi::K + (WT * rh + f) * 1024, 0));
  };
  auto fetch_cells = [&](int c, Cells& x) {
    c = min(c, count - 1);
    const auto vr = rows_from(vseg, c, rsv, DV * 2);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      x.v[i] = __builtin_amdgcn_raw_buffer_load_b16(
          vr, at_v + ((i >> 2) * 16 + (i & 3)) * rsv, 0, 0);
    if constexpr (MODE == CK_SSD && PART != 1) {
      const auto gr = rows_from(gseg, c, rsg, DV * 2);
#pragma unroll
      for (int i = 0; i < 8 / RH; ++i)
        x.gt[i] = __builtin_amdgcn_raw_buffer_load_b16(
            gr, at_g + ((i >> 2) * 16 + rh * 16 + (i & 3)) * rsg, 0, 0);
    }
  };
  auto head_buffer = [&] {
    return __builtin_amdgcn_make_buffer_rsrc((void*)h2, 0, Hd::TOTAL * 4,
                                             0x00020000);
  };
  auto load4 = [&](__amdgpu_buffer_rsrc_t r, unsigned at, int from) {
    return __builtin_bit_cast(
        ck_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, from, 0));
  };
  auto fetch_block = [&](int h, Block& x) {
    h = min(h, 2);
    const auto r = head_buffer();
    const int b = h == 2 ? 16 : 0;
    x.qk = load4(__builtin_amdgcn_make_buffer_rsrc((void*)g2, 0, Gi::TOTAL,
                                                   0x00020000),
                 at16, Gi::QK + h * 1024);
    x.x = load4(r, g * 16, (h == 1 ? Hd::SUF : Hd::A + b) * 4);
    x.w = load4(r, g * 16, (Hd::W + b) * 4);
    x.y = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
        r, m16 * 4, (h == 1 ? Hd::PRE : Hd::P + b) * 4, 0));
    x.u1 = ((CK_CONST const float*)h2)[Hd::P + b + 7];
    x.u2 = ((CK_CONST const float*)h2)[Hd::P + b + 11];
  };
  auto fetch_scales = [&](Scales& x) {
    const auto r = head_buffer();
    if constexpr (PART != 1) {
#pragma unroll
      for (int mt = 0; mt < 2 / RH; ++mt)
        x.dr[mt] = load4(r, g * 16, (Hd::DR + 16 * (mt + rh)) * 4);
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
      x.dk[mt] = load4(r, g * 16, (Hd::DK + 16 * mt) * 4);
    x.gam = ((CK_CONST const float*)h2)[Hd::GAM];
    x.odd = ((CK_CONST const unsigned*)h2)[Hd::FLAG];
  };
  // a block of M: rows s = 4 g + i of its half, column t = m16 of its own;
  // every decay between them by products of its own
  auto make_block = [&](int h, const Block& x, ck_u32x4* to) {
    h = min(h, 2);
    // no branches: where ways meet, waits are for the latest load of either
    // comparisons made anew, one each: kept, they spill scalar registers within
    // the loop
    int t = m16;
    asm volatile("" : "+v"(t));
    t = h == 1 ? 19 : t;
    const int b = t >> 2;
    float tail = b > g ? x.y : 1.f;
    // the blocks of four between: b 2 and 3 for g 0, b 3 for g 1
    tail *= (unsigned)(b - 2) < (g < 1 ? 2u : 0u) ? x.u1 : 1.f;
    tail *= (unsigned)(b - 3) < (g < 2 ? 1u : 0u) ? x.u2 : 1.f;
    ck_f32x4 e;
    e[3] = h == 1 ? tail * x.x[3] : tail;
#pragma unroll
    for (int i = 2; i >= 0; --i)
      e[i] = h == 1 ? tail * x.x[i]
                    : e[i + 1] * (4 * g + i + 1 <= t ? x.x[i + 1] : 1.f);
    ck_f32x4 m;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      m[i] = 4 * g + i <= t ? x.qk[i] * e[i] * x.w[i] : 0.f;
    CkTerms4 tm = ck_split(m);
    if constexpr (AGAIN) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!(fabsf(m[i]) < INFINITY)) {  // the first term is all of it
          const unsigned low = i & 1 ? 0xffffu : 0xffff0000u;
          const unsigned top = __float_as_uint(m[i] != m[i] ? NAN : m[i]) >> 16;
          tm.h[i >> 1] = (tm.h[i >> 1] & low) | top << (i & 1) * 16;
          tm.m[i >> 1] &= low;
          tm.l[i >> 1] &= low;
        }
    }
    // token tile, half of the lane's eight
    ck_u32x2* dst = (ck_u32x2*)(to + (h == 0 ? 0 : 192) + lane) + (h == 2);
    dst[0] = tm.h;
    dst[128] = tm.m;
    dst[256] = tm.l;
  };

  // a where it is a finite number, else b
  auto either = [](ck_f32x4 a, ck_f32x4 b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = fabsf(a[i]) < INFINITY ? a[i] : b[i];
    return a;
  };
  const ck_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  unsigned odd = 0;  // some chunk's flag
  // Chunk c; what is used makes room for a later chunk's at once. AGAIN: not, and
  // what comes to no finite number is made of the numbers themselves. The three
  // terms of an infinity are not its sum, and an infinite q or k beside a term of
  // zero makes no number of it, where the fp32 products would be infinite.
  auto walk = [&](int c, Cells& cells, Scales& sc, Block& blk) {
    // the next chunk's M
    if constexpr (PART != 1) {
      make_block(wave, blk, &mfrag[(c + 1) & 1][0][0][0]);
      if constexpr (!AGAIN) fetch_block(wave, blk);
    }
    ck_f32x4 V[2], W[2], O[2] = {zero, zero}, X[2] = {zero, zero};
    ck_f32x4 P[2] = {zero, zero};  // O of the numbers themselves
    float gt[8 / RH];
    const int left = n - 32 * c - 4 * g;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float y = __uint_as_float((unsigned)cells.v[i] << 16);
      if (MODE == CK_MLSTM && ncol)
        y = (i >> 2) * 16 + (i & 3) < left ? 1.f : 0.f;
      V[i >> 2][i & 3] = y;
    }
#pragma unroll
    for (int i = 0; i < 8 / RH; ++i)
      gt[i] = __uint_as_float((unsigned)cells.gt[i] << 16);
    const Scales s0 = sc;
    odd |= s0.odd;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!AGAIN) {
      fetch_cells(c + 2, cells);
      fetch_scales(sc);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) W[mt] = V[mt] * s0.dk[mt];
    if constexpr (PART != 1) {
      // values that are no finite numbers are left out here: beside the zeros
      // above M's diagonal they would reach earlier tokens
      ck_f32x4 F[2] = {V[0], V[1]};
      if constexpr (AGAIN) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (!(fabsf(V[i >> 2][i & 3]) < INFINITY)) F[i >> 2][i & 3] = 0.f;
      }
      const ck_u32x4 vb = {
          ck_pack_high(F[0][0], F[0][1]), ck_pack_high(F[0][2], F[0][3]),
          ck_pack_high(F[1][0], F[1][1]), ck_pack_high(F[1][2], F[1][3])};
      const ck_u32x4(*mf)[3][64] = mfrag[c & 1];
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int mt = 0; mt < 2 / RH; ++mt)
          X[mt] = ck_mfma(mf[mt + rh][q][lane], vb, X[mt]);
      if constexpr (AGAIN) {
        // what the left out values add
        float* tmp = vtmp[wave];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          tmp[((i >> 2) * 16 + 4 * g + (i & 3)) * 16 + m16] =
              V[i >> 2][i & 3];
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int s = 0; s < 32; ++s) {
          const float xs = tmp[s * 16 + m16];
          if (fabsf(xs) < INFINITY) continue;
#pragma unroll
          for (int i = 0; i < 8 / RH; ++i) {
            // entry (t, s) of M in fragment order
            const int at = ((s >> 2 & 3) * 16 + 4 * g + (i & 3)) * 8 +
                           (s >> 4) * 4 + (s & 3);
            float a = 0.f;
#pragma unroll
            for (int q = 2; q >= 0; --q)
              a += ps_bf16_to_f32(
                  ((const unsigned short*)mfrag[c & 1][(i >> 2) + rh][q])[at]);
            if (a != 0.f) X[i >> 2][i & 3] += a * xs;
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < WK; ++ks) {
      if constexpr (PART != 1) {
        const CkTerms8 ts = ck_split(S[2 * ks], S[2 * ks + 1]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          O[mt] = ck_mfma(Q[mt * WK + ks], ts.l, O[mt]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          O[mt] = ck_mfma(Q[mt * WK + ks], ts.m, O[mt]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          O[mt] = ck_mfma(Q[mt * WK + ks], ts.h, O[mt]);
      }
      if constexpr (PART != 1 && AGAIN) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int i = 0; i < 8; ++i)
            P[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                ck_bf16(Q[mt * WK + ks], i), S[2 * ks + (i >> 2)][i & 3], P[mt],
                0, 0, 0);
      }
      S[2 * ks] *= s0.gam;
      S[2 * ks + 1] *= s0.gam;
    }
    if constexpr (PART != 1 && AGAIN) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) O[mt] = either(O[mt], P[mt]);
    }
    if constexpr (PART != 1) {
      if constexpr (!AGAIN) fetch_q();
      if constexpr (RH == 2) share[c & 1][wave][lane] = O[1];
    }
    if constexpr (PART == 1) decay *= s0.gam;
    const CkTerms8 tw = ck_split(W[0], W[1]);
    if constexpr (AGAIN) {
#pragma unroll
      for (int t = 0; t < WT; ++t) {
        ck_f32x4 x = S[t];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          x = __builtin_amdgcn_mfma_f32_16x16x4f32(
              ck_bf16(K[t], i), W[i >> 2][i & 3], x, 0, 0, 0);
        S[t] = ck_mfma(K[t], tw.l, S[t]);
        S[t] = ck_mfma(K[t], tw.m, S[t]);
        S[t] = either(ck_mfma(K[t], tw.h, S[t]), x);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int t = 0; t < WT; ++t) S[t] = ck_mfma(K[t], tw.l, S[t]);
#pragma unroll
      for (int t = 0; t < WT; ++t) S[t] = ck_mfma(K[t], tw.m, S[t]);
#pragma unroll
      for (int t = 0; t < WT; ++t) S[t] = ck_mfma(K[t], tw.h, S[t]);
      fetch_k();
      g1 = g2;
      if (c + 3 < count) {
        g2 += gstep;
        h2 += hstep;
      }
    }
    if constexpr (PART != 1) {
      // also: the next chunk's M is there, this one's is read
      __syncthreads();
      if constexpr (RH == 2) O[0] += share[c & 1][wave ^ 1][lane];
      const auto orow =
          rows_from(oseg, c, rso, (MODE == CK_SSD ? DV : DV + 1) * 4);
#pragma unroll
      for (int i = 0; i < 8 / RH; ++i) {
        const int mt = i >> 2, e = i & 3;
        float o = fmaf(O[mt][e], s0.dr[mt][e], X[mt][e]);
        if (MODE == CK_SSD)
          o = fmaf(skip, rh ? V[1][e] : V[mt][e], o) * gt[i] *
              ck_sigmoid(gt[i]);
        __builtin_amdgcn_raw_buffer_store_b32(
            __float_as_uint(o), orow, at_o + (mt * 16 + rh * 16 + e) * rso, 0,
            0);
      }
    }
  };

  Cells ca, cb2;
  Scales sa, sb;
  Block blk;
  const char *gn = g2, *hn = h2;  // chunk 1's
  if (count > 1) {
    gn += gstep;
    hn += hstep;
  }
  if constexpr (PART != 1) {
    const ck_u32x2 none = {0, 0};
    for (int i = threadIdx.x; i < 384; i += 64 * NW * RH)  // tile 0, second half
      ((ck_u32x2*)&mfrag[i / 192][0][i / 64 % 3][i % 64])[1] = none;
    fetch_block(wave, blk);
    make_block(wave, blk, &mfrag[0][0][0][0]);
    __syncthreads();
  }
  if constexpr (AGAIN) {
#pragma unroll 1
    for (int c = 0; c < count; ++c) {
      g1 = a.gitems + ((size_t)(first + c) * G + grp) * Gi::TOTAL;
      g2 = g1;
      h2 = (const char*)(a.hitems + ((size_t)(first + c) * H + hd) * Hd::TOTAL);
      fetch_cells(c, ca);
      fetch_scales(sa);
      fetch_k();
      if constexpr (PART != 1) {
        fetch_q();
        if (c + 1 < count) {
          g2 += gstep;
          h2 += hstep;
        }
        fetch_block(wave, blk);
      }
      walk(c, ca, sa, blk);
    }
  } else {
    // the order in which a chunk's loads are asked for below: the waits of the
    // loop are for what is later in either
    fetch_cells(0, ca);
    fetch_scales(sa);
    __builtin_amdgcn_sched_barrier(0);
    g2 = gn;
    h2 = hn;
    if constexpr (PART != 1) fetch_block(wave, blk);
    __builtin_amdgcn_sched_barrier(0);
    fetch_cells(1, cb2);
    fetch_scales(sb);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PART != 1) fetch_q();
    __builtin_amdgcn_sched_barrier(0);
    fetch_k();
    __builtin_amdgcn_sched_barrier(0);
    g1 = gn;
    if (count > 2) {
      g2 += gstep;
      h2 += hstep;
    }
    int c = 0;
#pragma unroll 1
    for (; c + 1 < count; c += 2) {
      walk(c, ca, sa, blk);
      walk(c + 1, cb2, sb, blk);
    }
    if (c < count) walk(c, ca, sa, blk);
    // A value, key or decay that is no finite number leaves none in the state, and
    // there they stay; the flags tell of the others.
#pragma unroll
    for (int t = 0; t < WT; ++t) odd |= !ck_finite(S[t]);
    if (PART == 1 ? __any(odd) : __syncthreads_or(odd)) return false;
  }
  if (PART == 1 && cb == 0 && threadIdx.x == 0)
    pt[run * rec + (size_t)D * cols] = decay;
  if (PART == 2 && !last) return true;
  int rows = D;  // which rows there are, found again and not kept over the walk
  asm volatile("" : "+s"(rows));
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * (WT * rh + t) + 4 * g + i;
      if (d < rows) {
        if (PART == 1) {
          if (col || ncol) pt[run * rec + (size_t)d * cols + j] = S[t][i];
        } else {
          if (col) Sg[(size_t)d * DV] = S[t][i];
          if (ncol) Ng[d] = S[t][i];
        }
      }
    }
  return true;
}

template <int MODE, int DP, int PART, int NW>
__global__ __launch_bounds__(64 * NW * (DP % 64 == 0 ? 2 : 1),
                             PART == 1 && DP != 96 ? 4 : 2)  // waves a SIMD
void ck_sweep_wide_kernel(CkWideCall a) {
  __shared__ CkWideLds<DP, NW> lds;
  if (ck_walk_wide<MODE, DP, PART, NW, false>(a, lds)) return;
  // the arguments once more, so that nothing is kept for this over the first walk:
  // scalar registers would spill within its loop
  unsigned long at = (unsigned long)__builtin_amdgcn_kernarg_segment_ptr();
  unsigned low = at, high = at >> 32;
  asm volatile("" : "+s"(low), "+s"(high));
  at = (unsigned)__builtin_amdgcn_readfirstlane(low) |
       (unsigned long)(unsigned)__builtin_amdgcn_readfirstlane(high) << 32;
  ck_walk_wide<MODE, DP, PART, NW, true>(
      *(const CkWideCall*)(CK_CONST const CkWideCall*)at, lds);
}

// Read-out norm and gate: o / rms_DV(o) * weight * gate for the rows of
// segments that the sweep walked. A wave takes four heads of a row; a lane
// holds VEC neighbouring columns of each, 64 * VEC >= DV.
template <typename T, int MODE, int VEC>
__global__ __launch_bounds__(256) void ck_readout_kernel(
    T* __restrict__ out, int ldo, const float* __restrict__ raw,
    const T* __restrict__ gate, int ldg, const float* __restrict__ normw,
    const int* __restrict__ seq_rows, int S_, int H, int DV, float eps,
    const float* __restrict__ ge) {
  // the matrix LSTM's rows carry n.q behind a head's columns
  const int pitch = MODE == CK_MLSTM ? ck_pitch(DV) : DV;
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const int h0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 4;
  // rows of short segments are not this kernel's
  bool mine = false;
  for (int s0 = 0; s0 < S_ && !mine; s0 += 64) {
    const int s = s0 + lane;
    bool hit = false;
    if (s < S_) {
      const int a = seq_rows[4 * s], n = seq_rows[4 * s + 1];
      hit = n >= 16 && t >= a && t < a + n;
    }
    mine = __any(hit);
  }
  if (!mine) return;
  const float* r = raw + (size_t)t * ((size_t)H * pitch);
  const T* gp = gate + (size_t)t * ldg;
  T* op = out + (size_t)t * ldo;
  const int c0 = lane * VEC;
  float o[4][VEC], gv[4][VEC], nw[4][VEC], den[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int hd = min(h0 + h, H - 1);
#pragma unroll
    for (int u = 0; u < VEC; ++u) {
      const int c = min(c0 + u, DV - 1);
      o[h][u] = r[hd * pitch + c];
      gv[h][u] = MxElem<T>::ld(gp + hd * DV + c);
      nw[h][u] =
          normw[(MODE == CK_GD || MODE == CK_MLSTM ? hd * DV : 0) + c];
    }
    if (MODE == CK_MLSTM)
      den[h] = fmaxf(fabsf(r[hd * pitch + DV]), ge[(size_t)t * H + hd]) +
               1e-6f;
  }
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    float ss = 0.f;
    if (MODE == CK_MLSTM) {
#pragma unroll
      for (int u = 0; u < VEC; ++u) o[h][u] /= den[h];
    }
#pragma unroll
    for (int u = 0; u < VEC; ++u)
      if (c0 + u < DV) ss += o[h][u] * o[h][u];
    ss = mx_wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)DV + eps);
#pragma unroll
    for (int u = 0; u < VEC; ++u) {
      const float g = gv[h][u];
      float gt = ck_sigmoid(g);
      if (MODE == CK_GLA) gt *= g;
      if (h0 + h < H && c0 + u < DV)
        MxElem<T>::st(op + (h0 + h) * DV + c0 + u,
                      o[h][u] * inv * nw[h][u] * gt);
    }
  }
}

// The same for heads of 8 LPH columns whose rows lie on 16-byte borders: a lane has eight neighbouring columns, LPH lanes a head, so that
// every access is 16 bytes. Whether the rows are this kernel's is asked while they
// are on their way. Bound by memory; us, a lane with one to four columns of four
// heads / this: 8011 rows of 32 bf16 heads of 128 80 / 42 (6.2 TB/s), 6007 rows 55 /
// 33, 1501 rows of 8 heads of 256 15.8 / 7.0.
template <typename T, int MODE, int LPH>
__global__ __launch_bounds__(256) void ck_readout_wide_kernel(
    T* __restrict__ out, int ldo, const float* __restrict__ raw,
    const T* __restrict__ gate, int ldg, const float* __restrict__ normw,
    const int* __restrict__ seq_rows, int S_, int T_, int H, float eps,
    const float* __restrict__ ge) {
  constexpr int DV = 8 * LPH;
  constexpr int PITCH = MODE == CK_MLSTM ? ck_pitch(DV) : DV;
  struct alignas(16) vec8 {
    T e[8];
  };
  const unsigned units = H * LPH;  // of eight columns
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  const unsigned last = (unsigned)T_ * units - 1;
  const unsigned at = min(i, last);
  const int t = at / units, c = (at - t * units) * 8;
  const unsigned hd = c / DV;
  const float* rh = raw + (size_t)t * (H * PITCH) + hd * PITCH;
  const float* r = rh + c % DV;
  ck_f32x4 oa = *(const ck_f32x4*)r, ob = *(const ck_f32x4*)(r + 4);
  float den = 1.f;
  if (MODE == CK_MLSTM)
    den = fmaxf(fabsf(rh[DV]), ge[(size_t)t * H + hd]) + 1e-6f;
  const vec8 gv = *(const vec8*)(gate + (size_t)t * ldg + c);
  const float* w =
      normw + (MODE == CK_GD || MODE == CK_MLSTM ? c : c % DV);
  const ck_f32x4 wa = *(const ck_f32x4*)w, wb = *(const ck_f32x4*)(w + 4);
  // rows of short segments are not this kernel's; a wave has one row or a few
  const int lane = threadIdx.x & 63;
  bool mine = false;
  for (int s0 = 0; s0 < S_; s0 += 64) {
    const int s = min(s0 + lane, S_ - 1);
    const int a = seq_rows[4 * s], n = seq_rows[4 * s + 1];
    unsigned long long left =
        __ballot(s0 + lane < S_ && n >= 16 &&
                 a + n > __builtin_amdgcn_readfirstlane(t));
    while (left) {
      const int k = __ffsll((long long)left) - 1;
      const int first = __builtin_amdgcn_readlane(a, k);
      const int rows = __builtin_amdgcn_readlane(n, k);
      mine |= t >= first && t < first + rows;
      left &= left - 1;
      if (__all(mine)) break;
    }
    if (__all(mine)) break;
  }
  if (MODE == CK_MLSTM) {
    oa /= den;
    ob /= den;
  }
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) ss += oa[u] * oa[u] + ob[u] * ob[u];
#pragma unroll
  for (int d = 1; d < LPH; d <<= 1) ss += __shfl_xor(ss, d, 64);
  const float inv = 1.0f / sqrtf(ss / (float)DV + eps);
  vec8 y;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const float g = MxElem<T>::ld(&gv.e[u]);
    float gt = ck_sigmoid(g);
    if (MODE == CK_GLA) gt *= g;
    MxElem<T>::st(&y.e[u], (u < 4 ? oa[u & 3] : ob[u & 3]) * inv *
                               (u < 4 ? wa[u & 3] : wb[u & 3]) * gt);
  }
  if (mine && i <= last) *(vec8*)(out + (size_t)t * ldo + c) = y;
}

// Key width as the kernels pad it (0: not built).
static int ck_pad(int D) {
  const int pads[] = {32, 64, 96, 128};
  for (int p : pads)
    if (D <= p) return p;
  return 0;
}

// bf16 rows with one decay per head and token go in chunks of 32.
template <typename T, int MODE>
static constexpr bool ck_wide() {
  return MODE >= CK_SSD && sizeof(T) == 2;
}
// Floats per chunk of L rows: of all heads' (and groups') operands.
static long ck_chunk_floats(int mode, int dp, int H, int G, int L) {
  if (L == CK_WIDE)
    return (long)G * (32 * dp + 768) + (long)H * CkWideHead::TOTAL;
  if (mode >= CK_SSD)
    return (long)G * 32 * dp + (long)H * CkHead::TOTAL;
  const int rows = mode == CK_GD ? 4 : (mode == CK_CD ? 3 : 2);
  const int sq = mode == CK_GD ? 3 : (mode == CK_CD ? 2 : 1);
  return H * ((long)rows * 16 * dp + sq * 256 + dp + 4);
}

// Measured (bf16, one MI355X, whole operation; token by token -> this form):
//   general delta 32 heads 128x128, 8011 rows in 2 prompts   12.3 -> 0.68 ms
//     (operands 0.19, walk 0.45, read-out 0.04)
//   channel delta 32 x 128x128, 6007 rows in 3 prompts, 37 single tokens
//                                                            5.42 -> 0.48 ms
//     (operands 0.15, walk 0.27, tokens 0.03, read-out 0.03)
//   ssd 128 heads 128x64, 8192 rows in 2 prompts             6.91 -> 0.30 ms
//   gla 8 heads 128x256, 1501 rows                           2.12 -> 0.06 ms
//   mlstm 32 heads 128x128, 8192 rows in 2 prompts           6.41 -> 0.47 ms
// From 16 rows on a segment goes this way: one chunk costs about 15 us in
// three launches, 16 tokens one by one 24 us.
//
// Chunks laid down at once, and the passes over all of them. A step's segments
// of 16 rows and more have at most T / L + S chunks of L rows, and at most
// 2 T / L (T / 16 of 32); passes keep the scratch below CK_BYTES. They follow
// the chunks of one segment after the other: by chunk number within every
// segment, 256 segments of 48 rows took 250 passes for the one segment that
// could be (general delta, 32 heads of 128 x 128: 27 ms, 2.1 with two passes,
// 3.7 token by token).
#define CK_BYTES (1l << 30)
static void ck_plan(int mode, int T_, int S_, int H, int G, int D, int L,
                    int* cap, int* passes) {
  const long per = ck_chunk_floats(mode, ck_pad(D), H, G, L) * 4;
  long all = (long)T_ / L + S_;
  if (all > T_ / (L / 2) + 1) all = T_ / (L / 2) + 1;
  long fit = CK_BYTES / per;
  if (fit < 1) fit = 1;
  *cap = (int)(all < fit ? all : fit);
  *passes = (int)((all + *cap - 1) / *cap);
}

// Column tiles that a workgroup of the wide walk has: three where four would
// leave waves without columns.
static int ck_wide_tiles(int tiles) {
  return tiles % 3 == 0 && tiles % 4 != 0 ? 3 : 4;
}
// Runs that a segment's chunks are walked in (not the delta forms, whose state
// is multiplied by more than a decay). Two walks of count / runs chunks and
// their start take the place of one of count chunks, so it pays while the
// workgroups of all runs still find room: one a CU of the wide walk (eight
// waves), two of gla's. us in one walk, two, four, eight runs, bf16:
//   ssd    48 heads of 128 x 64, 1 prompt of  300   39   41   42   42
//                                             600   49   48   41   48
//                                            3000  182  133   83   91
//         128 heads,             1 prompt of  600   54   52   58   76
//                                            3000  186  140  149  168
//   mlstm  16 heads of 128 x 128,            3000  218  185  140  146
//   gla     8 heads of 128 x 256,             300   38   41   41   40
//                                             600   48   46   44   47
//                                            1501   88   75   68   71
//          16 heads,                          600   51   54   56   64
//                                            3000  172  160  159  173
// The fp32 walk of ssd and mlstm as it was measured first: four and more.
static int ck_parts(int mode, int T_, int S_, int H, int DV, int L) {
  if (mode == CK_GD || mode == CK_CD) return 1;
  const int tiles = (DV + (mode == CK_MLSTM ? 1 : 0) + 15) / 16;
  const bool narrow = mode != CK_GLA && L != CK_WIDE;
  const int wg = mode == CK_GLA ? 1 : (narrow ? 2 : ck_wide_tiles(tiles));
  const long blocks = (long)S_ * H * ((tiles + wg - 1) / wg);
  const int longest = (T_ - S_ + 1 + 15) / 16;
  long parts = (L == CK_WIDE ? 256 : 512) / blocks;
  if (parts > 16) parts = 16;
  if (parts > longest / 6) parts = longest / 6;
  const int fewest = narrow || longest < 64 ? 4 : 2;
  return parts < fewest || longest < 32 ? 1 : (int)parts;
}
// Floats of the runs' records.
static long ck_part_floats(int mode, int T_, int S_, int H, int D, int DV,
                           int L) {
  const int parts = ck_parts(mode, T_, S_, H, DV, L);
  if (parts == 1) return 0;
  const long rec = mode == CK_GLA ? (long)D * DV + ck_pad(D)
                                  : (long)D * (DV + 1) + 4;
  return (long)S_ * H * parts * rec;
}

#define CK_ARGS                                                              \
  void *out, int ldo, CkIn in, const void *normw, const void *p2,            \
      void *state, void *aux,                                                \
      const void *seq_rows, int S_, int T_, int H, int G, int D, int DV,     \
      float eps, float scale, float c0f, float *scratch, hipStream_t stream

#define CK_PASS                                                              \
  out, ldo, in, normw, p2, state, aux, seq_rows, S_, T_, H, G, D, DV, eps,   \
      scale, c0f, scratch, stream

// Floats of scratch per row: raw read-outs, and the matrix LSTM's gates.
static long ck_rows_floats(int mode, int T_, int H, int DV) {
  if (mode == CK_SSD) return 0;
  return (long)T_ * H * (mode == CK_MLSTM ? ck_pitch(DV) + 3 : DV);
}

template <typename T, int MODE>
static void ck_read(CK_ARGS, const float* raw, const float* gx) {
  const int border = 16 / sizeof(T);
  const size_t at = (size_t)out | (size_t)in.gate | (size_t)normw |
                    (size_t)raw;
  if (at % 16 == 0 && ldo % border == 0 && in.ldg % border == 0 &&
      (long)T_ * H * DV < 1l << 32) {
#define CK_READ(LPH)                                                         \
  case 8 * LPH:                                                              \
    hipLaunchKernelGGL((ck_readout_wide_kernel<T, MODE, LPH>),               \
                       dim3(((long)T_ * H * LPH + 255) / 256), dim3(256), 0, \
                       stream, (T*)out, ldo, raw, (const T*)in.gate, in.ldg, \
                       (const float*)normw, (const int*)seq_rows, S_, T_, H, \
                       eps, gx);                                             \
    return;
    switch (DV) {
      CK_READ(4)
      CK_READ(8)
      CK_READ(16)
      CK_READ(32)
    }
#undef CK_READ
  }
#define CK_READ(VEC)                                                         \
  hipLaunchKernelGGL((ck_readout_kernel<T, MODE, VEC>),                      \
                     dim3(T_, (H + 15) / 16), dim3(256), 0, stream, (T*)out, \
                     ldo, raw, (const T*)in.gate, in.ldg,                    \
                     (const float*)normw, (const int*)seq_rows, S_, H, DV,   \
                     eps, gx)
  if (DV <= 64)
    CK_READ(1);
  else if (DV <= 128)
    CK_READ(2);
  else
    CK_READ(4);
#undef CK_READ
}

template <typename T, int MODE, int DP>
static int ck_launch(CK_ARGS) {
  typedef CkItem<MODE, DP> It;
  int cap, passes;
  ck_plan(MODE, T_, S_, H, G, D, 16, &cap, &passes);
  float* raw = scratch;
  float* items = scratch + ((ck_rows_floats(MODE, T_, H, DV) + 3) & ~3l);
  const int parts = ck_parts(MODE, T_, S_, H, DV, 16);
  float* part = items + (((size_t)cap * H * It::TOTAL + 3) & ~(size_t)3);
  for (int p = 0; p < passes; ++p) {
    hipLaunchKernelGGL((ck_prep_kernel<T, MODE, DP>), dim3(cap, H), dim3(256),
                       0, stream, items, in, (const int*)seq_rows, S_, H, G,
                       D, scale, c0f, p * cap);
#define CK_SWEEP(PART, RUNS)                                                 \
  hipLaunchKernelGGL((ck_sweep_kernel<T, MODE, DP, PART>),                   \
                     dim3(S_ * H * ((DV + 15) / 16) * (RUNS)),               \
                     dim3(DP * 4 / ck_row_tiles(DP)), 0, stream, raw, items, \
                     cap, (const T*)in.v, in.ldv, (float*)state,             \
                     (const int*)seq_rows, S_, H, D, DV, p * cap, part,      \
                     parts)
    if constexpr (MODE == CK_GLA) {
      if (parts > 1) {
        CK_SWEEP(1, parts - 1);
        CK_SWEEP(2, parts);
        continue;
      }
    }
    CK_SWEEP(0, 1);
#undef CK_SWEEP
  }
  ck_read<T, MODE>(CK_PASS, raw, nullptr);
  return 0;
}

template <typename T, int MODE, int DP>
static int ck_launch_scalar(CK_ARGS) {
  int cap, passes;
  ck_plan(MODE, T_, S_, H, G, D, 16, &cap, &passes);
  const bool lstm = MODE == CK_MLSTM;
  float* raw = scratch;
  float* ga = raw + (lstm ? (size_t)T_ * H * ck_pitch(DV) : 0);
  float* gw = ga + (lstm ? (size_t)T_ * H : 0);
  float* ge = gw + (lstm ? (size_t)T_ * H : 0);
  float* gitems = scratch + ((ck_rows_floats(MODE, T_, H, DV) + 3) & ~3l);
  float* hitems = gitems + (size_t)cap * G * CkGroup<DP>::TOTAL;
  const int ncb = (DV + (lstm ? 1 : 0) + 31) / 32;
  const int parts = ck_parts(MODE, T_, S_, H, DV, 16);
  float* part = hitems + (((size_t)cap * H * CkHead::TOTAL + 3) & ~(size_t)3);
  if (lstm)
    hipLaunchKernelGGL((ck_gates_kernel<T>), dim3(S_ * H),
                       dim3(64 * ck_gate_waves(T_, S_, H)), 0,
                       stream, ga, gw, ge, (const T*)in.a, in.lda,
                       (const T*)in.dec, in.lddec, in.p0, in.p1, (float*)aux,
                       (const int*)seq_rows, H, D, c0f);
  // a group's heads over a few blocks where there are many
  const int slices = (H / G + 31) / 32;
  for (int p = 0; p < passes; ++p) {
    hipLaunchKernelGGL((ck_prep_scalar_kernel<T, MODE, DP>),
                       dim3(cap, G, slices), dim3(256), 0, stream, gitems,
                       hitems, in, ga, gw, (const int*)seq_rows, S_, H, G, D,
                       scale, p * cap);
#define CK_SWEEP(PART, RUNS)                                                 \
  hipLaunchKernelGGL((ck_sweep_scalar_kernel<T, MODE, DP, PART>),            \
                     dim3(S_ * H * ncb * (RUNS)), dim3(256), 0, stream,      \
                     lstm ? raw : (float*)out, lstm ? H * ck_pitch(DV) : ldo,    \
                     gitems, hitems, cap, in, (const float*)p2,              \
                     (float*)state, (float*)aux, (const int*)seq_rows, S_,   \
                     H, G, D, DV, p * cap, part, parts)
    if (parts > 1) {
      CK_SWEEP(1, parts - 1);
      CK_SWEEP(2, parts);
    } else {
      CK_SWEEP(0, 1);
    }
#undef CK_SWEEP
  }
  if constexpr (MODE == CK_MLSTM) ck_read<T, MODE>(CK_PASS, raw, ge);
  return 0;
}

template <int MODE, int DP>
static int ck_launch_wide(CK_ARGS) {
  int cap, passes;
  ck_plan(MODE, T_, S_, H, G, D, CK_WIDE, &cap, &passes);
  const bool lstm = MODE == CK_MLSTM;
  float* raw = scratch;
  float* ga = raw + (lstm ? (size_t)T_ * H * ck_pitch(DV) : 0);
  float* gw = ga + (lstm ? (size_t)T_ * H : 0);
  float* ge = gw + (lstm ? (size_t)T_ * H : 0);
  float* gitems = scratch + ((ck_rows_floats(MODE, T_, H, DV) + 3) & ~3l);
  float* hitems = gitems + (size_t)cap * G * (CkWide<DP>::TOTAL / 4);
  const int tiles = (DV + (lstm ? 1 : 0) + 15) / 16;
  const int parts = ck_parts(MODE, T_, S_, H, DV, CK_WIDE);
  float* part = hitems + (size_t)cap * H * CkWideHead::TOTAL;
  if (lstm)
    hipLaunchKernelGGL((ck_gates_kernel<mx_bf16>), dim3(S_ * H),
                       dim3(64 * ck_gate_waves(T_, S_, H)), 0,
                       stream, ga, gw, ge, (const mx_bf16*)in.a, in.lda,
                       (const mx_bf16*)in.dec, in.lddec, in.p0, in.p1,
                       (float*)aux, (const int*)seq_rows, H, D, c0f);
  // a group's heads over a few blocks where there are many
  const int slices = (H / G + 31) / 32;
  for (int p = 0; p < passes; ++p) {
    hipLaunchKernelGGL((ck_prep_wide_kernel<MODE, DP>), dim3(cap, G, slices),
                       dim3(256), 0, stream, (char*)gitems, hitems, in, ga,
                       gw, (const int*)seq_rows, S_, H, G, D, scale, p * cap);
    const CkWideCall call = {
        lstm ? raw : (float*)out, lstm ? H * ck_pitch(DV) : ldo,
        (const char*)gitems, hitems, cap, in, (const float*)p2, (float*)state,
        (float*)aux, (const int*)seq_rows, S_, H, G, D, DV, p * cap, part,
        parts};
#define CK_SWEEP_NW(PART, RUNS, NW)                                          \
  hipLaunchKernelGGL((ck_sweep_wide_kernel<MODE, DP, PART, NW>),             \
                     dim3(S_ * H * ((tiles + NW - 1) / NW) * (RUNS)),        \
                     dim3(64 * NW * (DP % 64 == 0 ? 2 : 1)), 0, stream, call)
#define CK_SWEEP(PART, RUNS)                                                 \
  if (ck_wide_tiles(tiles) == 3)                                             \
    CK_SWEEP_NW(PART, RUNS, 3);                                              \
  else                                                                       \
    CK_SWEEP_NW(PART, RUNS, 4)
    if (parts > 1) {
      CK_SWEEP(1, parts - 1);
      CK_SWEEP(2, parts);
    } else {
      CK_SWEEP(0, 1);
    }
#undef CK_SWEEP
#undef CK_SWEEP_NW
  }
  if constexpr (MODE == CK_MLSTM) ck_read<mx_bf16, MODE>(CK_PASS, raw, ge);
  return 0;
}

template <typename T, int MODE>
static int ck_dispatch(CK_ARGS) {
  switch (ck_pad(D)) {
#define CK_CASE(DP)                                                         \
  case DP:                                                                  \
    if constexpr (ck_wide<T, MODE>())                                       \
      return ck_launch_wide<MODE, DP>(CK_PASS);                             \
    else if constexpr (MODE >= CK_SSD)                                      \
      return ck_launch_scalar<T, MODE, DP>(CK_PASS);                        \
    else                                                                    \
      return ck_launch<T, MODE, DP>(CK_PASS);
    CK_CASE(32)
    CK_CASE(64)
    CK_CASE(96)
    CK_CASE(128)
  }
  return 1;
}

// One unit per form (CK_ONLY), so they build in parallel; unit 0 also
// carries the entry points.
#define CK_UNIT(NAME) extern "C" int NAME(int dtype, CK_ARGS)
CK_UNIT(ck_general);
CK_UNIT(ck_channel);
CK_UNIT(ck_gla);
CK_UNIT(ck_ssd);
CK_UNIT(ck_mlstm);
#define CK_BODY(MODE)                                                       \
  {                                                                         \
    if (dtype == MX_BF16) return ck_dispatch<mx_bf16, MODE>(CK_PASS);       \
    return ck_dispatch<float, MODE>(CK_PASS);                               \
  }
#if !defined(CK_ONLY) || CK_ONLY == 0
CK_UNIT(ck_general) CK_BODY(CK_GD)
#endif
#if !defined(CK_ONLY) || CK_ONLY == 1
CK_UNIT(ck_channel) CK_BODY(CK_CD)
#endif
#if !defined(CK_ONLY) || CK_ONLY == 2
CK_UNIT(ck_gla) CK_BODY(CK_GLA)
#endif
#if !defined(CK_ONLY) || CK_ONLY == 3
CK_UNIT(ck_ssd) CK_BODY(CK_SSD)
#endif
#if !defined(CK_ONLY) || CK_ONLY == 4
CK_UNIT(ck_mlstm) CK_BODY(CK_MLSTM)
#endif

#if !defined(CK_ONLY) || CK_ONLY == 0
// Floats of scratch that the chunk form needs for a step of T_ rows in S_
// segments, 0 where it does not cover it (no segment of 16 rows can be among
// them, or the head widths are not built).
extern "C" long mx_chunk_scratch(int mode, int T_, int S_, int H, int G,
                                 int D, int DV) {
  if (S_ <= 0 || T_ - S_ + 1 < 16 || ck_pad(D) == 0 || DV > 256) return 0;
  // of both element types' forms the larger
  long need = 0;
  for (int L = 16; L <= (mode >= CK_SSD ? CK_WIDE : 16); L += 16) {
    int cap, passes;
    ck_plan(mode, T_, S_, H, G, D, L, &cap, &passes);
    const long x =
        ((ck_rows_floats(mode, T_, H, DV) + 3) & ~3l) +
        ((cap * ck_chunk_floats(mode, ck_pad(D), H, G, L) + 3) & ~3l) +
        ck_part_floats(mode, T_, S_, H, D, DV, L);
    if (x > need) need = x;
  }
  return need;
}

extern "C" int mx_chunk_delta(void* out, int ldo, const void* r, int ldr,
                              const void* k, int ldk, const void* v, int ldv,
                              const void* zw, int ldzw, const void* za,
                              int ldza, const void* g, int ldg,
                              const void* w0, const void* ab,
                              const void* normw, void* state,
                              const void* seq_rows, int S_, int T_, int H,
                              int D, float eps, float decay_scale,
                              void* scratch, int dtype, void* stream) {
  CkIn in = {r, k, v, zw, za, g, ldr, ldk, ldv, ldzw, ldza, ldg,
             (const float*)w0, (const float*)ab};
  return ck_general(dtype, out, ldo, in, normw, nullptr, state, nullptr,
                    seq_rows, S_, T_, H, H, D, D, eps, decay_scale, 0.f,
                    (float*)scratch, (hipStream_t)stream);
}

extern "C" int mx_chunk_gated(void* out, int ldo, const void* q, int ldq,
                              const void* k, int ldk, const void* v, int ldv,
                              const void* beta, int ldb, const void* zdec,
                              int ldzd, const void* zgate, int ldzg,
                              const void* a_log, const void* dt_bias,
                              const void* normw, void* state,
                              const void* seq_rows, int S_, int T_, int H,
                              int G, int D, int DV, float eps, float qscale,
                              void* scratch, int dtype, void* stream) {
  CkIn in = {q, k, v, zdec, beta, zgate, ldq, ldk, ldv, ldzd, ldb, ldzg,
             (const float*)dt_bias, (const float*)a_log};
  return ck_channel(dtype, out, ldo, in, normw, nullptr, state, nullptr,
                    seq_rows, S_, T_, H, G, D, DV, eps, qscale, 0.f,
                    (float*)scratch, (hipStream_t)stream);
}

// mode: 0 gla, 1 ssd, 2 mlstm, arguments as mx_linear_scan's
extern "C" int mx_chunk_scan(
    int mode, void* out, int ldo, const void* q, int ldq, const void* k,
    int ldk, const void* v, int ldv, const void* dec, int lddec,
    const void* wr, int ldwr, const void* gate, int ldg, const void* p0,
    const void* p1, const void* p2, const void* normw, void* state, void* aux,
    const void* seq_rows, int S_, int T_, int H, int G, int D, int DV,
    float eps, float qscale, float c0, void* scratch, int dtype,
    void* stream) {
  CkIn in = {q, k, v, dec, wr, gate, ldq, ldk, ldv, lddec, ldwr, ldg,
             (const float*)p0, (const float*)p1};
#define CK_SCAN                                                              \
  (dtype, out, ldo, in, normw, p2, state, aux, seq_rows, S_, T_, H, G, D,    \
   DV, eps, qscale, c0, (float*)scratch, (hipStream_t)stream)
  switch (mode) {
    case 0: return ck_gla CK_SCAN;
    case 1: return ck_ssd CK_SCAN;
    case 2: return ck_mlstm CK_SCAN;
  }
  return 1;
}
#endif
