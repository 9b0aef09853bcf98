// Single tokens of attention whose raw scores are mixed over 32 heads, bfloat16 and
// fp32, on the matrix cores:
//     s_h = (q_h . k) scale,  s'_h = sum_j talk[h, j] s_j,
// softmax over the visible keys (aligned chunks, trailing window, sink in the
// denominator), weights times values. Paged cache as talk_attention.hip; head widths
// 64 or 128, KV heads of a multiple of four heads.
//
// Two waves (four, with half of a value row each, at widths of 128) walk tiles of 16
// keys, each with the output of 16 heads and the raw scores of its part of them; the
// scores go to all through LDS, nothing else needs an exchange between lanes (g =
// lane / 16, n = lane % 16):
//   scores  Q K^T, 16 heads as rows, keys as columns, one KV head at a time: of its
//           product only the four rows of its heads are taken, which are those of one
//           lane group, so that lane (g, n) ends up with heads 4 g + i of key n;
//   mix     S^T talk^T with v_mfma_f32_16x16x4_f32 (no term is rounded): the scores
//           of a half are left operands as they are, heads 4 g + i being step i, and
//           the result has keys 4 g + i of the wave's head n;
//   output  in fp32 by v_mfma_f32_4x4x1_16b_f32, sixteen blocks of 4 heads by 4
//           entries: a block is a lane group's key 4 g + i and a KV head, whose weights
//           are in its four lanes. Four sums of an output, one a lane group, are added
//           at the end.
// Keys and values go from memory into operands, a whole tile ahead. The four (two)
// such groups of a workgroup take turns at the tiles, and so do `KS` workgroups of a
// token (records merged by mx_attn_records).
//
// Bound by keys and values where there are enough tokens (64 of up to 2250 keys of 8
// x 128, bf16 77 us, 4.4 TB/s), by the latency of a tile and the merges of the groups
// and records otherwise. us, by the vector kernel of talk_attention.hip (which remains
// for other shapes) -> this one: 870 -> 77 there; 5 tokens of up to 2048 keys 255 ->
// 27, one of 8 90 -> 9, fp32 64 of up to 2250 1470 -> 148, bf16 of 64 428 -> 40. All 32
// heads by one wave, the output on 16 x 16 x 4 with weights of 0 in three of four
// columns: 101, 44, 18, 214, 55; by one wave on 4 x 4: spills at widths of 128 (198),
// 43 at 64; by two: 158 and 40.
#include "attn_common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tt_bf16x8;

struct TtArgs {
  void* out;
  int ldout;
  const void* q;
  int ldq;
  const void *kc, *vc;  // [NB, G, BS, D], [NB, G, BS, vr]
  int vr;
  const int* block_tables;
  int max_blocks;
  const int *token_seq, *token_pos;
  const float* talk;  // [32, 32]
  int T, G, BS;
  float scale;
  int chunk, window, sink;
  float cap;  // 0: none
  const float* sink_vals;
  int KS;
  float* part;  // [T, KS, 32, DV + 4]
};

#define TT_H 32

PS_DEV bool tt_odd(float x) { return !(fabsf(x) < INFINITY); }

// How far a score of bf16 rows may be above the one that set the reference that weights
// are relative to, before it moves; the reference is as much above it, so that no weight
// is above 1. Moving it is a product per sum. fp32 rows take the maximum itself: the
// distance of the largest scores to a reference above them is rounded (single tokens,
// errors against 64 bits 5.2e-7 so and 3.6e-7, the vector kernel's 4.6e-7; four sums of a
// score and two of a mix for two and one among it; 142 -> 148 us for 64 of up to 2250
// keys, portions 64 -> 67).
#define TT_FAR 8.f

// What a lane has of a tile, in 16-byte pieces of P entries: KF of key n for a KV head,
// every fourth one, and of key 4 g + i of the KV head of lane & 12 likewise.
template <typename T, int D>
struct TtLay;
template <int D>
struct TtLay<mx_bf16, D> {
  static constexpr int KF = D / 32, P = 8;
  static PS_DEV float value(const unsigned int* w, int e) {
    return __uint_as_float(e & 1 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16);
  }
};
template <int D>
struct TtLay<float, D> {
  static constexpr int KF = D / 16, P = 4;
  static PS_DEV float value(const unsigned int* w, int e) {
    return __uint_as_float(w[e]);
  }
};

PS_DEV float tt_quad(float v, int i) {  // that of lane i of the four
  const int u = __float_as_int(v);
  return __int_as_float(
      i == 0   ? __builtin_amdgcn_update_dpp(0, u, 0x00, 15, 15, true)
      : i == 1 ? __builtin_amdgcn_update_dpp(0, u, 0x55, 15, 15, true)
      : i == 2 ? __builtin_amdgcn_update_dpp(0, u, 0xaa, 15, 15, true)
               : __builtin_amdgcn_update_dpp(0, u, 0xff, 15, 15, true));
}

// Sums of four numbers over the lane groups: group g has that of number
// (g & 1) * 2 + g / 2.
PS_DEV float tt_gather(kv_f32x4 v) {
  float h[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(v[2 * i]), __float_as_uint(v[2 * i + 1]), false, false);
    h[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  const auto r = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(h[0]), __float_as_uint(h[1]), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename T, int D, int DV>
__global__ __launch_bounds__(512, 2) void talk_token_kernel(TtArgs a) {
  typedef TtLay<T, D> L;
  constexpr bool BF = sizeof(T) == 2;
  constexpr int KF = L::KF, P = L::P;
  // waves that share a value row, entries of it that a lane has, and pieces
  constexpr int SP = DV == 128 || (!BF && D == 128) ? 2 : 1;
  constexpr int NE = DV / SP / 4, VF = NE / P;
  constexpr int KB = 4 / SP;       // KV heads (4 heads each) of a wave's scores
  constexpr int NG = 4 / SP;       // tiles of a workgroup at a time
  constexpr int PA = DV + 4;
  extern __shared__ __align__(16) float sA[];  // [NG][32][PA]: the merge
  __shared__ float s_m[NG][TT_H], s_l[NG][TT_H];
  // scores of every other tile
  __shared__ __align__(16) kv_f32x4 s_sc[2][NG][2][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / (2 * SP), hf = wave / SP % 2, sp = wave % SP;
  const int g = lane >> 4, n = lane & 15;
  const int ks = blockIdx.x / a.T, tok = blockIdx.x - ks * a.T;
  const int pos = a.token_pos[tok];
  const int* table = a.block_tables + (size_t)a.token_seq[tok] * a.max_blocks;
  int lo = 0;
  if (a.chunk > 0) lo = pos / a.chunk * a.chunk;
  if (a.window > 0) lo = max(lo, pos - a.window + 1);
  const int nt = (pos - lo) / 16 + 1;
  const int G = a.G, BS = a.BS, rep = TT_H / G;
  const T* kc = (const T*)a.kc;
  const T* vc = (const T*)a.vc;

  // queries: left operands, row n is head 16 hf + n. Those of fp32 stay in LDS (in
  // registers they spill at widths of 128: 148 us became 199)
  constexpr int PQ = BF ? 0 : D + 4;
  __shared__ __align__(16) float s_q[BF ? 4 : TT_H * PQ];
  uint4 qf[BF ? KF : 1];
  const T* qp = (const T*)a.q + (size_t)tok * a.ldq;
  if constexpr (BF) {
#pragma unroll
    for (int f = 0; f < KF; ++f)
      qf[f] = *(const uint4*)(qp + (16 * hf + n) * D + (4 * f + g) * P);
  } else {
    for (int i = tid; i < TT_H * D / 4; i += 512)
      *(float4*)(s_q + i / (D / 4) * PQ + i % (D / 4) * 4) =
          *(const float4*)(qp + i * 4);
    __syncthreads();
  }
  const float* sq = s_q + (16 * hf + n) * PQ + g * P;
  // right operands of the mix: column n is output head 16 hf + n, step (h, i) takes
  // heads 16 h + 4 g + i
  float tb[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      tb[h][i] =
          a.talk[(16 * hf + n) * TT_H + 16 * h + 4 * g + i] * a.scale;

  float m = PS_NEG_INF, l = 0.f;
  // acc[e][i]: head 16 hf + (n & 12) + i, this lane's entry e
  kv_f32x4 acc[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) acc[e] = kv_f32x4{0.f, 0.f, 0.f, 0.f};
  // this lane's key of tile t, past the end the last one; its row, less the KV
  // head's
  auto key_of = [&](int t) { return min(lo + t * 16 + n, pos); };
  auto row_of = [&](int t, int page) { return page * G * BS + key_of(t) % BS; };
  uint4 kb[KB][KF], vb[4][VF];
  const int64_t vhead = (int64_t)((16 * hf + (n & 12)) / rep) * BS;
  auto fetch_k = [&](int s, int row) {
    const int head = (16 * hf + 4 * (KB * sp + s)) / rep;
    const T* p = kc + (row + (int64_t)head * BS) * D + g * P;
#pragma unroll
    for (int f = 0; f < KF; ++f) kb[s][f] = *(const uint4*)(p + 4 * f * P);
  };
  auto fetch_v = [&](int i, int row) {
    const T* p = vc + (__shfl(row, 4 * g + i, 64) + vhead) * a.vr +
                 DV / SP * sp + (n & 3) * P;
#pragma unroll
    for (int f = 0; f < VF; ++f) vb[i][f] = *(const uint4*)(p + 4 * f * P);
  };
  const int step = NG * a.KS, t0 = ks * NG;
  // pages two tiles ahead; tiles past the last repeat it, hidden
  int page = 0, tn = 0;
  if (t0 < nt) {
    tn = min(t0 + grp, nt - 1);
    const int row = row_of(tn, table[key_of(tn) / BS]);
    tn = min(t0 + grp + step, nt - 1);
    page = table[key_of(tn) / BS];
#pragma unroll
    for (int s = 0; s < KB; ++s) fetch_k(s, row);
#pragma unroll
    for (int i = 0; i < 4; ++i) fetch_v(i, row);
  }
  int turn = 0;
  for (int tw = t0; tw < nt; tw += step) {
    const int t = tw + grp;
    const int next = row_of(tn, page);
    tn = min(t + 2 * step, nt - 1);
    page = table[key_of(tn) / BS];
    kv_f32x4 sc[2], x;
#pragma unroll
    for (int s = 0; s < KB; ++s) {
      // sums of every other piece (fourth one): shorter chains of roundings
      constexpr int NS = BF ? 2 : 4;
      kv_f32x4 st[NS];
#pragma unroll
      for (int f = 0; f < NS; ++f) st[f] = kv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int f = 0; f < KF; ++f) {
        if constexpr (BF) {
          st[f % NS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(tt_bf16x8, qf[f]),
              __builtin_bit_cast(tt_bf16x8, kb[s][f]), st[f % NS], 0, 0, 0);
        } else {
          const float4 q = *(const float4*)(sq + 4 * f * P);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            st[f % NS] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                (&q.x)[e], __uint_as_float((&kb[s][f].x)[e]), st[f % NS], 0, 0,
                0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // no load earlier, it would spill
      fetch_k(s, next);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sc[0][i] = s == 0 || g == KB * sp + s
                       ? (BF ? st[0][i] + st[1][i]
                             : (st[0][i] + st[1][i]) +
                                   (st[NS - 2][i] + st[NS - 1][i]))
                       : sc[0][i];
    }
    if (SP == 1 || g / KB == sp) s_sc[turn][grp][hf][lane] = sc[0];
    __syncthreads();
    sc[0] = s_sc[turn][grp][0][lane];
    sc[1] = s_sc[turn][grp][1][lane];
    turn ^= 1;
    // mixed scores: keys 4 g + i of head 16 hf + n
    x = kv_f32x4{0.f, 0.f, 0.f, 0.f};
    kv_f32x4 y = x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x = __builtin_amdgcn_mfma_f32_16x16x4f32(sc[0][i], tb[0][i], x, 0, 0, 0);
      y = __builtin_amdgcn_mfma_f32_16x16x4f32(sc[1][i], tb[1][i], y, 0, 0, 0);
    }
    x += y;
    const int left = pos - lo - t * 16 - 4 * g;  // keys 4 g + i up to this i
    float mx = PS_NEG_INF;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = x[i];
      if (a.cap > 0.f) v = a.cap * tanhf(v / a.cap);
      x[i] = i <= left ? v : -INFINITY;
      mx = fmaxf(mx, x[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m)) {
      const float mn = mx > m ? (BF ? mx + TT_FAR : mx) : m;
      const float al = expf(m - mn);
      m = mn;
      l *= al;
      if (tw != t0) {
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = tt_quad(al, i);
#pragma unroll
        for (int e = 0; e < NE; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[e][i] *= f[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = expf(x[i] - m);
      l += x[i];
    }
    if (t >= nt - 1) {
      // keys past the last repeat it, with weights of 0
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int f = 0; f < VF; ++f)
          if (i > left) vb[i][f] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int e = 0; e < NE; ++e)
        acc[e] = __builtin_amdgcn_mfma_f32_4x4x1f32(
            x[i], L::value(&vb[i][e / P].x, e % P), acc[e], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      fetch_v(i, next);
    }
  }

  // merge of the tiles' groups; a lane group has the sums of one of four heads
  float* sw = sA + grp * TT_H * PA;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0 && sp == 0) {
    s_m[grp][16 * hf + n] = m;
    s_l[grp][16 * hf + n] = l;
  }
  float* so = sw + (16 * hf + (n & 12) + (g & 1) * 2 + g / 2) * PA +
              DV / SP * sp + (n & 3) * P;
#pragma unroll
  for (int e = 0; e < NE; e += 4) {
    *(float4*)(so + e / P * 4 * P + e % P) =
        make_float4(tt_gather(acc[e]), tt_gather(acc[e + 1]),
                    tt_gather(acc[e + 2]), tt_gather(acc[e + 3]));
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  constexpr int VPR = DV / 4;
#pragma unroll
  for (int u = 0; u < TT_H * VPR / 512; ++u) {
    const int idx = u * 512 + tid, head = idx / VPR, d = idx % VPR * 4;
    float mh = PS_NEG_INF;
#pragma unroll
    for (int w = 0; w < NG; ++w) mh = fmaxf(mh, s_m[w][head]);
    const bool sink = a.sink && ks == 0;  // the sink is share 0's
    const float sv = a.sink_vals != nullptr ? a.sink_vals[head] : 0.f;
    if (sink) mh = fmaxf(mh, sv);
    float lt = sink ? expf(sv - mh) : 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NG; ++w) {
      if (s_m[w][head] == PS_NEG_INF && s_l[w][head] == 0.f) continue;
      const float f = expf(s_m[w][head] - mh);
      const float4 v = *(const float4*)(sA + (w * TT_H + head) * PA + d);
      lt += s_l[w][head] * f;
      o[0] += v.x * f;
      o[1] += v.y * f;
      o[2] += v.z * f;
      o[3] += v.w * f;
    }
    if (a.KS == 1) {
      const float f = 1.0f / lt;
      T* dst = (T*)a.out + (size_t)tok * a.ldout + head * DV + d;
#pragma unroll
      for (int e = 0; e < 4; ++e) MxElem<T>::st(dst + e, o[e] * f);
    } else {
      float* rec = a.part + (((size_t)tok * a.KS + ks) * TT_H + head) * PA;
      if (d == 0) {
        rec[0] = mh;
        rec[1] = lt;
      }
      if (lt != 0.f)  // else no key of this share: no sums
        *(float4*)(rec + 4 + d) = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
}

// ---------------------------------------------------------------------------
// Prompt portions in fp32: as above, four consecutive rows a workgroup, whose eight
// waves take one tile of 16 keys at a time. A KV head's four heads of four rows are 16
// rows of one product, one KV head a wave, so that no part of it is idle; the way
// through LDS hands every wave the scores of its rows (one, or two with half of the
// value entries at widths of 128) as left operands of the mix. Queries stay in LDS.
//
// A tile takes 5100 cycles of a SIMD's matrix unit (8192 of 20000 for the scores, 2048
// for the mix, 8192 for the output, over four SIMDs) and 64 KB of keys and of values
// from the L2 each. us, by the vector kernel of talk_attention.hip -> this one, heads of
// 128: 149 rows behind 817 keys 4390 -> 71, 1000 rows 4520 -> 188 (a third of the fp32
// matrix rate: the phases between two barriers are the same in all waves), 80 rows
// behind 334 1800 -> 39; of 64 2460 -> 47, 2550 -> 121, 1010 -> 27.
// Hidden keys of a row have weights of zero, which values that are not finite would
// carry into its sums; where sums are not finite the walk goes again with those kept
// out of the products and added, weighted, to the rows that see them.
template <int D, int DV>
__global__ __launch_bounds__(512, 2) void talk_rows_f32_kernel(TtArgs a) {
  constexpr int KF = D / 16, P = 4;
  constexpr int SP = DV / 64;          // waves that share a value row
  constexpr int TW = SP;               // rows of a wave
  constexpr int NE = 16, VF = 4;
  // values when the keys are read, keys when half of the values are: with both a
  // tile ahead registers spill
  constexpr bool LATE = TW == 2;
  constexpr int PQ = D + 4, TQ = TT_H * PQ + 16;
  extern __shared__ __align__(16) float s_q[];  // [4][TQ]
  __shared__ __align__(16) kv_f32x4 s_sc[2][4][2][64];
  __shared__ int s_seq[4], s_pos[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hf = wave >> 2, sp = wave % SP, r0 = wave % 4 / SP * TW;
  const int g = lane >> 4, n = lane & 15;
  // rows that see the most keys first
  const int ks = blockIdx.x % a.KS;
  const int tok0 = ((a.T + 3) / 4 - 1 - blockIdx.x / a.KS) * 4;
  const int ntok = min(4, a.T - tok0);
  const int G = a.G, BS = a.BS, rep = TT_H / G;
  const float* kc = (const float*)a.kc;
  const float* vc = (const float*)a.vc;
  if (tid < 4) {
    const int t = tok0 + min(tid, ntok - 1);
    s_seq[tid] = a.token_seq[t];
    s_pos[tid] = a.token_pos[t];
  }
  for (int i = tid; i < 4 * TT_H * D / 4; i += 512) {
    const int r = i / (TT_H * D / 4), c = i % (TT_H * D / 4);
    *(float4*)(s_q + r * TQ + c / (D / 4) * PQ + c % (D / 4) * 4) =
        *(const float4*)((const float*)a.q +
                         (size_t)(tok0 + min(r, ntok - 1)) * a.ldq + c * 4);
  }
  // left operands: row n is head 4 wave + n % 4 of token n / 4
  const float* sq = s_q + (n >> 2) * TQ + (4 * wave + (n & 3)) * PQ + g * P;
  float tb[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      tb[h][i] =
          a.talk[(16 * hf + n) * TT_H + 16 * h + 4 * g + i] * a.scale;
  __syncthreads();

  auto low = [&](int p) {
    int lo = 0;
    if (a.chunk > 0) lo = p / a.chunk * a.chunk;
    if (a.window > 0) lo = max(lo, p - a.window + 1);
    return lo;
  };
  const int khead = 4 * wave / rep * BS;
  const int vhead = (16 * hf + (n & 12)) / rep * BS;
  int my_pos[TW], my_lo[TW];
#pragma unroll
  for (int q = 0; q < TW; ++q) {
    my_pos[q] = __builtin_amdgcn_readfirstlane(s_pos[r0 + q]);
    my_lo[q] = low(my_pos[q]);
  }
  float m[TW], l[TW];
  kv_f32x4 acc[TW][NE];
  bool careful = false;
#pragma unroll 1
  for (;;) {
#pragma unroll
    for (int q = 0; q < TW; ++q) {
      m[q] = PS_NEG_INF;
      l[q] = 0.f;
#pragma unroll
      for (int e = 0; e < NE; ++e) acc[q][e] = kv_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int turn = 0, rs = 0;
    while (rs < ntok) {
      // rows rs .. re - 1 continue one sequence
      int re = rs + 1;
      while (re < ntok && s_seq[re] == s_seq[rs] &&
             s_pos[re] == s_pos[re - 1] + 1)
        ++re;
      const int* table = a.block_tables + (size_t)s_seq[rs] * a.max_blocks;
      const int kmin = low(s_pos[rs]), kmax = s_pos[re - 1];
      const int nt = (kmax - kmin) / 16 + 1;
      auto key_of = [&](int t) { return min(kmin + t * 16 + n, kmax); };
      auto row_of = [&](int t, int page) {
        return page * G * BS + key_of(t) % BS;
      };
      float4 kb[KF], vb[4][VF];
      auto fetch_k = [&](int row) {
        const float* p = kc + ((int64_t)row + khead) * D + g * P;
#pragma unroll
        for (int f = 0; f < KF; ++f) kb[f] = *(const float4*)(p + 4 * f * P);
      };
      auto fetch_v = [&](int i, int row) {
        const float* p =
            vc + ((int64_t)__shfl(row, 4 * g + i, 64) + vhead) * a.vr + 64 * sp +
            (n & 3) * P;
#pragma unroll
        for (int f = 0; f < VF; ++f)
          vb[i][f] = *(const float4*)(p + 4 * f * P);
      };
      // pages two tiles ahead; tiles past the last repeat it, unread
      int tn = min(ks, nt - 1);
      int row = row_of(tn, table[key_of(tn) / BS]);
      tn = min(ks + a.KS, nt - 1);
      int page = table[key_of(tn) / BS];
      fetch_k(row);
      if constexpr (!LATE)
#pragma unroll
        for (int i = 0; i < 4; ++i) fetch_v(i, row);
      for (int t = ks; t < nt; t += a.KS) {
        const int next = row_of(tn, page);
        tn = min(t + 2 * a.KS, nt - 1);
        page = table[key_of(tn) / BS];
        kv_f32x4 st[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) st[f] = kv_f32x4{0.f, 0.f, 0.f, 0.f};
        // sums of every fourth piece: shorter chains of roundings
#pragma unroll
        for (int f = 0; f < KF; ++f) {
          const float4 q = *(const float4*)(sq + 4 * f * P);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            st[f & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                (&q.x)[e], (&kb[f].x)[e], st[f & 3], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // no load earlier, it would spill
        if constexpr (LATE) {
#pragma unroll
          for (int i = 0; i < 4; ++i) fetch_v(i, row);
        } else {
          fetch_k(next);
        }
        // heads 4 wave + i of token g: group wave % 4 of its half's operand
        s_sc[turn][g][hf][16 * (wave & 3) + n] =
            (st[0] + st[1]) + (st[2] + st[3]);
        __syncthreads();
        const int j0 = kmin + t * 16 + 4 * g;
        float x[TW][4];
        bool seen[TW][4];
#pragma unroll
        for (int q = 0; q < TW; ++q) {
          const int r = r0 + q;
          const kv_f32x4 s0 = s_sc[turn][r][0][lane];
          const kv_f32x4 s1 = s_sc[turn][r][1][lane];
          kv_f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(s0[i], tb[0][i], y, 0, 0,
                                                     0);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(s1[i], tb[1][i], y, 0, 0,
                                                     0);
          // keys 4 g + i of head 16 hf + n
          const int hi = r >= rs && r < re ? my_pos[q] : -1;
          float mx = PS_NEG_INF;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float v = y[i];
            if (a.cap > 0.f) v = a.cap * tanhf(v / a.cap);
            // a score that is no number hides its key
            seen[q][i] = j0 + i >= my_lo[q] && j0 + i <= hi && v > PS_NEG_INF;
            x[q][i] = seen[q][i] ? v : -INFINITY;
            mx = fmaxf(mx, x[q][i]);
          }
          mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
          mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
          if (__any(mx > m[q])) {
            const float mn = fmaxf(mx, m[q]);
            const float al = expf(m[q] - mn);
            m[q] = mn;
            l[q] *= al;
            float f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) f[i] = tt_quad(al, i);
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
              for (int i = 0; i < 4; ++i) acc[q][e][i] *= f[i];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x[q][i] = expf(x[q][i] - m[q]);
            l[q] += x[q][i];
          }
        }
        turn ^= 1;
        if (careful) {
#pragma unroll
          for (int q = 0; q < TW; ++q) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              // weights of the four heads, below 0 where the key is hidden
              const float own = seen[q][i] ? x[q][i] : -1.f;
              float w[4];
#pragma unroll
              for (int u = 0; u < 4; ++u) w[u] = tt_quad(own, u);
#pragma unroll
              for (int e = 0; e < NE; ++e) {
                const float v = (&vb[i][e / P].x)[e % P];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                  if (tt_odd(v) && !(w[u] < 0.f)) acc[q][e][u] += w[u] * v;
              }
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < NE; ++e) {
              float& v = (&vb[i][e / P].x)[e % P];
              if (tt_odd(v)) v = 0.f;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int e = 0; e < NE; ++e)
#pragma unroll
            for (int q = 0; q < TW; ++q)
              acc[q][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(
                  x[q][i], (&vb[i][e / P].x)[e % P], acc[q][e], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (!LATE)
            fetch_v(i, next);
          else if (i == 1)
            fetch_k(next);
        }
        row = next;
      }
      rs = re;
    }
    bool odd = false;
#pragma unroll
    for (int q = 0; q < TW; ++q)
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) odd |= tt_odd(acc[q][e][i]);
    if (!__syncthreads_or(odd) || careful) break;
    careful = true;
  }

  // a lane group has the sums of one of four heads
  const int own = (n & 12) + (g & 1) * 2 + g / 2, head = 16 * hf + own;
  const float sv = a.sink_vals != nullptr ? a.sink_vals[head] : 0.f;
#pragma unroll
  for (int q = 0; q < TW; ++q) {
    float lt = l[q];
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
    lt = __shfl(lt, own, 64);
    float mt = __shfl(m[q], own, 64), f = 1.f;
    if (a.sink && ks == 0) {  // the sink is share 0's
      const float mn = fmaxf(mt, sv);
      f = expf(mt - mn);
      lt = lt * f + expf(sv - mn);
      mt = mn;
    }
    const int r = r0 + q, tok = tok0 + r;
    const int at = 64 * sp + (n & 3) * P;
    float* rec = a.part + (((size_t)tok * a.KS + ks) * TT_H + head) * (DV + 4);
    if (a.KS > 1 && at == 0 && r < ntok) {
      rec[0] = mt;
      rec[1] = lt;
    }
    float* dst = a.KS > 1 ? rec + 4
                          : (float*)a.out + (size_t)tok * a.ldout + head * DV;
    if (a.KS == 1) f /= lt;
    const bool put = r < ntok && (a.KS == 1 || lt != 0.f);
#pragma unroll
    for (int e = 0; e < NE; e += 4) {
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = tt_gather(acc[q][e + i]) * f;
      if (put)
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[at + e * 4 + i] = o[i];
    }
  }
}

extern "C" void mx_attn_records(void* out, int ldout, const void* part, int T_,
                                int H, int DV, int KS, int counted,
                                int dtype, void* stream);

template <typename T, int D, int DV>
static int tt_launch(const TtArgs& a, hipStream_t stream) {
  // four tiles of a workgroup at a time, or two
  const int groups = DV == 128 || (sizeof(T) == 4 && D == 128) ? 2 : 4;
  const size_t lds = (size_t)groups * TT_H * (DV + 4) * 4;
  if (hipFuncSetAttribute((const void*)talk_token_kernel<T, D, DV>,
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  hipLaunchKernelGGL((talk_token_kernel<T, D, DV>), dim3(a.T * a.KS), dim3(512),
                     lds, stream, a);
  return 0;
}

// Returns 0 when launched, 1 when the shape is outside this kernel: 32 heads, KV
// heads of 4, 8, 16 or 32 of them, widths 64 or 128, rows on 16-byte borders.
// scratch fp32 [T, splits, 32, DV + 4] when splits > 1.
extern "C" int mx_talk_token(
    void* out, int ldout, const void* q, int ldq, const void* kc,
    const void* vc, const void* block_tables, int max_blocks,
    const void* token_seq, const void* token_pos, const void* talk, int T_,
    int H, int G, int D, int DV, int BS, float scale, int chunk, int window,
    int sink, float softcap, const void* sink_vals, int vrow, int dtype,
    int splits, void* scratch, void* stream) {
  if (T_ <= 0) return 0;
  if (splits > 16) return 1;
  const int vec = dtype == MX_BF16 ? 8 : 4;
  if (H != TT_H || G < 1 || H % G || H / G % 4 || BS < 1) return 1;
  if ((D != 64 && D != 128) || (DV != 64 && DV != 128)) return 1;
  if (ldq % vec || vrow % vec || vrow < DV ||
      (((size_t)q | (size_t)kc | (size_t)vc) & 15))
    return 1;
  const TtArgs a = {out, ldout, q, ldq, kc, vc, vrow,
                    (const int*)block_tables, max_blocks,
                    (const int*)token_seq, (const int*)token_pos,
                    (const float*)talk, T_, G, BS, scale, chunk, window, sink,
                    softcap > 0.f ? softcap : 0.f, (const float*)sink_vals,
                    splits > 1 && scratch != nullptr ? splits : 1,
                    (float*)scratch};
  hipStream_t s = (hipStream_t)stream;
  int rc = 1;
  MX_DISPATCH_DTYPE(dtype, {
    if (D == 64)
      rc = DV == 64 ? tt_launch<T, 64, 64>(a, s) : tt_launch<T, 64, 128>(a, s);
    else
      rc = DV == 64 ? tt_launch<T, 128, 64>(a, s)
                    : tt_launch<T, 128, 128>(a, s);
  })
  if (rc == 0 && a.KS > 1)
    mx_attn_records(out, ldout, scratch, T_, H, DV, a.KS, 0, dtype, stream);
  return rc;
}

template <int D, int DV>
static int tt_launch_rows(const TtArgs& a, hipStream_t stream) {
  const size_t lds = (size_t)4 * (TT_H * (D + 4) + 16) * 4;
  if (hipFuncSetAttribute((const void*)talk_rows_f32_kernel<D, DV>,
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  hipLaunchKernelGGL((talk_rows_f32_kernel<D, DV>), dim3((a.T + 3) / 4 * a.KS),
                     dim3(512), lds, stream, a);
  return 0;
}

// The same for prompt portions, fp32.
extern "C" int mx_talk_rows_f32(
    void* out, int ldout, const void* q, int ldq, const void* kc,
    const void* vc, const void* block_tables, int max_blocks,
    const void* token_seq, const void* token_pos, const void* talk, int T_,
    int H, int G, int D, int DV, int BS, float scale, int chunk, int window,
    int sink, float softcap, const void* sink_vals, int vrow, int splits,
    void* scratch, void* stream) {
  if (T_ <= 0) return 0;
  if (splits > 16) return 1;
  if (H != TT_H || G < 1 || H % G || H / G % 4 || BS < 1) return 1;
  if ((D != 64 && D != 128) || (DV != 64 && DV != 128)) return 1;
  if (ldq % 4 || vrow % 4 || vrow < DV ||
      (((size_t)q | (size_t)kc | (size_t)vc) & 15))
    return 1;
  const TtArgs a = {out, ldout, q, ldq, kc, vc, vrow,
                    (const int*)block_tables, max_blocks,
                    (const int*)token_seq, (const int*)token_pos,
                    (const float*)talk, T_, G, BS, scale, chunk, window, sink,
                    softcap > 0.f ? softcap : 0.f, (const float*)sink_vals,
                    splits > 1 && scratch != nullptr ? splits : 1,
                    (float*)scratch};
  hipStream_t s = (hipStream_t)stream;
  const int rc = D == 64 ? (DV == 64 ? tt_launch_rows<64, 64>(a, s)
                                     : tt_launch_rows<64, 128>(a, s))
                         : (DV == 64 ? tt_launch_rows<128, 64>(a, s)
                                     : tt_launch_rows<128, 128>(a, s));
  if (rc == 0 && a.KS > 1)
    mx_attn_records(out, ldout, scratch, T_, H, DV, a.KS, 0, MX_F32, stream);
  return rc;
}
