// Prompt portions of attention whose raw scores are mixed over the heads,
// bfloat16, on the matrix cores:
//     s_h = (q_h . k) scale,  s'_h = sum_j talk[h, j] s_j,
// softmax over the visible keys (aligned chunks, trailing window, sink in the
// denominator), weights times values. Paged cache, ragged batch, as
// talk_attention.hip; 32 heads, head widths 64 or 128.
//
// A workgroup of eight waves owns 16 consecutive rows and 16 output heads and
// walks tiles of 32 keys:
//   scores   of all 32 heads: wave w has heads 4 w .. 4 w + 3 (one KV head),
//            K Q^T as 16 x 16 tiles, keys straight from the cache as left
//            operands (no other wave reads them), queries in registers for the
//            whole walk. The other 16 output heads' workgroup repeats them:
//            an eighth of the work, and with 32 output heads the accumulators
//            alone would fill half the registers;
//   mix      through LDS as fp32 [head][row][key], since every output head
//            needs all of them: wave w mixes the 16 output heads for 4 keys,
//            the matrix and the scores as fp32 operands of
//            v_mfma_f32_16x16x4_f32 (no term of either is rounded);
//   softmax  a lane then holds one row's scores of 4 heads over 4 keys: the
//            maximum meets the other seven key shares in LDS, the
//            denominator stays a partial sum per share to the end;
//   output   the weights go back through the same LDS rows to the wave of
//            their head (wave w: two of the 16), there cut into three bf16
//            terms (exact products, fp32 accumulation), values through LDS
//            with transposed reads.
// A thread-per-(head, row) kernel on the vector pipe did this before (it
// remains for fp32 and other shapes): 13 TF/s, every product of the mix and of
// both contractions an fp32 multiply-add. Here a tile takes about 4600 cycles
// of a SIMD's matrix unit, 1024 of them the scores, 2048 the mix, 1536 the
// output, and 14200 in all: with one workgroup a CU (its LDS) the four barriers
// between those stages leave the matrix unit waiting. 32/8 heads of 128, 4099
// rows in two prompts, chunks of 2048: 0.42 ms (11.7 before; 0.63 with the blocks
// of rows from last to first).
#include "attn_common.h"
#include "scan_common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tm_bf16x8;
typedef __attribute__((ext_vector_type(4))) short tm_s4;
typedef __attribute__((address_space(3))) tm_s4 tm_lds_s4;
typedef __attribute__((ext_vector_type(4))) unsigned int tm_u4;
typedef __attribute__((ext_vector_type(2))) unsigned short tm_us2;

union TmPack {
  tm_bf16x8 v;
  tm_u4 q;
  unsigned int w[4];
  tm_s4 h[2];
};

#define TM_H 32
#define TM_KT 32
#define TM_PS 36  // LDS pitch of a row's keys: 16-byte units 9 apart

struct TmArgs {
  unsigned short* out;
  int ldout;
  const unsigned short* q;
  int ldq;
  const unsigned short *kc, *vc;  // [NB, G, BS, D], [NB, G, BS, vr]
  int vr;
  const int* block_tables;
  int max_blocks;
  const int *token_seq, *token_pos;
  const float* talk;  // [32, 32]
  int T, G, BS;
  float scale;
  int chunk, window, sink;
  float softcap;
  const float* sink_vals;
};

// A bf16 entry that is an infinity or no number.
PS_DEV bool tm_odd(unsigned int e) { return (e & 0x7f80u) == 0x7f80u; }

// First row of the workgroups' `rank`-th block of 16: those that see the most
// keys first, so that the CUs end together. Blocks are one or two a CU and see
// anything from one to all keys of a chunk; from the last row to the first, a
// second sequence's longest ones started when others were done (4099 rows of
// two sequences, chunks of 2048: 632 us, 421 by length). Every wave finds the
// same: the count of keys that `rank` blocks are above, by halves, then the block
// among those of that count. Up to 128 blocks all start at once.
PS_DEV int tm_first_row(const TmArgs& a, int rank, int blocks) {
  constexpr int PER = 16;
  if (blocks <= 128 || blocks > 64 * PER) return (blocks - 1 - rank) * 16;
  const int lane = threadIdx.x & 63;
  int keys[PER], top = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int b = k * 64 + lane;
    keys[k] = -1;
    if (k * 64 < blocks) {
      const int first = a.token_pos[min(b * 16, a.T - 1)];
      const int last = a.token_pos[min(b * 16 + 15, a.T - 1)];
      int low = 0;
      if (a.chunk > 0) low = first / a.chunk * a.chunk;
      if (a.window > 0) low = max(low, first - a.window + 1);
      // of two sequences: to the end of one and from the other's start
      const int see = last >= first ? last - low : first - low + last;
      keys[k] = b < blocks ? min(max(see, 0), 0xffffff) : -1;
      top = max(top, keys[k]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    top = max(top, __shfl_xor(top, off, 64));
  // largest v that more than `rank` blocks have at least
  int v = 0;
  for (int bit = 31 - __clz(top | 1); bit >= 0; --bit) {
    const int at = v | 1 << bit;
    int count = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k)
      if (k * 64 < blocks) count += __popcll(__ballot(keys[k] >= at));
    if (count > rank) v = at;
  }
#pragma unroll
  for (int k = 0; k < PER; ++k)
    if (k * 64 < blocks) rank -= __popcll(__ballot(keys[k] > v));
  int block = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (k * 64 < blocks) {
      const unsigned long long same = __ballot(keys[k] == v);
      const bool mine =
          keys[k] == v && __popcll(same & ((1ull << lane) - 1)) == rank;
      const unsigned long long hit = __ballot(mine);
      if (hit) block = k * 64 + __ffsll(hit) - 1;
      rank -= __popcll(same);  // below zero behind the hit: no more
    }
  }
  return block * 16;
}

// ND = D / 32, NV = DV / 16; CAP: with a score cap
template <int ND, int NV, bool CAP>
__global__ __launch_bounds__(512) void talk_mfma_kernel(TmArgs a) {
  constexpr int D = ND * 32, DV = NV * 16;
  constexpr int PV = DV + 8;          // LDS pitch of a value row
  constexpr int PR = DV / 8;          // 16-byte pieces of a value row
  constexpr int RI = 64 / PR;         // value rows per load of a wave
  constexpr int NL = TM_KT / 2 / RI;
  extern __shared__ __align__(16) float lds[];
  float* sS = lds;                                 // [32][16][TM_PS]
  float* sPM = sS + TM_H * 16 * TM_PS;             // [8][16][16]
  float* sAL = sPM + 8 * 256;                      // [16][16]
  unsigned short* sV = (unsigned short*)(sAL + 256);  // [4][32][PV]
  __shared__ int s_seq[16], s_pos[16];
  // first and last tile of a run whose values (of two waves) are not all finite
  __shared__ int s_odd[4][2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, n = lane & 15;
  // the two halves of the output heads (16 hb ..) of a block eight apart: they
  // share an XCD's L2
  const int blocks = (a.T + 15) / 16;
  const int hb = blockIdx.x >> 3 & 1;
  const int rank = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
  if (rank >= blocks) return;
  const int rep = TM_H / a.G;
  const int grp = wave * 4 / rep;                     // KV head of the scores
  const int vgrp = (16 * hb + (wave >> 1) * 4) / rep;  // and of the output
  sV += (wave >> 1) * TM_KT * PV;  // two waves' values, half a tile from each

  const int tok0 =
      __builtin_amdgcn_readfirstlane(tm_first_row(a, rank, blocks));
  const int ntok = min(16, a.T - tok0);
  if (threadIdx.x < 16) {
    const int t = tok0 + min((int)threadIdx.x, ntok - 1);
    s_seq[threadIdx.x] = a.token_seq[t];
    s_pos[threadIdx.x] = a.token_pos[t];
  }
  // queries: right operands, lane (g, n) holds entries 32 d + 8 g + i of row n
  TmPack qf[4][ND];
  {
    const unsigned short* qp =
        a.q + (size_t)(tok0 + min(n, ntok - 1)) * a.ldq + wave * 4 * D + 8 * g;
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int d = 0; d < ND; ++d)
        qf[h][d].q = *(const tm_u4*)(qp + h * D + 32 * d);
  }
  float ta[8];  // left operand of the mix: step j takes heads 4 j + g
#pragma unroll
  for (int j = 0; j < 8; ++j)
    ta[j] = a.talk[(16 * hb + n) * TM_H + 4 * j + g];
  __syncthreads();

  const int pos = s_pos[n];
  // this lane's heads of the softmax: 16 hb + 4 g + i, row n
  const int h0 = 16 * hb + 4 * g;
  float m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = a.sink ? (a.sink_vals != nullptr
                         ? fmaxf(a.sink_vals[h0 + i], PS_NEG_INF)
                         : 0.f)
                  : PS_NEG_INF;
    l[i] = a.sink && wave == 0 ? 1.f : 0.f;
  }
  ck_f32x4 acc[2][NV];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < NV; ++t) acc[h][t] = ck_f32x4{0.f, 0.f, 0.f, 0.f};

  int rs = 0;
  while (rs < ntok) {
    // batch rows rs .. re - 1 continue one sequence
    int re = rs + 1;
    while (re < ntok && s_seq[re] == s_seq[rs] &&
           s_pos[re] == s_pos[re - 1] + 1)
      ++re;
    const bool mine = n >= rs && n < re;
    const int* table = a.block_tables + (size_t)s_seq[rs] * a.max_blocks;
    auto low = [&](int p) {
      int lo = 0;
      if (a.chunk > 0) lo = p / a.chunk * a.chunk;
      if (a.window > 0) lo = max(lo, p - a.window + 1);
      return lo;
    };
    const int kmin = low(s_pos[rs]), kmax = s_pos[re - 1];
    const int nt = (kmax - kmin) / TM_KT + 1;
    const int my_lo = low(pos), my_hi = mine ? pos : -1;
    // cache row, less its KV head's, of key (lane & 31) of a tile; keys past
    // the last repeat it
    auto row_of = [&](int t) {
      const int j = min(kmin + t * TM_KT + (lane & 31), kmax);
      return table[j / a.BS] * a.G * a.BS + j % a.BS;
    };
    TmPack kf[2][ND];
    auto fetch_k = [&](int ridx) {
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) {
        const unsigned short* kp =
            a.kc + (int64_t)(__shfl(ridx, 16 * kh + n, 64) + grp * a.BS) * D +
            8 * g;
#pragma unroll
        for (int d = 0; d < ND; ++d)
          kf[kh][d].q = *(const tm_u4*)(kp + 32 * d);
      }
    };
    int ridx = row_of(0);
    fetch_k(ridx);
    int rnext = row_of(min(1, nt - 1));
    for (int t = 0; t < nt; ++t) {
      const int j0 = kmin + t * TM_KT;
      // raw scores: lane (g, n) has keys 16 kh + 4 g + i of row n
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
          ck_f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int d = 0; d < ND; ++d)
            st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                kf[kh][d].v, qf[h][d].v, st, 0, 0, 0);
          *(ck_f32x4*)(sS + ((wave * 4 + h) * 16 + n) * TM_PS + 16 * kh +
                       4 * g) = st * a.scale;
        }
      // values: on their way during the mix
      tm_u4 vr[NL];
#pragma unroll
      for (int u = 0; u < NL; ++u)
        vr[u] = *(const tm_u4*)(
            a.vc +
            (int64_t)(__shfl(ridx, (wave & 1) * 16 + u * RI + lane / PR, 64) +
                      vgrp * a.BS) *
                a.vr +
            (lane % PR) * 8);
      __syncthreads();
      if (t == 0 && threadIdx.x < 4) {  // read by all for the run before
        s_odd[threadIdx.x][0] = nt;
        s_odd[threadIdx.x][1] = -1;
      }

      // mixed scores x[e][i]: key 4 wave + e, head h0 + i, row n
      ck_f32x4 x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = ck_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const ck_f32x4 b = *(const ck_f32x4*)(
            sS + ((4 * j + g) * 16 + n) * TM_PS + 4 * wave);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta[j], b[e], x[e], 0, 0,
                                                      0);
      }
      if constexpr (CAP) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            x[e][i] = a.softcap * tanhf(x[e][i] / a.softcap);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + 4 * wave + e;
        const bool vis = j >= my_lo && j <= my_hi;
#pragma unroll
        for (int i = 0; i < 4; ++i)  // no number counts as hidden
          x[e][i] = vis ? fmaxf(x[e][i], PS_NEG_INF) : PS_NEG_INF;
      }
      float* pm = sPM + 4 * g * 16 + n;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        pm[wave * 256 + i * 16] =
            fmaxf(fmaxf(x[0][i], x[1][i]), fmaxf(x[2][i], x[3][i]));
      __syncthreads();  // also: the raw scores are read

#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float mn = m[i];
#pragma unroll
        for (int k = 0; k < 8; ++k) mn = fmaxf(mn, pm[k * 256 + i * 16]);
        // nothing visible yet: weights of 0 below, whatever is subtracted
        // (ck_exp of minus infinity; no branches around it)
        const float ms = mn > PS_NEG_INF ? mn : 0.f;
        const float al = ck_exp(m[i] - ms);
        m[i] = mn;
        if (wave == 0) sAL[(4 * g + i) * 16 + n] = al;
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e][i] = ck_exp(x[e][i] - ms);
          sum += x[e][i];
        }
        l[i] = l[i] * al + sum;
        *(ck_f32x4*)(sS + ((4 * g + i) * 16 + n) * TM_PS + 4 * wave) =
            ck_f32x4{x[0][i], x[1][i], x[2][i], x[3][i]};
      }
      // Values that are not finite stay out of the products, where a hidden
      // key's weight of zero would carry them to rows that do not see it (rows
      // of other sequences among them); they join behind the walk.
      tm_us2 top = {0, 0};
#pragma unroll
      for (int u = 0; u < NL; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          top = __builtin_elementwise_max(
              top, __builtin_bit_cast(tm_us2, vr[u][i] & 0x7fff7fffu));
      if (__any(tm_odd(top[0]) || tm_odd(top[1]))) {
#pragma unroll
        for (int u = 0; u < NL; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const unsigned int e = vr[u][i];
            vr[u][i] = (tm_odd(e) ? 0u : e & 0xffffu) |
                       (tm_odd(e >> 16) ? 0u : e & 0xffff0000u);
          }
        if (lane == 0) {
          atomicMin(&s_odd[wave >> 1][0], t);
          atomicMax(&s_odd[wave >> 1][1], t);
        }
      }
#pragma unroll
      for (int u = 0; u < NL; ++u)
        *(tm_u4*)(sV + ((wave & 1) * 16 + u * RI + lane / PR) * PV +
                  (lane % PR) * 8) = vr[u];
      ridx = rnext;
      rnext = row_of(min(t + 2, nt - 1));
      __syncthreads();

      TmPack vf[NV];  // left operands: columns 16 c .., keys 8 g + i
      const unsigned short* va =
          sV + (8 * g + (n >> 2)) * PV + 4 * (n & 3);
#pragma unroll
      for (int c = 0; c < NV; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          vf[c].h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (tm_lds_s4*)(va + 4 * h * PV + 16 * c));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int head = wave * 2 + h;  // of the 16
        const float al = sAL[head * 16 + n];
        if (__any(al != 1.f)) {
#pragma unroll
          for (int c = 0; c < NV; ++c) acc[h][c] *= al;
        }
        const float* ps = sS + (head * 16 + n) * TM_PS + 8 * g;
        const ck_f32x4 pa = *(const ck_f32x4*)ps;
        const ck_f32x4 pb = *(const ck_f32x4*)(ps + 4);
        TmPack b0, b1, b2;
        kv_split(pa[0], pa[1], &b0.w[0], &b1.w[0], &b2.w[0]);
        kv_split(pa[2], pa[3], &b0.w[1], &b1.w[1], &b2.w[1]);
        kv_split(pb[0], pb[1], &b0.w[2], &b1.w[2], &b2.w[2]);
        kv_split(pb[2], pb[3], &b0.w[3], &b1.w[3], &b2.w[3]);
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          acc[h][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf[c].v, b0.v, acc[h][c], 0, 0, 0);
          acc[h][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf[c].v, b1.v, acc[h][c], 0, 0, 0);
          acc[h][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf[c].v, b2.v, acc[h][c], 0, 0, 0);
        }
      }
      // not before: beside the value operands they would spill
      fetch_k(ridx);
      __syncthreads();  // the weights are read
    }
    // values that are not finite, to the rows that see their keys: whatever
    // the weight, which is above zero, they decide the sum
    const int odd0 = s_odd[wave >> 1][0], odd1 = s_odd[wave >> 1][1];
#pragma unroll 1
    for (int j = kmin + odd0 * TM_KT;
         j < min(kmin + (odd1 + 1) * TM_KT, kmax + 1); ++j) {
      if (j < my_lo || j > my_hi) continue;
      const unsigned short* p =
          a.vc + ((int64_t)(table[j / a.BS] * a.G + vgrp) * a.BS + j % a.BS) *
                     a.vr + 4 * g;
#pragma unroll
      for (int c = 0; c < NV; ++c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned int e = p[16 * c + i];
          const float x = tm_odd(e) ? __uint_as_float(e << 16) : 0.f;
          acc[0][c][i] += x;
          acc[1][c][i] += x;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    rs = re;
  }

  // denominators: eight key shares per (head, row)
#pragma unroll
  for (int i = 0; i < 4; ++i) sPM[wave * 256 + (4 * g + i) * 16 + n] = l[i];
  __syncthreads();
  if (n >= ntok) return;
  unsigned short* o = a.out + (size_t)(tok0 + n) * a.ldout +
                      (16 * hb + wave * 2) * DV + 4 * g;
  const bool vec = (a.ldout & 3) == 0 && ((size_t)a.out & 7) == 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float lt = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) lt += sPM[k * 256 + (wave * 2 + h) * 16 + n];
    const float f = 1.0f / lt;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      unsigned short e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = ps_f32_to_bf16(acc[h][c][i] * f);
      unsigned short* p = o + h * DV + 16 * c;
      if (vec) {
        *(uint2*)p = make_uint2((unsigned int)e[0] | ((unsigned int)e[1] << 16),
                                (unsigned int)e[2] | ((unsigned int)e[3] << 16));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = e[i];
      }
    }
  }
}

template <int ND, int NV, bool CAP>
static int tm_launch_as(const TmArgs& a, hipStream_t stream) {
  const size_t lds = (size_t)(TM_H * 16 * TM_PS + 9 * 256) * 4 +
                     (size_t)4 * TM_KT * (NV * 16 + 8) * 2;
  if (hipFuncSetAttribute((const void*)talk_mfma_kernel<ND, NV, CAP>,
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  // 16 workgroups for eight blocks of rows
  hipLaunchKernelGGL((talk_mfma_kernel<ND, NV, CAP>),
                     dim3((a.T + 127) / 128 * 16), dim3(512), lds, stream, a);
  return 0;
}

template <int ND, int NV>
static int tm_launch(const TmArgs& a, hipStream_t stream) {
  return a.softcap > 0.f ? tm_launch_as<ND, NV, true>(a, stream)
                         : tm_launch_as<ND, NV, false>(a, stream);
}

// Returns 0 when launched, 1 when the shape is outside this kernel: 32 heads
// over at most 8 KV heads (a wave's four heads share one), widths 64 or 128,
// rows on 16-byte borders.
extern "C" int mx_talk_mfma(
    void* out, int ldout, const void* q, int ldq, const void* kc,
    const void* vc, const void* block_tables, int max_blocks,
    const void* token_seq, const void* token_pos, const void* talk, int T_,
    int H, int G, int D, int DV, int BS, float scale, int chunk, int window,
    int sink, float softcap, const void* sink_vals, int vrow, void* stream) {
  if (T_ <= 0) return 0;
  if (H != TM_H || G < 1 || H % G || H / G % 4) return 1;
  if ((D != 64 && D != 128) || (DV != 64 && DV != 128)) return 1;
  if (ldq % 8 || vrow % 8 || ((size_t)q | (size_t)kc | (size_t)vc) % 16)
    return 1;
  TmArgs a = {(unsigned short*)out, ldout, (const unsigned short*)q, ldq,
              (const unsigned short*)kc, (const unsigned short*)vc, vrow,
              (const int*)block_tables, max_blocks, (const int*)token_seq,
              (const int*)token_pos, (const float*)talk, T_, G, BS, scale,
              chunk, window, sink, softcap, (const float*)sink_vals};
  hipStream_t s = (hipStream_t)stream;
  if (D == 64)
    return DV == 64 ? tm_launch<2, 4>(a, s) : tm_launch<2, 8>(a, s);
  return DV == 64 ? tm_launch<4, 4>(a, s) : tm_launch<4, 8>(a, s);
}
