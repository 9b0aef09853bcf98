// Prompt portions of attention whose raw scores are mixed over the heads,
// bfloat16, on the matrix cores:
//     s_h = (q_h . k) scale,  s'_h = sum_j talk[h, j] s_j,
// softmax over the visible keys (aligned chunks, trailing window, sink in the
// denominator), weights times values. Paged cache, ragged batch, as
// talk_attention.hip; 32 heads, head widths 64 or 128.
//
// A workgroup of eight waves owns 16 consecutive rows and 16 output heads and
// walks tiles of 32 keys by halves of 16, one barrier each. Between two barriers
//   scores   of the next half, all 32 heads: wave w has heads 4 w .. 4 w + 3 (one
//            KV head), K Q^T as 16 x 16 tiles, keys straight from the cache as
//            left operands (no other wave reads them), queries in registers for
//            the whole walk. The other 16 output heads' workgroup repeats them:
//            an eighth of the work, and with 32 output heads the accumulators
//            alone would fill half the registers;
//   mix      of this half through LDS as fp32 [head][row][key], since every
//            output head needs all of them: wave w mixes the 16 output heads for
//            2 keys, the matrix and the scores as fp32 operands of
//            v_mfma_f32_16x16x4_f32 (no term of either is rounded);
//   softmax  a lane then holds one row's scores of 4 heads over 2 keys, whose
//            weights are relative to a reference that all waves share, not to the
//            half's own maximum: it lies TM_FAR above the score that set it and
//            moves, by an exchange behind the barrier, only where a score is above
//            it. The denominator stays a partial sum per key share to the end;
//   output   of the tile before, in every other half: the weights go through LDS
//            to the wave of their head (wave w: two of the 16), there cut into
//            three bf16 terms (exact products, fp32 accumulation), values through
//            LDS with transposed reads.
// Scores have two halves in LDS, weights three, so that none of this waits for
// another wave. A tile takes about 4600 cycles of a SIMD's matrix unit, 1024 of
// them the scores, 2048 the mix, 1536 the output, 4000 of vector instructions, and
// 12000 in all (14200 with four barriers a tile of 32 and the maximum through LDS
// in each): both waves of a SIMD come to the products and to the softmax at about
// the same time. 32/8 heads of 128, 4099 rows in two prompts, chunks of 2048: 0.32
// ms (0.42 with four barriers, 0.63 with the blocks of rows from last to first, 11.7
// on the vector pipe, whose kernel remains for fp32 and other shapes). Sixteen waves
// spill at widths of 128 and are no faster at 64 (284 us, 272 with eight); orders of
// the four parts that differ between the two waves of a SIMD spill as well.
// Few rows behind many keys are a chain of tiles (3.5 us each) on a few CUs: there
// several workgroups share a block's keys, as many as have two tiles, and
// mx_attn_records merges what they have (70 rows behind 2000 keys 276 us whole, 50 in
// 16 shares; a portion with too few keys for shares 3 us more for that launch).
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
#define TM_SHARE 2  // tiles of a share at least
// How far scores, in powers of two, may be above those that set the reference that
// weights are relative to. The reference is as much above them: no weight is above 1.
#define TM_FAR 8.f

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
  int KS;       // workgroups that share a block's keys
  float* part;  // [T, KS, 32, DV + 4]: maximum (a power of two), denominator,
                // shares, -, sums
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

// Where a (row, unit) of LDS rows of 16 keys is: units of two keys, turned by the
// row and one bit of the head so that the 32 lanes of a pass meet all banks.
PS_DEV int tm_at(int head, int row, int unit, int bit) {
  return (head * 16 + row) * 16 + 2 * (unit ^ (row >> 2 | (bit & 1) << 2));
}

// ND = D / 32, NV = DV / 16; CAP: with a score cap; PART: several workgroups to a
// block's keys (as a choice at run time whole blocks took 1 to 2 % longer)
template <int ND, int NV, bool CAP, bool PART>
__global__ __launch_bounds__(512) void talk_mfma_kernel(TmArgs a) {
  constexpr int D = ND * 32, DV = NV * 16;
  constexpr int PV = DV + 8;          // LDS pitch of a value row
  constexpr int PR = DV / 8;          // 16-byte pieces of a value row
  constexpr int RI = 64 / PR;         // value rows per load of a wave
  constexpr int NL = TM_KT / 2 / RI;
  constexpr int SS = TM_H * 256, SP = 16 * 256;
  extern __shared__ __align__(16) float lds[];
  float* sS = lds;                                 // [2][32][16][16 keys]
  float* sP = sS + 2 * SS;                         // [3][16][16][16 keys]
  float* sPM = sP + 3 * SP;                        // [8][16][16]
  float* sAL = sPM + 8 * 256;                      // [16][16]
  unsigned short* sV = (unsigned short*)(sAL + 256);  // [4][32][PV]
  __shared__ int s_seq[16], s_pos[16];
  // first and last tile of a run whose values (of two waves) are not all finite
  __shared__ int s_odd[4][2];
  __shared__ int s_high[3];  // a half has scores above the reference
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
  // left operand of the mix: step j takes heads 4 j + g. Scores in powers of two
  // (with a cap behind it).
  float ta[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    ta[j] = a.talk[(16 * hb + n) * TM_H + 4 * j + g] *
            (CAP ? a.scale : a.scale * KV_LOG2E);
  __syncthreads();

  const int pos = s_pos[n];
  // this lane's heads of the softmax: 16 hb + 4 g + i, row n
  const int h0 = 16 * hb + 4 * g;
  float m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // the product may be past the largest float
    m[i] = a.sink && (!PART || blockIdx.y == 0)  // the sink is share 0's
               ? (a.sink_vals != nullptr
                         ? fminf(fmaxf(a.sink_vals[h0 + i] * KV_LOG2E,
                                       PS_NEG_INF),
                                 -KV_LOW)
                         : 0.f) + TM_FAR
                  : PS_NEG_INF;
    l[i] = a.sink && (!PART || blockIdx.y == 0) && wave == 0 ? __builtin_amdgcn_exp2f(-TM_FAR) : 0.f;
  }
  ck_f32x4 acc[2][NV];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < NV; ++t) acc[h][t] = ck_f32x4{0.f, 0.f, 0.f, 0.f};

  // one of the two waves of a SIMD first, so that its softmax comes beside
  // products of the other (324 -> 320 us)
  if (ND == 4 && wave < 4) __builtin_amdgcn_s_setprio(1);
  int rs = 0, my_eff = 1;  // shares of this lane's row
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
    int kmin = low(s_pos[rs]), kmax = s_pos[re - 1];
    if constexpr (PART) {  // this share's tiles
      // the workgroups that have a share of these tiles
      const int all = (kmax - kmin) / TM_KT + 1, ks = blockIdx.y;
      const int eff = max(1, min(a.KS, all / TM_SHARE));
      if (mine) my_eff = eff;
      if (ks >= eff) {
        rs = re;
        continue;
      }
      const int t0 = all * ks / eff, t1 = all * (ks + 1) / eff;
      kmax = min(kmax, kmin + t1 * TM_KT - 1);
      kmin += t0 * TM_KT;
    }
    const int nt = (kmax - kmin) / TM_KT + 1;
    const int my_lo = low(pos), my_hi = mine ? pos : -1;
    // cache row, less its KV head's, of key (lane & 31) of a tile; keys past
    // the last repeat it
    auto row_of = [&](int t) {
      const int j = min(kmin + t * TM_KT + (lane & 31), kmax);
      return table[j / a.BS] * a.G * a.BS + j % a.BS;
    };
    TmPack kf[ND];  // keys of a half: left operands
    auto fetch_k = [&](int ridx, int half) {
      const unsigned short* kp =
          a.kc +
          (int64_t)(__shfl(ridx, 16 * half + n, 64) + grp * a.BS) * D + 8 * g;
#pragma unroll
      for (int d = 0; d < ND; ++d) kf[d].q = *(const tm_u4*)(kp + 32 * d);
    };
    tm_u4 vr[NL];
    auto fetch_v = [&](int ridx) {
#pragma unroll
      for (int u = 0; u < NL; ++u)
        vr[u] = *(const tm_u4*)(
            a.vc +
            (int64_t)(__shfl(ridx, (wave & 1) * 16 + u * RI + lane / PR, 64) +
                      vgrp * a.BS) *
                a.vr +
            (lane % PR) * 8);
    };
    // raw scores of a half: lane (g, n) has keys 4 g + i of row n
    auto scores = [&](int half) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        ck_f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < ND; ++d)
          st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[d].v, qf[h][d].v, st,
                                                       0, 0, 0);
        float* to = sS + half * SS;
        *(float2*)(to + tm_at(wave * 4 + h, n, 2 * g, h)) =
            make_float2(st[0], st[1]);
        *(float2*)(to + tm_at(wave * 4 + h, n, 2 * g + 1, h)) =
            make_float2(st[2], st[3]);
      }
    };
    // mixed scores x[e][i]: key 2 wave + e of a half, head h0 + i, row n
    auto mix = [&](int t, int half, ck_f32x4(&x)[2]) {
      x[0] = x[1] = ck_f32x4{0.f, 0.f, 0.f, 0.f};
      float2 b[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        b[j] = *(const float2*)(sS + half * SS + tm_at(4 * j + g, n, wave, g));
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta[j], b[j].x, x[0], 0, 0,
                                                    0);
        x[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta[j], b[j].y, x[1], 0, 0,
                                                    0);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int j = kmin + t * TM_KT + 16 * half + 2 * wave + e;
        const bool vis = j >= my_lo && j <= my_hi;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (CAP)
            x[e][i] = a.softcap * KV_LOG2E * tanhf(x[e][i] / a.softcap);
          // no number counts as hidden
          x[e][i] = vis ? fmaxf(x[e][i], PS_NEG_INF) : PS_NEG_INF;
        }
      }
    };
    // weights of a half, its third of sP, their sums
    auto weigh = [&](ck_f32x4(&x)[2], float* to, float(&sum)[4]) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // nothing visible yet: weights of 0, whatever is subtracted
        const float ms = m[i] > PS_NEG_INF ? m[i] : 0.f;
        const float p0 = __builtin_amdgcn_exp2f(x[0][i] - ms);
        const float p1 = __builtin_amdgcn_exp2f(x[1][i] - ms);
        sum[i] = p0 + p1;
        *(float2*)(to + tm_at(4 * g + i, n, wave, g)) = make_float2(p0, p1);
      }
    };
    // A half with scores above the reference, behind the barrier that ends its
    // turn: the reference moves to TM_FAR above the largest, and with it
    // what was made by the one before: the half's weights, those of the other
    // half of an unfinished tile, sums and outputs.
    auto raise = [&](int t, int half, int third, float(&sum)[4]) {
      ck_f32x4 x[2];
      mix(t, half, x);
      float* pm = sPM + 4 * g * 16 + n;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        pm[wave * 256 + i * 16] = fmaxf(x[0][i], x[1][i]);
      __syncthreads();
      float* other = sP + (third + 2) % 3 * SP;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float mn = m[i];
#pragma unroll
        for (int k = 0; k < 8; ++k) mn = fmaxf(mn, pm[k * 256 + i * 16] + TM_FAR);
        const float al =
            __builtin_amdgcn_exp2f(m[i] - (mn > PS_NEG_INF ? mn : 0.f));
        m[i] = mn;
        l[i] *= al;
        if (wave == 0) sAL[(4 * g + i) * 16 + n] = al;
        if (half == 1) {
          float2* p = (float2*)(other + tm_at(4 * g + i, n, wave, g));
          *p = make_float2(p->x * al, p->y * al);
        }
      }
      weigh(x, sP + third * SP, sum);
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float al = sAL[(wave * 2 + h) * 16 + n];
#pragma unroll
        for (int c = 0; c < NV; ++c) acc[h][c] *= al;
      }
    };
    // Values that are not finite stay out of the products, where a hidden
    // key's weight of zero would carry them to rows that do not see it (rows
    // of other sequences among them); they join behind the walk.
    auto put_v = [&](int t) {
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
    };
    // a tile's output: its weights are in thirds `first` and the next
    auto output = [&](int first) {
      TmPack vf[NV];  // left operands: columns 16 c .., keys 8 g + i
      const unsigned short* va =
          sV + (8 * g + (n >> 2)) * PV + 4 * (n & 3);
#pragma unroll
      for (int c = 0; c < NV; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          vf[c].h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (tm_lds_s4*)(va + 4 * h * PV + 16 * c));
      const float* from = sP + (first + (g >> 1)) % 3 * SP;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int head = wave * 2 + h;  // of the 16
        TmPack b0, b1, b2;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float2 p = *(const float2*)(
              from + tm_at(head, n, 4 * (g & 1) + q, head >> 2));
          kv_split(p.x, p.y, &b0.w[q], &b1.w[q], &b2.w[q]);
        }
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
    };

    int rcur = row_of(0), rnext = row_of(min(1, nt - 1));
    fetch_k(rcur, 0);
    if (threadIdx.x < 4) {
      s_odd[threadIdx.x][0] = nt;
      s_odd[threadIdx.x][1] = -1;
    }
    if (threadIdx.x < 3) s_high[threadIdx.x] = 0;
    scores(0);
    fetch_k(rcur, 1);
    __syncthreads();
    float sum[4];
    int third = 0;  // of sP for the coming half
    // One half: its weights, the scores of the next one, beside either the output
    // of the tile before or the writing of this one's values.
    auto turn = [&](int t, int half) {
      // read before the last barrier; set again behind the next
      if (threadIdx.x == 0) s_high[(third + 1) % 3] = 0;
      auto weights = [&] {
        ck_f32x4 x[2];
        mix(t, half, x);
        bool high = false;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          high |= fmaxf(x[0][i], x[1][i]) > m[i];
        if (__any(high) && lane == 0) s_high[third] = 1;
        weigh(x, sP + third * SP, sum);
      };
      auto others = [&] {
        scores(half ^ 1);
        if (half == 0) {
          if (t > 0) output((third + 1) % 3);
          // not before: beside the value operands they would spill
          __builtin_amdgcn_sched_barrier(0);
          fetch_k(rnext, 0);
          fetch_v(rcur);
        } else {
          put_v(t);
          rcur = rnext;
          rnext = row_of(min(t + 2, nt - 1));
          fetch_k(rcur, 1);
        }
      };
      // us, weights first / last: heads of 128 329 / 324, of 64 262 / 277
      if constexpr (ND == 4) {
        others();
        weights();
      } else {
        weights();
        others();
      }
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(s_high[third]))
        raise(t, half, third, sum);
#pragma unroll
      for (int i = 0; i < 4; ++i) l[i] += sum[i];
      third = third == 2 ? 0 : third + 1;
    };
    for (int t = 0; t < nt; ++t) {
      turn(t, 0);
      turn(t, 1);
    }
    output((third + 1) % 3);
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
    __syncthreads();  // the run's LDS is read
    rs = re;
  }

  // denominators: eight key shares per (head, row)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sPM[wave * 256 + (4 * g + i) * 16 + n] = l[i];
    if (PART && wave == 0) sAL[(4 * g + i) * 16 + n] = m[i];
  }
  __syncthreads();
  if (n >= ntok || (PART && (int)blockIdx.y >= my_eff)) return;
  unsigned short* o = a.out + (size_t)(tok0 + n) * a.ldout +
                      (16 * hb + wave * 2) * DV + 4 * g;
  const bool vec = (a.ldout & 3) == 0 && ((size_t)a.out & 7) == 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float lt = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) lt += sPM[k * 256 + (wave * 2 + h) * 16 + n];
    if constexpr (PART) {
      float* rec = a.part + (((size_t)(tok0 + n) * a.KS + blockIdx.y) * TM_H +
                             16 * hb + wave * 2 + h) * (DV + 4);
      if (g == 0) {
        const float mt = sAL[(wave * 2 + h) * 16 + n];
        rec[0] = lt != 0.f ? mt : PS_NEG_INF;
        rec[1] = lt;
        rec[2] = (float)my_eff;
      }
      if (my_eff > 1) {
        if (lt != 0.f)  // else no key of this share: no sums
#pragma unroll
          for (int c = 0; c < NV; ++c)
            *(float4*)(rec + 4 + 16 * c + 4 * g) = make_float4(
                acc[h][c][0], acc[h][c][1], acc[h][c][2], acc[h][c][3]);
        continue;
      }
    }
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

template <int ND, int NV, bool CAP, bool PART>
static int tm_launch_as(const TmArgs& a, hipStream_t stream) {
  const size_t lds = (size_t)(2 * TM_H * 256 + 3 * 16 * 256 + 9 * 256) * 4 +
                     (size_t)4 * TM_KT * (NV * 16 + 8) * 2;
  if (hipFuncSetAttribute((const void*)talk_mfma_kernel<ND, NV, CAP, PART>,
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  // 16 workgroups for eight blocks of rows
  hipLaunchKernelGGL((talk_mfma_kernel<ND, NV, CAP, PART>),
                     dim3((a.T + 127) / 128 * 16, a.KS), dim3(512), lds, stream, a);
  return 0;
}

template <int ND, int NV>
static int tm_launch(const TmArgs& a, hipStream_t stream) {
  if (a.KS > 1)
    return a.softcap > 0.f ? tm_launch_as<ND, NV, true, true>(a, stream)
                           : tm_launch_as<ND, NV, false, true>(a, stream);
  return a.softcap > 0.f ? tm_launch_as<ND, NV, true, false>(a, stream)
                         : tm_launch_as<ND, NV, false, false>(a, stream);
}

extern "C" void mx_attn_records(void* out, int ldout, const void* part, int T_,
                                int H, int DV, int KS, int counted,
                                int dtype, void* stream);

// Returns 0 when launched, 1 when the shape is outside this kernel: 32 heads
// over at most 8 KV heads (a wave's four heads share one), widths 64 or 128,
// rows on 16-byte borders. scratch fp32 [T, splits, 32, DV + 4] when splits > 1.
extern "C" int mx_talk_mfma(
    void* out, int ldout, const void* q, int ldq, const void* kc,
    const void* vc, const void* block_tables, int max_blocks,
    const void* token_seq, const void* token_pos, const void* talk, int T_,
    int H, int G, int D, int DV, int BS, float scale, int chunk, int window,
    int sink, float softcap, const void* sink_vals, int vrow, int splits,
    void* scratch, void* stream) {
  if (T_ <= 0) return 0;
  if (splits > 16) return 1;
  if (H != TM_H || G < 1 || H % G || H / G % 4) return 1;
  if ((D != 64 && D != 128) || (DV != 64 && DV != 128)) return 1;
  if (ldq % 8 || vrow % 8 || ((size_t)q | (size_t)kc | (size_t)vc) % 16)
    return 1;
  TmArgs a = {(unsigned short*)out, ldout, (const unsigned short*)q, ldq,
              (const unsigned short*)kc, (const unsigned short*)vc, vrow,
              (const int*)block_tables, max_blocks, (const int*)token_seq,
              (const int*)token_pos, (const float*)talk, T_, G, BS, scale,
              chunk, window, sink, softcap, (const float*)sink_vals,
              splits > 1 && scratch != nullptr ? splits : 1, (float*)scratch};
  hipStream_t s = (hipStream_t)stream;
  const int rc = D == 64 ? (DV == 64 ? tm_launch<2, 4>(a, s) : tm_launch<2, 8>(a, s))
                         : (DV == 64 ? tm_launch<4, 4>(a, s) : tm_launch<4, 8>(a, s));
  if (rc == 0 && a.KS > 1)
    mx_attn_records(out, ldout, scratch, T_, H, DV, a.KS, 1, MX_BF16, stream);
  return rc;
}
