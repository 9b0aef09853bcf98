// Grouped-query attention with keys and values of their own over the paged
// cache, bf16, gfx950 matrix cores: trailing window with kept first keys (or
// everything), capped scores, sink in the denominator. Head widths up to 128.
//
// Both kernels are built as those of keyval_attention.hip, whose rows serve as
// keys and values at once:
//   prompt   4 waves, 128 (token, head) rows of one KV head, 32 a wave, queries
//            in registers; 64 keys and their values at a time in one of two LDS
//            buffers, the next ones on their way during the products, one
//            barrier a tile. S^T = K Q^T, O^T = V^T P^T on
//            v_mfma_f32_32x32x16_bf16, values through transposed LDS reads.
//   token    one (token, KV head, share of the keys) a workgroup, 32 keys at a
//            time per wave in private LDS, no barrier before the merge.
// The lanes of a score tile hold runs of 8 consecutive keys of one row, so the
// softmax is lane-local plus one (two) exchanges and the weights pack straight
// into the second product as three bf16 terms (exact, fp32 accumulation).
//
// What bounds the prompt form: per 32 x 64 scores of a wave 2048 cycles of
// matrix products (1536 of them the three terms of P V) stand beside about as
// many of vector instructions (cap, softmax, cut); two workgroups a CU let them
// overlap. The form before (mfma_attention.hip; it remains for pooled blocks,
// wider values and odd widths) staged 32 keys between two barriers with nothing
// in flight and read values as single 16-bit words. 32/8 heads of 128, two
// prompts of 2048: 159 us, 159 with a window of 1024 and a cap (598 and 408
// before; 182 with the cap's subtraction of the reference on its own); 256
// rows behind 2048 keys 91 (302). A reference that stays while no score passes it
// by 16 times: 8069 rows of two prompts, window 2048 and a cap, 530 -> 503 us, 32/8
// heads of 64 86 -> 72. (Matrix pipe busy 48 % of it, each wave issuing 45 %.)
// Raised wave priority during the products made it 5 % slower, the bf16
// dot product in the weights' cut 2 %; bank conflicts in half the value reads, gone
// with the row pitch, and the first 32 keys' scores beside the second 32 keys'
// products cost and gave nothing.
// The token form is bound by the keys and values it reads, at few tokens by the
// latency of its tiles: 64 tokens x 4001 keys 177 us, 5.9 TB/s (424 before);
// window 1024 42 us (119); 8 tokens of it 16 us (32).
#include "attn_common.h"

struct WaArgs {
  unsigned short* out;
  int ldout;
  const unsigned short* q;
  int ldq;
  const unsigned short *kc, *vc;  // [NB, G, BS, D], [NB, G, BS, vr]
  int vr;
  const int* block_tables;
  int max_blocks;
  const int* token_seq;
  const int* token_pos;
  int T, H, G, D, DV, BS;
  float scale2;    // score scale times log2(e)
  float cap2;      // cap times log2(e), 0: none
  float icap2;     // 2 scale log2(e) / cap
  int window, keep, sink;
  const float* sink_vals;  // per head (nullptr: score 0)
  int KS;
  float* part;
  int hpb, hblocks;  // heads per workgroup, head blocks per KV head
  int tpt;           // tokens per workgroup (prompt form)
  int order;         // tokens by their keys (token form)
};

// A raw product as a score in powers of two, less `base`. With a cap: cap
// tanh(s / cap) = cap (1 - 2 / (exp(2 s / cap) + 1)); top = cap - base.
template <bool CAP>
PS_DEV float wa_score(const WaArgs& a, float st, float base, float top) {
  if constexpr (!CAP) return st * a.scale2 - base;
  const float e = __builtin_amdgcn_exp2f(st * a.icap2);
  return top - 2.f * a.cap2 * __builtin_amdgcn_rcpf(e + 1.f);
}

#define WA_KT 64

#define WA_HEAD 4   // leading entries of a partial record
#define WA_SHARE 3  // tiles of a portion's share at least

// DK: 16-entry steps of a key (D <= 16 DK), VB: 32-column blocks of a value, PART:
// several workgroups (up to KS, neighbours) share a tile's keys
template <int DK, int VB, bool CAP, bool PART>
__global__ __launch_bounds__(256, 2) void window_prompt_kernel(WaArgs a) {
  // values: the four rows of a transposed read lie 16 banks apart
  constexpr int PK = DK * 16 + 8, PV = VB * 32 + 32;
  __shared__ __align__(16) unsigned short sK[2][WA_KT * PK];
  __shared__ __align__(16) unsigned short sV[2][WA_KT * PV];
  __shared__ int s_row[2][WA_KT];
  __shared__ int s_seq[128], s_pos[128];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row = lane & 31, hi = lane >> 5;
  const int D = a.D, DV = a.DV, rep = a.H / a.G, HPB = a.hpb;
  const int TPT = a.tpt;
  const int NT = (a.T + TPT - 1) / TPT;
  // rows that see the most keys first
  const int GH = a.G * a.hblocks;
  const int gh = blockIdx.x % GH;
  const int ks = PART ? blockIdx.x / GH % a.KS : 0;
  const int tile = NT - 1 - blockIdx.x / GH / (PART ? a.KS : 1);
  const int g = gh / a.hblocks, hb = gh % a.hblocks;
  const int tok0 = tile * TPT, ntok = min(TPT, a.T - tok0);
  for (int c = tid; c < ntok; c += 256) {
    s_seq[c] = a.token_seq[tok0 + c];
    s_pos[c] = a.token_pos[tok0 + c];
  }
  __syncthreads();

  // this lane's (token, head)
  const int my = wave * 32 + row;
  const int my_i = my / HPB, my_h = hb * HPB + my % HPB;
  const bool valid = my_i < ntok && my_h < rep;
  const int head = g * rep + min(my_h, rep - 1);
  const int tok = tok0 + min(my_i, ntok - 1);
  const int my_pos = s_pos[min(my_i, ntok - 1)];
  // queries: B operand, lane (row, hi) holds entries 16 s + 8 hi + i
  kv_bf16x8 qr[DK];
  {
    const unsigned short* qp = a.q + (size_t)tok * a.ldq + (size_t)head * D;
#pragma unroll
    for (int s = 0; s < DK; ++s) {
      const int c = 16 * s + 8 * hi;
      KvPack u;
      u.q = c < D ? *(const uint4*)(qp + c) : make_uint4(0, 0, 0, 0);
      qr[s] = u.v;
    }
  }
  float m = KV_LOW, l = 0.f;
  kv_f32x16 acc[VB];
#pragma unroll
  for (int c = 0; c < VB; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[c][r] = 0.f;

  constexpr int CK = DK * 2, CV = VB * 4;  // 16-byte pieces per row
  constexpr int NK = WA_KT * CK / 256, NV = WA_KT * CV / 256;
  kv_u4 pk[NK], pv[NV];
  // LDS row of this lane's key in a 32-key score tile
  const int krow = (row & 0x13) | ((row & 4) << 1) | ((row & 8) >> 1);
  const int i16 = lane & 15;
  // this lane's part of a transposed read
  const int vat = (8 * hi + (i16 >> 2)) * PV + 16 * ((lane >> 4) & 1) +
                  4 * (i16 & 3);
  const unsigned vis = a.window > 0 ? a.window : 0x7fffffff;

  // rows that do not continue the sequence of the row before them
  auto starts = [&](int i) {
    return i < ntok && (i == 0 || s_seq[i] != s_seq[i - 1] ||
                        s_pos[i] != s_pos[i - 1] + 1);
  };
  const unsigned long long start0 = __ballot(starts(lane)),
                           start1 = __ballot(starts(64 + lane));
  auto next_start = [&](int i) {  // behind row i
    unsigned long long m = i < 63 ? start0 & (~1ull << i) : 0;
    if (m) return __ffsll(m) - 1;
    m = i < 64 ? start1 : i < 127 ? start1 & (~1ull << (i - 64)) : 0;
    return m ? __ffsll(m) + 63 : ntok;
  };
  int rs = 0, my_eff = 1, my_ks = ks, from = 0;
  while (rs < ntok) {
    // batch rows rs .. re - 1 continue one sequence
    const int re = next_start(rs);
    const bool mine = valid && my_i >= rs && my_i < re;
    const bool all_mine = __all(mine);
    const int* table = a.block_tables + (size_t)s_seq[rs] * a.max_blocks;
    const int kmin = a.window > 0 ? max(0, s_pos[rs] - a.window + 1) : 0;
    const int kmax = s_pos[re - 1];
    // kept first keys behind the run's earliest window, then the windows
    const int k0 = min(a.keep, kmin);
    const int nt0 = (k0 + WA_KT - 1) / WA_KT;
    const int all = nt0 + (kmax - kmin) / WA_KT + 1;
    // the workgroups that have a share of these tiles (from behind those of the run
    // before on, so that short runs are not all the first one's), and this one's
    const int eff = PART ? max(1, min(a.KS, all / WA_SHARE)) : 1;
    const int share = PART ? (ks >= from ? ks - from : ks - from + a.KS) : 0;
    if (PART) {
      from += eff;
      if (from >= a.KS) from -= a.KS;
      if (mine) {
        my_eff = eff;
        my_ks = share;
      }
      if (share >= eff) {
        rs = re;
        continue;
      }
    }
    const int n0 = PART ? all * share / eff : 0;
    const int nt = PART ? all * (share + 1) / eff : all;
    // rows of other runs see nothing of this one
    const int pos = mine ? my_pos : -1;
    const int ia = max(wave * 32 / HPB, rs);
    const int ib = min((wave * 32 + 31) / HPB, re - 1);
    const bool live = ia <= ib;
    const int w_first = live ? s_pos[ia] : 0, w_last = live ? s_pos[ib] : 0;
    const int w_lo = a.window > 0 ? max(0, w_first - a.window + 1) : 0;
    const int w_full_lo = a.window > 0 ? max(0, w_last - a.window + 1) : 0;

    // key of row (tid & 63) of a tile; rows past the range's last key repeat
    // it (they are masked). The page number is loaded well ahead of its use.
    auto key_of = [&](int n) {
      return n < nt0 ? min(n * WA_KT + (tid & 63), k0 - 1)
                     : min(kmin + (n - nt0) * WA_KT + (tid & 63), kmax);
    };
    auto put_row = [&](int n, int page, int buf) {
      if (tid < WA_KT)
        s_row[buf][tid] = (page * a.G + g) * a.BS + key_of(n) % a.BS;
    };
    auto fetch = [&](int buf) {
      // columns past a row's end repeat its last piece: finite numbers that
      // meet zero query entries or land in columns never stored
#pragma unroll
      for (int u = 0; u < NK; ++u) {
        const int idx = u * 256 + tid;
        pk[u] = *(const kv_u4*)(a.kc + (int64_t)s_row[buf][idx / CK] * D +
                                min(idx % CK * 8, D - 8));
      }
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int idx = u * 256 + tid;
        pv[u] = *(const kv_u4*)(a.vc + (int64_t)s_row[buf][idx / CV] * a.vr +
                                min(idx % CV * 8, DV - 8));
      }
    };
    put_row(n0, table[key_of(n0) / a.BS], 1 - (n0 & 1));
    __syncthreads();  // also: the previous run's tiles are fully read
    fetch(1 - (n0 & 1));
    int page = table[key_of(min(n0 + 1, nt - 1)) / a.BS];
    for (int n = n0; n < nt; ++n) {
      // tile n from registers to its buffer, which tile n - 2 has left; what
      // lies past the last tile repeats it
#pragma unroll
      for (int u = 0; u < NK; ++u) {
        const int idx = u * 256 + tid;
        *(kv_u4*)(&sK[n & 1][idx / CK * PK + idx % CK * 8]) = pk[u];
      }
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int idx = u * 256 + tid;
        *(kv_u4*)(&sV[n & 1][idx / CV * PV + idx % CV * 8]) = pv[u];
      }
      put_row(min(n + 1, nt - 1), page, n & 1);
      __syncthreads();
      fetch(n & 1);
      page = table[key_of(min(n + 2, nt - 1)) / a.BS];
      const unsigned short* sk = sK[n & 1];
      const unsigned short* sv = sV[n & 1];
      const bool kept = n < nt0;
      const int j0 = kept ? n * WA_KT : kmin + (n - nt0) * WA_KT;
      if (!live) continue;
      if (!kept &&
          (j0 > w_last || (j0 + WA_KT - 1 < w_lo && j0 >= a.keep)))
        continue;

      kv_f32x16 st[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) st[0][r] = st[1][r] = 0.f;
#pragma unroll
      for (int s = 0; s < DK; ++s) {
        const unsigned short* ka = sk + krow * PK + 16 * s + 8 * hi;
        const kv_bf16x8 a0 = *(const kv_bf16x8*)ka;
        const kv_bf16x8 a1 = *(const kv_bf16x8*)(ka + 32 * PK);
        st[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, qr[s], st[0], 0,
                                                        0, 0);
        st[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, qr[s], st[1], 0,
                                                        0, 0);
      }
      // st[h][8 s + i] belongs to key j0 + 32 h + 16 s + 8 hi + i
      const float base = m == KV_LOW ? 0.f : m;
      float w[32];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          w[16 * h + r] = wa_score<CAP>(a, st[h][r], base, a.cap2 - base);
      const int dist = pos - j0 - 8 * hi;  // of this lane's first key
      if (kept) {
        const int left = mine ? k0 - j0 - 8 * hi : 0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * h + 16 * (r >> 3) + (r & 7) >= left)
              w[16 * h + r] = -INFINITY;
      } else if (!all_mine || j0 < w_full_lo || j0 + WA_KT - 1 > w_first) {
        // kept keys inside the run's key range
        const int kl = min(a.keep - j0 - 8 * hi, dist + 1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            // a distance below zero (a later key) is a huge unsigned number
            const int o = 32 * h + 16 * (r >> 3) + (r & 7);
            const bool hide = ((unsigned)(dist - o) >= vis) & (o >= kl);
            w[16 * h + r] = hide ? -INFINITY : w[16 * h + r];
          }
      }
      float mx = w[0];
#pragma unroll
      for (int i = 1; i < 32; ++i) mx = fmaxf(mx, w[i]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      bool moved;
      const float alpha = kv_softmax<32>(w, mx, &m, &l, &moved);
      if (moved) {
#pragma unroll
        for (int c = 0; c < VB; ++c)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[c][r] *= alpha;
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        KvPack b0, b1, b2;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          kv_split(w[8 * s + 2 * i], w[8 * s + 2 * i + 1], &b0.w[i],
                   &b1.w[i], &b2.w[i]);
#pragma unroll
        for (int c = 0; c < VB; ++c) {
          KvPack v;
#pragma unroll
          for (int h = 0; h < 2; ++h)
            v.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (kv_lds_s4*)(sv + vat + (16 * s + 4 * h) * PV + 32 * c));
          acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v.v, b0.v, acc[c],
                                                           0, 0, 0);
          acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v.v, b1.v, acc[c],
                                                           0, 0, 0);
          acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v.v, b2.v, acc[c],
                                                           0, 0, 0);
        }
      }
    }
    rs = re;
  }

  l += __shfl_xor(l, 32, 64);  // a lane summed its own keys
  if (!valid || (PART && my_ks >= my_eff)) return;
  float own = 1.f;
  if (a.sink && (!PART || my_ks == 0)) {  // the sink is share 0's
    const float sink = a.sink_vals != nullptr ? a.sink_vals[head] : 0.f;
    if (PART && m == KV_LOW) {  // none of its keys: the sink alone
      m = fminf(fmaxf(sink * KV_LOG2E, KV_LOW), -KV_LOW);
      l = 1.f;
    } else {
      own = kv_sink(sink, &m, &l);
    }
  }
  if constexpr (PART) {
    // partial record per (token, share, head): max (in powers of two),
    // denominator, shares, one unused, DV sums
    float* rec = a.part + (((size_t)tok * a.KS + my_ks) * a.H + head) *
                              (size_t)(DV + WA_HEAD);
    if (hi == 0) {
      rec[0] = l != 0.f ? m : PS_NEG_INF;
      rec[1] = l;
      rec[2] = (float)my_eff;
    }
    if (my_eff > 1) {
      if (l == 0.f) return;  // no key of this share: no sums
#pragma unroll
      for (int c = 0; c < VB; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int col = 32 * c + 8 * q + 4 * hi;
          if (col < DV)  // in steps of 8
            *(float4*)(rec + WA_HEAD + col) =
                make_float4(acc[c][4 * q] * own, acc[c][4 * q + 1] * own,
                            acc[c][4 * q + 2] * own, acc[c][4 * q + 3] * own);
        }
      return;
    }
  }
  const float f = own / l;
  unsigned short* o = a.out + (size_t)tok * a.ldout + (size_t)head * DV;
  const bool vec = ((DV | a.ldout) & 3) == 0 && ((size_t)a.out & 7) == 0;
  // acc[c][4 q + i] = O[row][32 c + 8 q + 4 hi + i]
#pragma unroll
  for (int c = 0; c < VB; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int col = 32 * c + 8 * q + 4 * hi;
      unsigned short e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = ps_f32_to_bf16(acc[c][4 * q + i] * f);
      if (vec) {
        if (col < DV)
          *(uint2*)(o + col) =
              make_uint2((unsigned int)e[0] | ((unsigned int)e[1] << 16),
                         (unsigned int)e[2] | ((unsigned int)e[3] << 16));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (col + i < DV) o[col + i] = e[i];
      }
    }
}

// ---------------------------------------------------------------------------
// single tokens
// ---------------------------------------------------------------------------
#define WA_TT 32    // keys per tile of a wave

// DK: 32-entry steps of a key (D <= 32 DK), VB: 32-column blocks of a value
template <int DK, int VB, bool CAP>
__global__ __launch_bounds__(256, 2) void window_token_kernel(WaArgs a) {
  constexpr int PV = VB * 32 + 8;   // LDS pitch of a value row
  constexpr int PA = VB * 32 + 4;   // and of an output row in the merge
  constexpr int NB = VB * 2;        // 16-column blocks of the output
  static_assert(16 * PA * 4 <= WA_TT * PV * 2, "merge fits the value tile");
  __shared__ __align__(16) unsigned short sV[4][WA_TT * PV];
  __shared__ float s_m[4][16], s_l[4][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // heads first, then tokens, then shares
  const int GH = a.G * a.hblocks;
  const int gh = blockIdx.x % GH, place = blockIdx.x / GH;
  const int ks = place / a.T;
  int t = place - ks * a.T;
  const int g = gh / a.hblocks, hb = gh % a.hblocks;
  if (a.order) {
    auto tiles_of = [&](int i) {
      const int keys = a.token_pos[i] + 1;
      return ((a.window > 0 ? min(keys, a.window) : keys) + WA_TT - 1) / WA_TT;
    };
    t = kv_order(tiles_of, a.T, t, lane, 256 / GH, tiles_of(t),
                 (a.max_blocks * a.BS + WA_TT - 1) / WA_TT);
  }
  const int D = a.D, DV = a.DV, rep = a.H / a.G;
  const int nh = min(16, rep - hb * 16);      // heads of this workgroup
  const int h0 = g * rep + hb * 16;
  const int pos = a.token_pos[t];
  const int* table = a.block_tables + (size_t)a.token_seq[t] * a.max_blocks;
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int k0 = min(a.keep, lo);             // kept keys behind the window
  const int nt0 = (k0 + WA_TT - 1) / WA_TT;
  const int nt = nt0 + (pos - lo) / WA_TT + 1;
  const int hr = lane & 15, kq = lane >> 4;   // head row, key group
  const int head = h0 + min(hr, nh - 1);
  unsigned short* sw = sV[wave];

  // queries: B operand, lane (hr, kq) holds entries 32 s + 8 kq + i
  kv_bf16x8 qr[DK];
  {
    const unsigned short* qp = a.q + (size_t)t * a.ldq + (size_t)head * D;
#pragma unroll
    for (int s = 0; s < DK; ++s) {
      const int c = 32 * s + 8 * kq;
      KvPack u;
      u.q = c < D ? *(const uint4*)(qp + c) : make_uint4(0, 0, 0, 0);
      qr[s] = u.v;
    }
  }
  float m = KV_LOW, l = 0.f;
  // Values the compiler cannot see through where there is a sink: knowing the
  // first tile's state, it lays the walk out such that every tile waits longer
  // (32/8 heads of 64, 8000 keys among 16 x 1000: 54 -> 59 us).
  if (a.sink && ks == 0 && wave == 0) asm volatile("" : "+v"(m), "+v"(l));
  kv_f32x4 acc[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) acc[c] = {0.f, 0.f, 0.f, 0.f};

  // Keys go from memory straight into left operands (a wave's keys are its
  // own), values through LDS for the transposed reads.
  constexpr int CV = VB * 4;                // 16-byte pieces of a value row
  constexpr int NP = WA_TT * CV / 64;       // per lane
  kv_u4 kf[2][DK], pre[NP];
  // key of lane & 31 in tile n; keys past the range's end repeat its last one
  auto first = [&](int n) {
    return n < nt0 ? n * WA_TT : lo + (n - nt0) * WA_TT;
  };
  auto key_of = [&](int n) {
    return min(first(n) + (lane & 31), n < nt0 ? k0 - 1 : pos);
  };
  // score tile x holds keys 8 (row >> 2) + 4 x + (row & 3): a lane's four
  // entries of both are keys 8 kq .. 8 kq + 7
  auto fetch = [&](int n, int page) {
    const int rowi = (page * a.G + g) * a.BS + key_of(n) % a.BS;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int64_t kr = __shfl(rowi, 8 * (hr >> 2) + 4 * x + (hr & 3), 64);
#pragma unroll
      for (int s = 0; s < DK; ++s)
        kf[x][s] = *(const kv_u4*)(a.kc + kr * D +
                                   min(32 * s + 8 * kq, D - 8));
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int idx = u * 64 + lane;
      const int64_t vr = __shfl(rowi, idx / CV, 64);
      pre[u] = *(const kv_u4*)(a.vc + vr * a.vr + min(idx % CV * 8, DV - 8));
    }
  };
  // Loads of tiles past the last repeat it (nothing reads them): without a
  // branch around them no wait is longer than its use asks for. The page
  // number is loaded two tiles ahead.
  const int step = 4 * a.KS;
  int n = ks * 4 + wave, page = 0;
  if (n < nt) {
    fetch(n, table[key_of(n) / a.BS]);
    page = table[key_of(min(n + step, nt - 1)) / a.BS];
  }
  const unsigned short* va = sw + (8 * kq + (hr >> 2)) * PV + 4 * (hr & 3);
  for (; n < nt; n += step) {
    kv_f32x4 st[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < DK; ++s)
#pragma unroll
      for (int x = 0; x < 2; ++x)
        st[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(kv_bf16x8, kf[x][s]), qr[s], st[x], 0, 0, 0);
    kv_wave_sync();  // the previous tile is fully read
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int idx = u * 64 + lane;
      *(kv_u4*)(sw + idx / CV * PV + idx % CV * 8) = pre[u];
    }
    kv_wave_sync();
    fetch(min(n + step, nt - 1), page);
    page = table[key_of(min(n + 2 * step, nt - 1)) / a.BS];
    const int left = (n < nt0 ? k0 : pos + 1) - first(n) - 8 * kq;
    const float base = m == KV_LOW ? 0.f : m;
    float p[8], mx = -INFINITY;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * x + r;
        p[i] = wa_score<CAP>(a, st[x][r], base, a.cap2 - base);
        if (i >= left) p[i] = -INFINITY;
        mx = fmaxf(mx, p[i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    bool moved;
    const float alpha = kv_softmax<8>(p, mx, &m, &l, &moved);
    if (moved) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[c][r] *= alpha;
    }
    KvPack b0, b1, b2;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      kv_split(p[2 * i], p[2 * i + 1], &b0.w[i], &b1.w[i], &b2.w[i]);
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      KvPack v;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        v.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (kv_lds_s4*)(va + 4 * h * PV + 16 * c));
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, b0.v, acc[c], 0, 0,
                                                       0);
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, b1.v, acc[c], 0, 0,
                                                       0);
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, b2.v, acc[c], 0, 0,
                                                       0);
    }
  }

  // merge of the four waves
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lane < 16) {
    s_m[wave][lane] = m;
    s_l[wave][lane] = l;
  }
  kv_wave_sync();  // the wave's last tile is fully read
  // acc[c][r] = O[head row hr][16 c + 4 kq + r]
  float* sa = (float*)sw + hr * PA + 4 * kq;
#pragma unroll
  for (int c = 0; c < NB; ++c)
    *(float4*)(sa + 16 * c) =
        make_float4(acc[c][0], acc[c][1], acc[c][2], acc[c][3]);
  __syncthreads();
  const int vpr = DV / 4;                   // DV is a multiple of 8
  const bool vec = (a.ldout & 3) == 0 && ((size_t)a.out & 7) == 0;
  for (int idx = tid; idx < nh * vpr; idx += 256) {
    const int h = idx / vpr, c = (idx - h * vpr) * 4;
    float mh = fmaxf(fmaxf(s_m[0][h], s_m[1][h]),
                     fmaxf(s_m[2][h], s_m[3][h]));
    float lt = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __builtin_amdgcn_exp2f(s_m[w][h] - mh);
      const float4 v = *(const float4*)((const float*)sV[w] + h * PA + c);
      lt += s_l[w][h] * f;
      o[0] += v.x * f;
      o[1] += v.y * f;
      o[2] += v.z * f;
      o[3] += v.w * f;
    }
    if (a.sink && ks == 0) {  // the sink is share 0's
      const float own = kv_sink(
          a.sink_vals != nullptr ? a.sink_vals[h0 + h] : 0.f, &mh, &lt);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] *= own;
    }
    if (a.KS == 1) {
      const float f = 1.0f / lt;
      unsigned short* dst =
          a.out + (size_t)t * a.ldout + (size_t)(h0 + h) * DV + c;
      unsigned short e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = ps_f32_to_bf16(o[i] * f);
      if (vec)
        *(uint2*)dst =
            make_uint2((unsigned int)e[0] | ((unsigned int)e[1] << 16),
                       (unsigned int)e[2] | ((unsigned int)e[3] << 16));
      else
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = e[i];
    } else {
      // partial record per (token, share, head): max (natural log units),
      // denominator, two unused, DV sums
      float* rec = a.part + (((size_t)t * a.KS + ks) * a.H + h0 + h) *
                                (size_t)(DV + WA_HEAD);
      if (c == 0) {
        rec[0] = lt > 0.f ? mh * 0.69314718f : PS_NEG_INF;
        rec[1] = lt;
      }
      *(float4*)(rec + WA_HEAD + c) = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
}

extern "C" {

void mx_latent_combine(void* out, int ldout, const void* part, int T_, int H,
                       int DV, int KS, void* stream);
void mx_attn_records(void* out, int ldout, const void* part, int T_, int H,
                     int DV, int KS, int counted, int dtype, void* stream);

// Returns 0 when launched, 1 when the shape is outside these kernels: widths of
// whole 16-byte vectors up to 128, rows on 16-byte borders. token: single
// tokens (every batch row on its own; scratch fp32 [T, splits, H, DV + 4] when
// splits > 1), else prompt portions.
int mx_window_attention(void* out, int ldout, const void* q, int ldq,
                        const void* kc, const void* vc,
                        const void* block_tables, int max_blocks,
                        const void* token_seq, const void* token_pos, int T_,
                        int H, int G, int D, int DV, int BS, float scale,
                        int window, int sink, int keep_first, float softcap,
                        const void* sink_vals, int vrow, int token,
                        int splits, void* scratch, void* stream) {
  if (T_ <= 0) return 0;
  if (G < 1 || H < 1 || H % G || BS < 1 || D < 8 || D % 8 || D > 128 ||
      DV < 8 || DV % 8 || DV > 128 || ldq % 8 || vrow % 8 || vrow < DV ||
      (((size_t)q | (size_t)kc | (size_t)vc) & 15))
    return 1;
  typedef unsigned short U;
  const int rep = H / G;
  const bool cap = softcap > 0.f;
  WaArgs a = {(U*)out, ldout, (const U*)q, ldq, (const U*)kc, (const U*)vc,
              vrow, (const int*)block_tables, max_blocks,
              (const int*)token_seq, (const int*)token_pos, T_, H, G, D, DV,
              BS, scale * KV_LOG2E, softcap * KV_LOG2E,
              cap ? 2.f * scale * KV_LOG2E / softcap : 0.f, window,
              keep_first > 0 && window > 0 ? keep_first : 0, sink,
              (const float*)sink_vals, 1, nullptr, 0, 0, 0, 0};
  dim3 grid;
  if (!token) {
    a.hpb = rep < 128 ? rep : 128;
    a.hblocks = (rep + a.hpb - 1) / a.hpb;
    const unsigned gh = G * a.hblocks;
    // 128 rows a workgroup, fewer (to one wave's 32) where those leave CUs idle:
    // a portion of one sequence loses nothing, and short portions of several
    // no longer wait for each other in one workgroup. us, 128 rows -> this (the
    // kernel before): 16 heads of 128 on their own, 8 portions of 16 behind 4000
    // keys 1314 -> 344 (876), 32 of 20 behind 100 70 -> 40 (58); 32/8 heads, 64 of
    // 5 behind 1000 356 -> 185 (366), 64 rows behind 2000 87 -> 81 (226). Down to
    // 16 rows, half a wave's: 344 -> 177, but 81 -> 97; up to 512 workgroups: 2
    // prompts of 2048, 8 heads of 40 60 -> 67. With shares of the keys whole ones fill
    // the CUs (70 rows behind 2500 keys 26 us, 37 with fewer rows). Portions that
    // end up without shares, runs of a workgroup's rows over the workgroups that share
    // them: four of 17 11.4 (20 with all of them the first one's, 11.8 without
    // shares), eight of 30 14.0 (12.0 without shares and their merge, as they are
    // planned where the call says how long and how many they are).
    a.tpt = 128 / a.hpb;
    a.KS = splits > 1 && scratch != nullptr ? splits : 1;
    if (a.KS > 16) return 1;
    a.part = (float*)scratch;
    while (a.KS == 1 && a.tpt > 1 && a.tpt * a.hpb > 32 &&
           (unsigned)((T_ + a.tpt / 2 - 1) / (a.tpt / 2)) * gh <= 256)
      a.tpt /= 2;
    grid = dim3((unsigned)((T_ + a.tpt - 1) / a.tpt) * gh * a.KS);
  } else {
    a.KS = splits > 1 && scratch != nullptr ? splits : 1;
    if (a.KS > 16) return 1;
    a.part = (float*)scratch;
    a.hpb = 16;
    a.hblocks = (rep + 15) / 16;
    const long groups = (long)T_ * G * a.hblocks;
    // By keys (kv_order) where CUs have more than one workgroup and enough keys may
    // be visible, with two or less a CU in a longer window than with more. 32/8
    // heads of 128, us, as they come -> so: 61 tokens of 300 to 4000 keys 114 -> 91,
    // window 2048 77.6 -> 76.3, 1500 54.6 -> 56.4 (50 tokens 47.6 -> 50.1, 1800 57.0 ->
    // 57.7; 40 tokens 44.8 -> 41.1, 64 of 100 to 2500 45.4 -> 43.1); 70 tokens, window
    // 1100 59.4 -> 53.6, 1024 53.3; 100 of 50 to 8000 365 -> 301, 313 of 1000 to 4000
    // 561 -> 536, window 1280 279 -> 278; 64 of 4000 178 -> 176. Where most of two
    // rounds' tokens see a whole window it costs up to 5 % (64 of 300 to 4000, window
    // 2048 76.0 -> 79.8; of 100 to 2500 64.9 -> 56.4).
    // (Heads first, without an order, 512 of 300 to 3000, window 2048 560 -> 542.)
    a.order = a.KS == 1 && groups > 256 && T_ <= KV_ORDER &&
              max_blocks * BS > 1024 &&
              (window <= 0 || window > (groups > 512 ? 1024 : 1536));
    grid = dim3((unsigned)(groups * a.KS));
  }
#define WA_GO(DK, VB, CAP)                                                   \
  do {                                                                       \
    if (token)                                                               \
      hipLaunchKernelGGL((window_token_kernel<DK, VB, CAP>), grid,           \
                         dim3(256), 0, (hipStream_t)stream, a);              \
    else if (a.KS > 1)                                                       \
      hipLaunchKernelGGL((window_prompt_kernel<2 * DK, VB, CAP, true>),      \
                         grid, dim3(256), 0, (hipStream_t)stream, a);        \
    else                                                                     \
      hipLaunchKernelGGL((window_prompt_kernel<2 * DK, VB, CAP, false>),     \
                         grid, dim3(256), 0, (hipStream_t)stream, a);        \
  } while (0)
#define WA_CAP(DK, VB)     \
  do {                     \
    if (cap)               \
      WA_GO(DK, VB, true); \
    else                   \
      WA_GO(DK, VB, false); \
  } while (0)
  if (D <= 64 && DV <= 64)
    WA_CAP(2, 2);
  else if (D <= 64)
    WA_CAP(2, 4);
  else if (DV <= 64)
    WA_CAP(4, 2);
  else
    WA_CAP(4, 4);
#undef WA_CAP
#undef WA_GO
  if (a.KS > 1) {
    if (token)
      mx_latent_combine(out, ldout, scratch, T_, H, DV, a.KS, stream);
    else
      mx_attn_records(out, ldout, scratch, T_, H, DV, a.KS, 1, MX_BF16, stream);
  }
  return 0;
}

}  // extern "C"
