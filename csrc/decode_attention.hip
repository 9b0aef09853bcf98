// Paged decode attention, one query token per sequence, gfx950 matrix cores:
// bf16 or fp8 (e4m3) KV cache [num_blocks, kv_heads, 16, head_dim].
//
// A workgroup has one (sequence, KV head, split of the keys): the query heads
// of a KV head share every byte read. Each of its four waves walks tiles of
// its own (32 keys) in private LDS, no barrier before the merge; the next tile's
// 16 KB (8 of fp8 or heads of 64) are on their way during a tile. Sequences of a
// few tiles of many heads have a wave per head instead.
// Keys go from memory straight into left operands of K Q^T (16 x 16 x 32, the
// query heads padded to 16), so a lane holds runs of 8 consecutive keys of one
// head: the softmax is lane-local plus two exchanges, and the weights pack into
// the second product as three bf16 terms (exact, fp32 accumulation). Values
// pass through LDS for the transposed reads. fp8 entries become bf16 on the way
// (exact).
//
// Bound by the cache read; 32/8 heads of 128 (before: a lane per 8 entries of a
// key on the vector pipe, whose conversions and dot products stood in the way,
// most of all with fp8):
//   64 x 4000 keys   bf16 175 us, 6.0 TB/s (203-235)   fp8  93 us (222)
//   256 x 2000 keys  bf16 346 us (375)                 fp8 183 us (390)
//   32 x 2000 keys   bf16  40 us (58)                  fp8  25 us (65)
//   1 x 4000 keys    bf16 8.7 us (22)                  fp8 8.2 us (22)
// At few keys per CU it is bound by the latency of one tile after another.
#include "attn_common.h"

struct DaArgs {
  unsigned short* out;     // [S, QH, D]
  float* ws_acc;           // [S, QH, splits, D] (splits > 1)
  float* ws_ml;            // [S, QH, splits, 2]: maximum, denominator
  const unsigned short* q;
  const void *kc, *vc;
  const int* block_tables;
  const int* seq_lens;
  int max_blocks, KH, GQ;
  long q_stride;
  float scale2;            // score scale times log2(e)
  int window;
  int seqs;
  int splits;              // of the grid and the workspaces
  int fill;                // splits that a sequence gets at any length
  int packed;              // a wave per head up to this many tiles
  int order;               // sequences by length (da_order)
};

// Keys of one split at most, where the grid has splits left: a workgroup alone
// takes 38 us for 4000 keys, which a batch of 32 sequences hides and one of
// 30000 keys among short ones would not.
#define DA_SPLIT_KEYS 4096

// Splits of a sequence with `keys` visible keys: no more than there are tiles
// for the four waves of each. The others' workgroups end at once.
template <int TT>
PS_DEV int da_splits(int keys, int nsplit, int fill) {
  const int want = max(fill, (keys + DA_SPLIT_KEYS - 1) / DA_SPLIT_KEYS);
  return max(1, min(min(nsplit, want), (keys + 4 * TT - 1) / (4 * TT)));
}

// Tiles of a sequence of `ctx` keys.
template <int TT>
PS_DEV int da_tiles(const DaArgs& a, int ctx) {
  return ((a.window > 0 ? min(ctx, a.window) : ctx) + TT - 1) / TT;
}

// The sequence of a place (see kv_order). 32/8 heads of 128, us, as they come /
// longest first / this / all of one length: 61 sequences of 300 to 4000 keys 117 /
// 105 / 93 / 92, 100 of 500 to 3000 157 / 136 / 131 / 142; fp8, 192 of 1200 to 5500
// 250 / 228 / 227 / 227. With sequences in splits as they come: by length fp8, 34 of
// 300 to 6000 took 53 us instead of 48, 36 of 1000 to 8000 91 instead of 83, bf16 61
// of 1000 to 8000 210 instead of 201 (three draws each).
template <int TT>
PS_DEV int da_order(const DaArgs& a, int pos, int ctx, int lane) {
  return kv_order([&](int s) { return da_tiles<TT>(a, a.seq_lens[s]); }, a.seqs,
                  pos, lane, 256 / a.KH, da_tiles<TT>(a, ctx),
                  (a.max_blocks * 16 + TT - 1) / TT,
                  a.splits > 1 ? DA_SPLIT_KEYS / TT : 0x7fffffff);
}

// 8 fp8 entries as bf16
PS_DEV kv_bf16x8 da_bf16(unsigned int lo, unsigned int hi) {
  KvPack u;
  u.w[0] = __builtin_bit_cast(
      unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false));
  u.w[1] = __builtin_bit_cast(
      unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true));
  u.w[2] = __builtin_bit_cast(
      unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false));
  u.w[3] = __builtin_bit_cast(
      unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true));
  return u.v;
}

template <int D, int TT, bool FP8, int WPE>
__global__ __launch_bounds__(256, WPE) void paged_attn_decode_kernel(DaArgs a) {
  constexpr int EB = FP8 ? 1 : 2;      // bytes per entry
  constexpr int RB = D * EB;           // per cache row
  constexpr int CR = RB / 16;          // 16-byte pieces of a row
  constexpr int NK = CR / 4;           // of them per lane and score tile
  constexpr int NX = TT / 16;          // score tiles
  constexpr int DK = D / 32;           // 32-entry steps of a key
  constexpr int NP = TT * CR / 64;     // pieces of a value tile per lane
  constexpr int PV = D + 8;            // LDS pitch of a value row
  constexpr int PA = D + 4;            // and of an output row in the merge
  constexpr int NB = D / 16;           // 16-column blocks of the output
  constexpr int BS = 16;               // keys per page
  static_assert(16 * PA * 4 <= TT * PV * 2, "merge fits the value tile");
  __shared__ __align__(16) unsigned short sV[4][TT * PV];
  __shared__ float s_m[4][16], s_l[4][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int KH = a.KH, GQ = a.GQ;
  // Workgroups go round the XCDs and their shader engines in turn. Heads are
  // counted first, so that a long sequence is on all of them; splits last, so
  // that those with something to do are not always the same ones (32 sequences
  // of 2000 keys, one split in four in use: 81 us with the sequence last, 40
  // here); and each split starts one sequence on, which moves a sequence's
  // splits apart where there are few heads (32 sequences, one of 30000 keys:
  // 176 us with its splits on one XCD).
  int kvh = blockIdx.x % KH;
  const int r = blockIdx.x / KH;
  const int split = r / a.seqs;
  const int pos = (r - split * a.seqs + split) % a.seqs;
  int seq = pos, ctx = a.seq_lens[pos];
  if (a.order) {
    seq = da_order<TT>(a, pos, ctx, lane);
    if (seq != pos) ctx = a.seq_lens[seq];
  }
  const int lo = a.window > 0 && ctx > a.window ? ctx - a.window : 0;
  const int nt = (ctx - lo + TT - 1) / TT;
  const int nsplit = da_splits<TT>(ctx - lo, a.splits, a.fill);
  if (split >= nsplit) return;
  // Few tiles of many heads: one workgroup of four has a wave for each of four
  // heads, the other three end here. Which one goes with the place such
  // that all XCDs, and all of an XCD's engines, get the same share (512 x 40
  // keys of 16/8 heads 42 us with kvh + seq, 20 so).
  const bool packed = a.packed > 0 && nt <= a.packed;
  if (packed) {
    if (((kvh + pos + (pos >> 2)) & 3) != 0) return;
    kvh = (kvh & ~3) + wave;
  }
  const int* table = a.block_tables + (long)seq * a.max_blocks;
  const int hr = lane & 15, kq = lane >> 4;   // head row, key group
  const unsigned char* kc = (const unsigned char*)a.kc;
  const unsigned char* vc = (const unsigned char*)a.vc;
  unsigned short* sw = sV[wave];

  // Queries: B operand. A lane's 16 bytes of a key are 8 entries of one step
  // (bf16) or of two steps (fp8); the entries of a step may stand in any order
  // that keys and queries share.
  kv_bf16x8 qr[DK];
  {
    const unsigned short* qp = a.q + (long)seq * a.q_stride +
                               (long)(kvh * GQ + min(hr, GQ - 1)) * D;
#pragma unroll
    for (int s = 0; s < DK; ++s)
      qr[s] = *(const kv_bf16x8*)(
          qp + (FP8 ? 64 * (s >> 1) + 16 * kq + 8 * (s & 1)
                    : 32 * s + 8 * kq));
  }
  float m = KV_LOW, l = 0.f;
  kv_f32x4 acc[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) acc[c] = {0.f, 0.f, 0.f, 0.f};

  kv_u4 kf[NX][NK], pre[NP];
  // this lane's key of tile n; keys past the context repeat its last one
  auto key_of = [&](int n) {
    return min(lo + n * TT + (lane & (TT - 1)), ctx - 1);
  };
  // score tile x holds keys 32 (x >> 1) + 8 (row >> 2) + 4 (x & 1) + (row & 3):
  // a lane's entries of a pair are keys 8 kq .. 8 kq + 7 of 32
  auto fetch = [&](int n, int page) {
    const int rowi = (page * KH + kvh) * BS + key_of(n) % BS;
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int64_t kr = __shfl(
          rowi, 32 * (x >> 1) + 8 * (hr >> 2) + 4 * (x & 1) + (hr & 3), 64);
#pragma unroll
      for (int s = 0; s < NK; ++s)
        kf[x][s] = *(const kv_u4*)(kc + kr * RB + 64 * s + 16 * kq);
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int idx = u * 64 + lane;
      const int64_t vr = __shfl(rowi, idx / CR, 64);
      pre[u] = *(const kv_u4*)(vc + vr * RB + idx % CR * 16);
    }
  };
  // Loads of tiles past the last are all of the last key (nothing reads them):
  // without a branch around them no wait is longer than its use asks for. The
  // page number is loaded two tiles ahead.
  const int step = packed ? 1 : 4 * nsplit;
  int n = packed ? 0 : split * 4 + wave, page = 0;
  if (n < nt) {
    fetch(n, table[key_of(n) / BS]);
    page = table[key_of(n + step) / BS];
  }
  const unsigned short* va = sw + (8 * kq + (hr >> 2)) * PV + 4 * (hr & 3);
  for (; n < nt; n += step) {
    kv_f32x4 st[NX];
#pragma unroll
    for (int x = 0; x < NX; ++x) st[x] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NK; ++s)
#pragma unroll
      for (int x = 0; x < NX; ++x) {
        if constexpr (FP8) {
          st[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              da_bf16(kf[x][s][0], kf[x][s][1]), qr[2 * s], st[x], 0, 0, 0);
          st[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              da_bf16(kf[x][s][2], kf[x][s][3]), qr[2 * s + 1], st[x], 0, 0,
              0);
        } else {
          st[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(kv_bf16x8, kf[x][s]), qr[s], st[x], 0, 0, 0);
        }
      }
    kv_wave_sync();  // the previous tile is fully read
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int idx = u * 64 + lane;
      unsigned short* d = sw + idx / CR * PV + idx % CR * (16 / EB);
      if constexpr (FP8) {
        *(kv_bf16x8*)d = da_bf16(pre[u][0], pre[u][1]);
        *(kv_bf16x8*)(d + 8) = da_bf16(pre[u][2], pre[u][3]);
      } else {
        *(kv_u4*)d = pre[u];
      }
    }
    kv_wave_sync();
    fetch(n + step, page);
    page = table[key_of(n + 2 * step) / BS];

    const int left = ctx - (lo + n * TT) - 8 * kq;
    const float base = m == KV_LOW ? 0.f : m;
    float p[4 * NX], mx = -INFINITY;
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * x + r;
        p[i] = st[x][r] * a.scale2 - base;
        if (32 * (x >> 1) + 4 * (x & 1) + r >= left) p[i] = -INFINITY;
        mx = fmaxf(mx, p[i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    bool moved;
    const float alpha = kv_softmax<4 * NX>(p, mx, &m, &l, &moved);
    if (moved) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[c][r] *= alpha;
    }
#pragma unroll
    for (int y = 0; y < TT / 32; ++y) {
      KvPack b0, b1, b2;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        kv_split(p[8 * y + 2 * i], p[8 * y + 2 * i + 1], &b0.w[i], &b1.w[i],
                 &b2.w[i]);
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        KvPack v;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (kv_lds_s4*)(va + (32 * y + 4 * h) * PV + 16 * c));
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, b0.v, acc[c], 0,
                                                         0, 0);
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, b1.v, acc[c], 0,
                                                         0, 0);
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, b2.v, acc[c], 0,
                                                         0, 0);
      }
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
  if (packed) {
    kv_wave_sync();
    for (int idx = lane; idx < GQ * (D / 4); idx += 64) {
      const int h = idx / (D / 4), c = idx % (D / 4) * 4;
      const float lt = s_l[wave][h];
      const float f = lt > 0.f ? 1.0f / lt : 0.f;
      const float4 v = *(const float4*)((const float*)sw + h * PA + c);
      *(uint2*)(a.out + (((long)seq * KH + kvh) * GQ + h) * D + c) =
          make_uint2((unsigned int)ps_f32_to_bf16(v.x * f) |
                         ((unsigned int)ps_f32_to_bf16(v.y * f) << 16),
                     (unsigned int)ps_f32_to_bf16(v.z * f) |
                         ((unsigned int)ps_f32_to_bf16(v.w * f) << 16));
    }
    return;
  }
  __syncthreads();
  for (int idx = tid; idx < GQ * (D / 4); idx += 256) {
    const int h = idx / (D / 4), c = idx % (D / 4) * 4;
    const float mh = fmaxf(fmaxf(s_m[0][h], s_m[1][h]),
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
    const long head = ((long)seq * KH + kvh) * GQ + h;
    if (nsplit == 1) {
      const float f = lt > 0.f ? 1.0f / lt : 0.f;
      unsigned short e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = ps_f32_to_bf16(o[i] * f);
      *(uint2*)(a.out + head * D + c) =
          make_uint2((unsigned int)e[0] | ((unsigned int)e[1] << 16),
                     (unsigned int)e[2] | ((unsigned int)e[3] << 16));
    } else {
      *(float4*)(a.ws_acc + (head * a.splits + split) * D + c) =
          make_float4(o[0], o[1], o[2], o[3]);
      if (c == 0)
        *(float2*)(a.ws_ml + (head * a.splits + split) * 2) =
            make_float2(mh, lt);
    }
  }
}

// Merges the splits of one head, maxima in powers of two. A wave takes every
// fourth split. Where all sequences are split (EAGER) the maxima and the first
// eight shares of each wave are asked for beside the context's length: one trip to
// memory instead of one for each in turn (attention and merge, 32/8 heads of 128, 1 x
// 4000 keys 9.9 -> 9.2 us, 2 x 2000 11.0 -> 9.6; 32/8 of 64, 1 x 517 7.2 -> 6.7).
// Otherwise most heads are in place and their workgroups end at once.
template <int D, int TT, bool EAGER>
__global__ __launch_bounds__(256) void paged_attn_combine_kernel(DaArgs a) {
  const int pitch = a.splits;
  constexpr int E = D / 64;  // entries per lane
  constexpr int PRE = EAGER ? 8 : 0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long head = blockIdx.x;
  const float* ml = a.ws_ml + head * pitch * 2;
  const float* acc = a.ws_acc + head * pitch * D + lane * E;
  const int ctx = a.seq_lens[head / (a.KH * a.GQ)];
  float2 own = *(const float2*)(ml + 2 * min(lane, pitch - 1));
  float pre[PRE + 1][E];
#pragma unroll
  for (int i = 0; i < PRE; ++i)
#pragma unroll
    for (int e = 0; e < E; ++e)
      pre[i][e] = acc[(long)min(wave + 4 * i, pitch - 1) * D + e];
  if constexpr (EAGER) asm volatile("" ::: "memory");  // not behind the branch
  const int keys = a.window > 0 && ctx > a.window ? a.window : ctx;
  const int nsplit = da_splits<TT>(keys, pitch, a.fill);
  if (nsplit == 1) return;   // already in place
  __shared__ float s_o[4][D];
  if (lane >= nsplit) own = make_float2(KV_LOW, 0.f);
  float M = own.x;
  for (int s = lane + 64; s < nsplit; s += 64) M = fmaxf(M, ml[2 * s]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    M = fmaxf(M, __shfl_xor(M, off, 64));
  float L = own.y * __builtin_amdgcn_exp2f(own.x - M);
  for (int s = lane + 64; s < nsplit; s += 64)
    L += ml[2 * s + 1] * __builtin_amdgcn_exp2f(ml[2 * s] - M);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off, 64);
  float o[E];
#pragma unroll
  for (int i = 0; i < E; ++i) o[i] = 0.f;
#pragma unroll
  for (int i = 0; i < PRE; ++i) {
    const int s = wave + 4 * i;
    const float f = __builtin_amdgcn_exp2f(
        __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(own.x), s)) -
        M);
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] += s < nsplit ? pre[i][e] * f : 0.f;
  }
#pragma unroll 8
  for (int s = wave + 4 * PRE; s < nsplit; s += 4) {
    const float f = __builtin_amdgcn_exp2f(ml[2 * s] - M);
#pragma unroll
    for (int i = 0; i < E; ++i) o[i] += acc[(long)s * D + i] * f;
  }
#pragma unroll
  for (int i = 0; i < E; ++i) s_o[wave][lane * E + i] = o[i];
  __syncthreads();
  if (threadIdx.x < D) {
    const int c = threadIdx.x;
    const float t = (s_o[0][c] + s_o[1][c]) + (s_o[2][c] + s_o[3][c]);
    a.out[head * D + c] = ps_f32_to_bf16(L > 0.f ? t / L : 0.f);
  }
}

// num_splits: splits of the grid (and of the workspaces); fill: how many of
// them a sequence gets whatever its length.
extern "C" int ps_paged_attn_decode(
    void* out, void* ws_acc, void* ws_ml, const void* q, const void* k_cache,
    const void* v_cache, const void* block_tables, const void* seq_lens,
    int num_seqs, int max_blocks, float scale, int KH, int GQ, int head_dim,
    int block_size, int num_splits, int fill, long q_stride, int kv_fp8,
    int window, hipStream_t stream) {
  if (GQ < 1 || GQ > 8 || GQ == 5 || block_size != 16 || num_splits < 1)
    return -1;
  if (head_dim != 128 &&
      (head_dim != 64 || kv_fp8 || GQ == 3 || GQ == 6 || GQ == 7))
    return -1;
  // A wave per head where four waves would not have a tile each and every CU has
  // eight workgroups to go through: their chain of loads and the merge take
  // longer than the few keys (us, four waves a head -> one, in brackets the
  // vector kernel that was here before; 32 heads of their own, 128: bf16 512 x 40
  // keys 93 -> 67 (73), 256 x 60 50 -> 43 (43); fp8 512 x 40 72 -> 41 (41), 256 x
  // 100 46 -> 36 (37), 64 x 100 15.8 -> 15.7 (13.7)). Of bf16 up to two tiles (64
  // x 100 keys 20.8 -> 23.0 with three), of heads of 64 twice the workgroups (64 x
  // 40 8.0 -> 8.6, 128 x 30 14.0 -> 11.4).
  const bool many = (long)num_seqs * KH >= (head_dim == 64 ? 4096 : 2048);
  const int packed = KH % 4 == 0 && many ? (kv_fp8 ? 4 : 2) : 0;
  // By length (da_order) where CUs have more than one workgroup and there may be
  // more than 1024 keys: below, the trip to memory for all lengths costs more than
  // the order gives (64 sequences of up to 1000 keys 33.6 us, 30.5 ordered, but 256
  // of up to 500 60.7 / 63.5; 64 of one length 94 / 95; 61 of up to 4000 of which a
  // window shows 1500 54 / 56). Over 320 sequences fill the CUs five times over, and
  // the order's counts take their time in each workgroup: fp8, 512 of up to 1000
  // keys 111 / 120. Long ones would gain even so (400 of 1000 to 8000 689 / 649), but
  // lengths are not known here, and a lane would hold more counts.
  const int width =
      window > 0 ? std::min(window, max_blocks * 16) : max_blocks * 16;
  const int order =
      num_seqs * KH > 256 && num_seqs <= KV_ORDER &&
      width > (window > 0 ? 2048 : 1024);
  const DaArgs a = {(unsigned short*)out,
                    (float*)ws_acc,
                    (float*)ws_ml,
                    (const unsigned short*)q,
                    k_cache,
                    v_cache,
                    (const int*)block_tables,
                    (const int*)seq_lens,
                    max_blocks,
                    KH,
                    GQ,
                    q_stride,
                    scale * KV_LOG2E,
                    window,
                    num_seqs,
                    num_splits,
                    fill,
                    packed,
                    order};
  const dim3 grid((unsigned)num_seqs * KH * num_splits), block(256);
  const dim3 heads(num_seqs * KH * GQ);
#define DA_GO(D, TT, FP8, WPE)                                               \
  do {                                                                       \
    paged_attn_decode_kernel<D, TT, FP8, WPE><<<grid, block, 0, stream>>>(a); \
    if (fill > 1)                                                            \
      paged_attn_combine_kernel<D, TT, true><<<heads, block, 0, stream>>>(a); \
    else if (num_splits > 1)                                                 \
      paged_attn_combine_kernel<D, TT, false>                                \
          <<<heads, block, 0, stream>>>(a);                                  \
  } while (0)
  // Tiles of 32 keys everywhere: short contexts share out among the waves (us, 64
  // keys -> 32, before in brackets: heads of 64, 64 x 300 keys, 32 heads of their
  // own 30.7 -> 26.3 (27.1), 32/8 heads 256 x 200 23.4 -> 19.5; fp8, 32 heads of
  // their own, 64 x 300 36.6 -> 28.9 (28.3), 256 x 300 137 -> 111 (119), 64 x 4000
  // 348 -> 347 (409), 32 x 2000 94 -> 99 (111); 32/8 256 x 300 37.0 -> 28.9).
  // bf16 of 128: a third workgroup a CU where there is one and heads have keys of
  // their own (32 heads, 256 x 100 keys 90 -> 78 (84), 64 x 100 23.4 -> 20.9 (20.3)).
  // Heads that share them are 5 % faster or slower with it as the lengths differ
  // (32/8, 100 sequences of 500 to 3000 keys 156 -> 151, 150 of 40 to 2000 127 ->
  // 132); two a CU cost its registers 3 % (8 x 1000 keys of 8 heads 10.0 -> 10.3).
  if (head_dim == 64)
    DA_GO(64, 32, false, 2);
  else if (kv_fp8)
    DA_GO(128, 32, true, 2);
  else if (GQ == 1 && (long)num_seqs * KH * fill > 512)
    DA_GO(128, 32, false, 3);
  else
    DA_GO(128, 32, false, 2);
#undef DA_GO
  return 0;
}
