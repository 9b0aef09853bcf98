// Grouped-query attention over the paged cache in fp32, gfx950 matrix cores:
// trailing window with kept first keys, aligned chunks or everything, capped
// scores, sink in the denominator; ragged prompt portions and single tokens.
// Head widths up to 128 in steps of 16.
//
// A wave has 16 or 32 columns, (token, head) pairs of one KV head, and walks
// tiles of 16 keys on its own: S^T = K Q^T, O^T = V^T P^T by
// v_mfma_f32_16x16x4_f32. Its operands need no exchange at all. The contraction
// runs over four lane groups g; what a group's index stands for is free as long as
// both operands agree:
//   scores  step e of 16 entries takes entries 4 g + e: a lane's four steps are one
//           16-byte load of its key's row;
//   output  step i takes keys 4 g + i, which is where the scores of keys 4 g + i
//           are, so that weights go from the softmax straight into the product;
//           its rows are entries 4 n + e, again one 16-byte load of a value row.
// So keys and values go from memory into operands, no LDS and no barrier in the
// walk. Values of a tile and keys of the next are on their way during the other
// product (2000 to 4000 cycles with 16 or 32 columns of 128).
//
// The four waves of a workgroup share their columns and take turns at the tiles,
// and where that leaves CUs idle `splits` workgroups share them too (records merged
// by mx_attn_records): a few rows behind a long history are a chain of tiles
// otherwise. Workgroups of a KV head are eight apart and meet in one XCD's L2.
//
// Bound by the fp32 matrix unit and what a wave alone cannot lay beside it (prompts,
// two waves a SIMD at widths of 128) and by memory (single tokens, whose heads fill a
// quarter of the columns). 32/8 heads of 128, us, by the vector kernels of
// talk_attention.hip -> by this one: 254 rows in 3 portions, one behind 2264 keys, cap
// 7430 -> 84; 80 rows behind 334 keys 1360 -> 21; 1000 rows of 64 in 3 prompts 562 ->
// 35; 1000 rows 120, with a cap 130, half the fp32 matrix rate; one token behind 947
// keys 345 -> 19; 64 behind 1500 139, 5.7 TB/s.
// Errors against 64 bits are those of the vector kernels or less (40 tokens of up to 900
// keys 2.3e-7 and 2.1e-7, 128 of up to 300 2.1e-7 and 2.0e-7): with 16 columns a wave
// sums are short chains that are added up, scores by 16 entries, outputs by tiles (40
// tokens with outputs in one chain over all keys and scores by 32 3.3e-7 and 78.7 us,
// 79.8 so). With 32 there are no registers for that: scores by 64 entries, outputs in
// one chain over a wave's keys (vector / 16 / 32 columns: 523 rows 2.7e-7 / 1.4e-7 /
// 2.2e-7, 1000 behind 3000 keys 1.4e-6 / 2.4e-7 / 5.9e-7, 523 behind 6000 1.8e-6 /
// 2.7e-7 / 7.6e-7).
#include "attn_common.h"

struct AfArgs {
  float* out;
  int ldout;
  const float* q;
  int ldq;
  const float *kc, *vc;  // [NB, G, BS, D], [NB, G, BS, vr]
  int vr;
  const int* block_tables;
  int max_blocks;
  const int *token_seq, *token_pos;
  int T, H, G, D, DV, BS;
  float scale, cap;  // cap 0: none
  int chunk, window, keep, sink;
  const float* sink_vals;  // per head (nullptr: score 0)
  int hide;                // scores that are no number hide their keys
  int tpt;                 // tokens per workgroup
  int KS;
  float* part;  // [T, KS, H, DV + AF_HEAD]
};

#define AF_HEAD 4  // leading entries of a partial record: max, denominator
#define AF_KT 16

PS_DEV bool af_odd(float x) { return !(fabsf(x) < INFINITY); }

// NT: 16-entry steps of a key (D <= 16 NT), NV: 64-entry blocks of a value, NC:
// 16-column tiles of a wave
template <int NT, int NV, int NC, bool CAP>
__global__ __launch_bounds__(256, 2) void attn_f32_kernel(AfArgs a) {
  constexpr int COLS = 16 * NC, PA = NV * 64 + 4;
  constexpr int NS = NC * NT > 8 ? 2 : NT;  // sums of a score; more would spill
  constexpr bool APART = NC == 1;
  // Which keys are hidden is kept for the careful walk as masks or, with a cap and 32
  // columns, found again there: registers (masks / found again, 1000 rows of 128 with a
  // cap 132.8 / 130.0 us, without one 120.0 / 122.2).
  constexpr bool AGAIN = NC == 2 && CAP;
  extern __shared__ __align__(16) float sA[];  // [4][COLS][PA]: the merge
  __shared__ float s_m[4][COLS], s_l[4][COLS];
  __shared__ int s_seq[COLS], s_pos[COLS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, n = lane & 15;
  // KV heads first, then shares, then rows, the last ones, which see the most
  // keys, ahead
  const int G = a.G, rep = a.H / G, BS = a.BS;
  const int kvh = blockIdx.x % G;
  const int place = blockIdx.x / G;
  const int ks = place % a.KS;
  const int tile = (a.T + a.tpt - 1) / a.tpt - 1 - place / a.KS;
  const int tok0 = tile * a.tpt, ntok = min(a.tpt, a.T - tok0);
  if (tid < ntok) {
    s_seq[tid] = a.token_seq[tok0 + tid];
    s_pos[tid] = a.token_pos[tok0 + tid];
  }
  __syncthreads();

  auto low = [&](int p) {
    int lo = 0;
    if (a.chunk > 0) lo = p / a.chunk * a.chunk;
    if (a.window > 0) lo = max(lo, p - a.window + 1);
    return lo;
  };
  // this lane's columns
  int my_i[NC], my_pos[NC], my_lo[NC];
  float4 qf[NC][NT];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int col = c * 16 + n;
    const bool on = col < ntok * rep;
    const int i = on ? col / rep : 0, h = on ? col - i * rep : 0;
    my_i[c] = on ? i : -1;
    my_pos[c] = s_pos[i];
    my_lo[c] = low(my_pos[c]);
    const float* qp =
        a.q + (size_t)(tok0 + i) * a.ldq + (size_t)(kvh * rep + h) * a.D + 4 * g;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      qf[c][t] = 16 * t < a.D ? *(const float4*)(qp + 16 * t)
                              : make_float4(0.f, 0.f, 0.f, 0.f);
  }

  float m[NC], l[NC];
  kv_f32x4 acc[NC][NV][4];
  // The walk; again, `careful`, where values that are not finite were met: they
  // stay out of the products, in which a hidden key's weight of zero would carry
  // them to columns that do not see it, and join those that do with their weights.
  bool careful = false;
#pragma unroll 1
  for (;;) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      m[c] = PS_NEG_INF;
      l[c] = 0.f;
#pragma unroll
      for (int h = 0; h < NV; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[c][h][e] = kv_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int rs = 0;
    while (rs < ntok) {
      // tokens rs .. re - 1 continue one sequence
      int re = rs + 1;
      while (re < ntok && s_seq[re] == s_seq[rs] &&
             s_pos[re] == s_pos[re - 1] + 1)
        ++re;
      const int* table = a.block_tables + (size_t)s_seq[rs] * a.max_blocks;
      const int kmin = low(s_pos[rs]), kmax = s_pos[re - 1];
      const int k0 = min(a.keep, kmin);  // kept keys behind the window
      const int nt0 = (k0 + AF_KT - 1) / AF_KT;
      const int nt = nt0 + (kmax - kmin) / AF_KT + 1;
      auto first = [&](int t) {
        return t < nt0 ? t * AF_KT : kmin + (t - nt0) * AF_KT;
      };
      // this lane's key of tile t; those past the range's end repeat its last
      auto key_of = [&](int t) {
        return min(first(t) + n, t < nt0 ? k0 - 1 : kmax);
      };
      auto row_of = [&](int t, int page) {
        return (page * G + kvh) * BS + key_of(t) % BS;
      };
      float4 kf[NT], vf[4][NV];
      auto fetch_k = [&](int row) {
        const float* kp = a.kc + (int64_t)row * a.D + 4 * g;
#pragma unroll
        for (int t = 0; t < NT; ++t)
          kf[t] = 16 * t < a.D ? *(const float4*)(kp + 16 * t)
                               : make_float4(0.f, 0.f, 0.f, 0.f);
      };
      auto fetch_v = [&](int row) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* vp =
              a.vc + (int64_t)__shfl(row, 4 * g + i, 64) * a.vr;
#pragma unroll
          for (int h = 0; h < NV; ++h)
            vf[i][h] = *(const float4*)(vp + min(64 * h + 4 * n, a.DV - 4));
        }
      };
      const int step = 4 * a.KS;
      int t = ks * 4 + wave;
      if (t < nt) {
        // pages two tiles ahead; tiles past the last repeat it, unread
        int row = row_of(t, table[key_of(t) / BS]);
        int tn = min(t + step, nt - 1);
        int page = table[key_of(tn) / BS];
        fetch_k(row);
        for (; t < nt; t += step) {
          const int here = row;
          fetch_v(here);
          kv_f32x4 st[NC][NS];
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int s = 0; s < NS; ++s) st[c][s] = kv_f32x4{0.f, 0.f, 0.f, 0.f};
          // sums of every NS-th 16 entries: shorter chains of roundings
#pragma unroll
          for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int c = 0; c < NC; ++c)
                st[c][s % NS] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                    (&kf[s].x)[e], (&qf[c][s].x)[e], st[c][s % NS], 0, 0, 0);
          row = row_of(tn, page);
          tn = min(t + 2 * step, nt - 1);
          page = table[key_of(tn) / BS];
          __builtin_amdgcn_sched_barrier(0);
          fetch_k(row);
          // scores: lane (g, n) has keys 4 g + i of column n
          const int j0 = first(t) + 4 * g;
          const int end = t < nt0 ? k0 - 1 : kmax;
          bool seen[NC][4];
          unsigned hid = 0;
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const bool mine = my_i[c] >= rs && my_i[c] < re;
            float p[4], mx = PS_NEG_INF;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = j0 + i;
              float y[NS];
#pragma unroll
              for (int s = 0; s < NS; ++s) y[s] = st[c][s][i];
#pragma unroll
              for (int w = NS / 2; w > 0; w /= 2)
#pragma unroll
                for (int s = 0; s < w; ++s) y[s] += y[s + w];
              float x = y[0] * a.scale;
              if constexpr (CAP) x = a.cap * tanhf(x / a.cap);
              const bool vis = mine && j <= min(end, my_pos[c]) &&
                               (j >= my_lo[c] || j < a.keep);
              seen[c][i] = vis && (x > PS_NEG_INF || !a.hide);
              p[i] = seen[c][i] ? x : -INFINITY;
              mx = fmaxf(mx, p[i]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            if (AGAIN && careful) {
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (p[i] == -INFINITY) hid |= 1u << (4 * c + i);
            }
            if (__any(mx > m[c])) {
              const float mn = fmaxf(m[c], mx);
              const float al = expf(m[c] - mn);
              m[c] = mn;
              l[c] *= al;
#pragma unroll
              for (int h = 0; h < NV; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[c][h][e] *= al;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              p[i] = expf(p[i] - m[c]);
              st[c][0][i] = p[i];
            }
            l[c] += (p[0] + p[1]) + (p[2] + p[3]);
          }
          if (careful) {
#pragma unroll 1
            for (int k = 0; k < AF_KT; ++k) {
              const float* vp = a.vc + (int64_t)__shfl(here, k, 64) * a.vr;
              int d0 = 16 * g;  // not known ahead: addresses are made here
              asm volatile("" : "+v"(d0));
              float w[NC];  // weights of key k, below 0 where it is hidden
#pragma unroll
              for (int c = 0; c < NC; ++c) {
                float own = -1.f;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  if ((k & 3) == i &&
                      (AGAIN ? !(hid >> (4 * c + i) & 1) : seen[c][i]))
                    own = st[c][0][i];
                w[c] = __shfl(own, k / 4 * 16 + n, 64);
              }
#pragma unroll
              for (int h = 0; h < NV; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const float4 x =
                      *(const float4*)(vp + min(64 * h + d0 + 4 * i, a.DV - 4));
#pragma unroll
                  for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                      if (!(w[c] < 0.f) && af_odd((&x.x)[e]))
                        acc[c][h][e][i] += w[c] * (&x.x)[e];
                  __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int h = 0; h < NV; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  if (af_odd((&vf[i][h].x)[e])) (&vf[i][h].x)[e] = 0.f;
          }
          // a tile's products on their own where registers allow: added one by
          // one to the sums of all tiles before, roundings grow with their number
          kv_f32x4 sum[NC][NV][4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int h = 0; h < NV; ++h)
#pragma unroll
              for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                  kv_f32x4& to = APART ? sum[c][h][e] : acc[c][h][e];
                  const kv_f32x4 from =
                      APART && i == 0 ? kv_f32x4{0.f, 0.f, 0.f, 0.f} : to;
                  to = __builtin_amdgcn_mfma_f32_16x16x4f32(
                      (&vf[i][h].x)[e], st[c][0][i], from, 0, 0, 0);
                }
          if constexpr (APART) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
              for (int h = 0; h < NV; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[c][h][e] += sum[c][h][e];
          }
        }
      }
      rs = re;
    }
    bool odd = false;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int h = 0; h < NV; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) odd |= af_odd(acc[c][h][e][i]);
    if (careful || !__any(odd)) break;
    careful = true;
  }

  // merge of the four waves; acc[c][h][e][i]: entry 64 h + 16 g + 4 i + e
  float* sw = sA + wave * COLS * PA;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float lt = l[c];
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
    if (g == 0) {
      s_m[wave][c * 16 + n] = m[c];
      s_l[wave][c * 16 + n] = lt;
    }
#pragma unroll
    for (int h = 0; h < NV; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *(float4*)(sw + (c * 16 + n) * PA + 64 * h + 16 * g + 4 * i) =
            make_float4(acc[c][h][0][i], acc[c][h][1][i], acc[c][h][2][i],
                        acc[c][h][3][i]);
  }
  __syncthreads();
  const int vpr = a.DV / 4;
  for (int idx = tid; idx < ntok * rep * vpr; idx += 256) {
    const int col = idx / vpr, d = (idx - col * vpr) * 4;
    const int i = col / rep, head = kvh * rep + col - i * rep;
    float mh = PS_NEG_INF;
#pragma unroll
    for (int w = 0; w < 4; ++w) mh = fmaxf(mh, s_m[w][col]);
    const bool sink = a.sink && ks == 0;  // the sink is share 0's
    const float sv = a.sink_vals != nullptr ? a.sink_vals[head] : 0.f;
    if (sink) mh = fmaxf(mh, sv);
    float lt = sink ? expf(sv - mh) : 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = expf(s_m[w][col] - mh);
      if (s_m[w][col] == PS_NEG_INF && !(s_l[w][col] != s_l[w][col])) continue;
      const float4 v = *(const float4*)(sA + (w * COLS + col) * PA + d);
      lt += s_l[w][col] * f;
      o[0] += v.x * f;
      o[1] += v.y * f;
      o[2] += v.z * f;
      o[3] += v.w * f;
    }
    if (a.KS == 1) {
      const float f = 1.0f / lt;
      float* dst = a.out + (size_t)(tok0 + i) * a.ldout + head * a.DV + d;
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[e] = o[e] * f;
    } else {
      float* rec = a.part + (((size_t)(tok0 + i) * a.KS + ks) * a.H + head) *
                                (size_t)(a.DV + AF_HEAD);
      if (d == 0) {
        rec[0] = mh;
        rec[1] = lt;
      }
      if (lt != 0.f)  // else no key of this share: no sums
        *(float4*)(rec + AF_HEAD + d) = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
}

// Merge of `KS` (at most AF_KS) partial records of every (token, head): 256 threads
// of four entries each. Shares without a key have a denominator of 0 and no sums.
// counted: the first record's third entry is how many there are, of a single one the
// result is already there, and maxima are powers of two (as natural logarithms, ones
// around 100 were rounded by 1e-5 of a share's weight).
#define AF_KS 16
template <typename T>
__global__ __launch_bounds__(256) void attn_records_kernel(
    T* __restrict__ out, int ldout, const float* __restrict__ part, int H,
    int DV, int KS, int counted) {
  const int vpr = DV / 4, idx = blockIdx.y * 256 + threadIdx.x;
  if (idx >= H * vpr) return;
  const int h = idx / vpr, d = (idx - h * vpr) * 4;
  const float* rec =
      part + ((size_t)blockIdx.x * KS * H + h) * (DV + AF_HEAD);
  const size_t step = (size_t)H * (DV + AF_HEAD);
  float2 ml[AF_KS];
#pragma unroll
  for (int s = 0; s < AF_KS; ++s)
    ml[s] = s < KS ? *(const float2*)(rec + s * step)
                   : make_float2(PS_NEG_INF, 0.f);
  const int count = counted ? (int)rec[2] : KS;
  if (counted && count == 1) return;
  float mh = PS_NEG_INF;
#pragma unroll
  for (int s = 0; s < AF_KS; ++s) {
    if (s >= count) ml[s].y = 0.f;
    if (ml[s].y != 0.f) mh = fmaxf(mh, ml[s].x);
  }
  float l = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < AF_KS; ++s) {
    if (ml[s].y == 0.f) continue;
    const float4 v = *(const float4*)(rec + s * step + AF_HEAD + d);
    const float d = ml[s].x - mh;
    const float f = counted ? __builtin_amdgcn_exp2f(d) : expf(d);
    l += ml[s].y * f;
    o[0] += v.x * f;
    o[1] += v.y * f;
    o[2] += v.z * f;
    o[3] += v.w * f;
  }
  const float f = 1.0f / l;
  T* dst = out + (size_t)blockIdx.x * ldout + h * DV + d;
#pragma unroll
  for (int e = 0; e < 4; ++e) MxElem<T>::st(dst + e, o[e] * f);
}

// Merge pass over records [T, KS, H, DV + 4] (DV in steps of 4, KS up to 16).
extern "C" void mx_attn_records(void* out, int ldout, const void* part, int T_,
                                int H, int DV, int KS, int counted,
                                int dtype, void* stream) {
  MX_DISPATCH_DTYPE(dtype, {
    hipLaunchKernelGGL((attn_records_kernel<T>),
                       dim3(T_, (H * (DV / 4) + 255) / 256), dim3(256), 0,
                       (hipStream_t)stream, (T*)out, ldout, (const float*)part,
                       H, DV, KS, counted);
  })
}

template <int NT, int NV, int NC, bool CAP>
static int af_launch(const AfArgs& a, hipStream_t stream) {
  const size_t lds = (size_t)4 * 16 * NC * (NV * 64 + 4) * 4;
  if (hipFuncSetAttribute((const void*)attn_f32_kernel<NT, NV, NC, CAP>,
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  const unsigned tiles = (a.T + a.tpt - 1) / a.tpt;
  hipLaunchKernelGGL((attn_f32_kernel<NT, NV, NC, CAP>),
                     dim3(tiles * a.KS * a.G), dim3(256), lds, stream, a);
  return 0;
}

// Returns 0 when launched, 1 when the shape is outside this kernel: up to 16 heads
// a KV head, key widths in steps of 16 and value widths in steps of 4 up to 128,
// rows on 16-byte borders. token: single tokens (every batch row on its own), else
// prompt portions. scratch fp32 [T, splits, H, DV + 4] when splits > 1; rows:
// columns of a workgroup, 16 or 32 (single tokens and widths up to 64: 16).
extern "C" int mx_attn_f32(void* out, int ldout, const void* q, int ldq,
                           const void* kc, const void* vc,
                           const void* block_tables, int max_blocks,
                           const void* token_seq, const void* token_pos,
                           int T_, int H, int G, int D, int DV, int BS,
                           float scale, int chunk, int window, int sink,
                           int keep_first, float softcap,
                           const void* sink_vals, int vrow, int token,
                           int rows, int splits, void* scratch,
                           void* stream) {
  if (T_ <= 0) return 0;
  if (splits > AF_KS) return 1;
  if (G < 1 || H < 1 || H % G || H / G > 16 || BS < 1 || D < 16 || D % 16 ||
      D > 128 || DV < 4 || DV % 4 || DV > 128 || ldq % 4 || vrow % 4 ||
      vrow < DV || (((size_t)q | (size_t)kc | (size_t)vc) & 15))
    return 1;
  const bool wide = rows == 32 && !token && (D > 64 || DV > 64);
  AfArgs a = {(float*)out, ldout, (const float*)q, ldq, (const float*)kc,
              (const float*)vc, vrow, (const int*)block_tables, max_blocks,
              (const int*)token_seq, (const int*)token_pos, T_, H, G, D, DV,
              BS, scale, softcap, chunk, window,
              keep_first > 0 && (window > 0 || chunk > 0) ? keep_first : 0,
              sink, (const float*)sink_vals, !token,
              token ? 1 : (wide ? 32 : 16) / (H / G),
              splits > 1 && scratch != nullptr ? splits : 1, (float*)scratch};
  hipStream_t s = (hipStream_t)stream;
  int rc;
#define AF_GO(NT, NV, NC)                                    \
  rc = softcap > 0.f ? af_launch<NT, NV, NC, true>(a, s) \
                     : af_launch<NT, NV, NC, false>(a, s)
  if (D <= 64 && DV <= 64)
    AF_GO(4, 1, 1);
  else if (wide)
    AF_GO(8, 2, 2);
  else
    AF_GO(8, 2, 1);
#undef AF_GO
  if (rc == 0 && a.KS > 1)
    mx_attn_records(out, ldout, scratch, T_, H, DV, a.KS, 0, MX_F32, stream);
  return rc;
}
