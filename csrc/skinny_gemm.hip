// Skinny-batch GEMM for decode steps: out[M, N] = x[M, K] @ W[N, K]^T,
// bf16 inputs, fp32 accumulation, M <= 256.
//
// Why it exists: the library's tiles for the products of a decode batch leave
// the read of W, which bounds them, at a third to a half of the rate that memory
// gives. Up to 16 rows go without splits (x in LDS where it fits, also with the
// norm before and the activation or rotary embedding behind the products); more
// go by the tiled form, or by the short form where a workgroup's range of K is
// short or the tiles leave CUs waiting. Figures stand at each.
// mfma_f32_16x16x32_bf16; operand k-pattern as verified in
// csrc/tools/mfma_probe.hip.
#include "ps_common.h"
#include <algorithm>

typedef __attribute__((ext_vector_type(8))) __bf16 ps_gbf16x8;
typedef __attribute__((ext_vector_type(4))) float ps_gf32x4;

// Waves of skinny_lds_kernel, and the most entries of x that it takes: with the
// norm (their fp32 values stay in registers between its two passes) and without.
#define SL_WAVES 16
#define SL_NORM_X 16384
#define SL_X 65536

PS_DEV ps_gbf16x8 ps_as_gbf16(ps_bf16x8 u) {
  union {
    ps_bf16x8 u16;
    ps_gbf16x8 bf;
  } v;
  v.u16 = u;
  return v.bf;
}

// Up to 16 rows of x: a workgroup owns 16 rows of W and all of K, its NW waves
// take every NW-th 128-byte piece of them, UC pieces in flight each, and add up in
// LDS at the end: no second kernel and no partial sums in memory. W and x go
// straight into operands; what lies past the last row of x or the last piece reads
// as zero without an access (W's last piece again instead: 4096 x 4096 10.8 us, 8.7
// so). Bound by the read of W, at few rows of W by its latency. Reading x costs as
// many load instructions as reading W: where x fits in LDS and W is more than a
// few MB the form below takes over.
// GATED: W holds N / 2 gate rows, then as many up rows; a workgroup takes eight
// of each and writes silu(gate) up, both rounded to bf16 first: [M, N / 2].
// HALF: eight rows of W a workgroup, two pieces of each at a time. Left rows 8 to
// 15 are the second piece of rows 0 to 7, right columns 8 to 15 that piece of up
// to eight rows of x; the two diagonal blocks of the product add up, the others
// are nothing. Where 16 rows a workgroup leave half of the CUs without one (us at
// one row, 16 rows / 8 / the library: 2048 x 2048 5.4 / 4.5 / 11.0, 2048 x 8192
// 12.0 / 8.6 / 12.7, 1024 x 4096 7.4 / 5.4 / 14.4).
// FAR: W by its addresses, where 31-bit offsets do not reach a tile's last row or
// it is not aligned to 16 bytes.
template <int UC, int NW, bool GATED, bool HALF, bool FAR>
__global__ __launch_bounds__(NW * 64) void skinny_rows_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, int M, int N, int K, int x_stride) {
  constexpr int PN = 20;  // pitch of a row of sums
  __shared__ __align__(16) float s_sum[NW][16 * PN];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rc = lane & 15, g = lane >> 4;
  constexpr int PC = HALF ? 128 : 64;  // columns of a step
  // rows of W, columns of the result
  constexpr int NR = HALF ? 8 : 16, NO = GATED ? NR / 2 : NR;
  const int n0 = blockIdx.x * NO;
  const int nc = K / PC;  // steps
  const int r8 = HALF ? rc & 7 : rc;
  const int k0 = g * 8 + (HALF ? (rc >> 3) * 64 : 0);
  const int wrow = r8 >= NO ? N / 2 + r8 - NO : r8;
  const unsigned short* wp = w + (long)(n0 + wrow) * K + k0;
  // what lies past the end reads as zero without an access
  const unsigned int off = 0x80000000u;
  const auto wr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(w + (long)n0 * K), 0, (int)off - 1, 0x00020000);
  const auto xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)x, 0, ((M - 1) * x_stride + K) * 2, 0x00020000);
  const unsigned int wo = (unsigned int)(wrow * K + k0) * 2;
  const unsigned int xo =
      r8 < M ? (unsigned int)(r8 * x_stride + k0) * 2 : off;
  ps_gf32x4 acc = {0.f, 0.f, 0.f, 0.f};
  ps_gbf16x8 wf[UC][2], xf[UC][2];
  auto load = [&](int u, int c) {
    const unsigned int o = c < nc ? 0u : off;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned int k = c * (2 * PC) + 64 * h;
      if constexpr (FAR)
        wf[u][h] =
            *(const ps_gbf16x8*)(wp + min(c, nc - 1) * PC + 32 * h);
      else
        wf[u][h] = __builtin_bit_cast(
            ps_gbf16x8,
            __builtin_amdgcn_raw_buffer_load_b128(wr, wo | o, k, 0));
      xf[u][h] = __builtin_bit_cast(
          ps_gbf16x8,
          __builtin_amdgcn_raw_buffer_load_b128(xr, xo | o, k, 0));
    }
  };
  const int w0 = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
  for (int u = 0; u < UC; ++u) load(u, w0 + NW * u);
  for (int c = w0; c < nc; c += NW * UC) {
#pragma unroll
    for (int u = 0; u < UC; ++u) {
      if (!FAR || c + NW * u < nc) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][h], xf[u][h],
                                                        acc, 0, 0, 0);
      }
      load(u, c + NW * (UC + u));
    }
  }
  // acc[r]: row rc of x, row n0 + 4 g + r of W
  *(ps_gf32x4*)(&s_sum[wave][rc * PN + 4 * g]) = acc;
  __syncthreads();
  if (tid < 64) {
    const int m = tid >> 2, n = (tid & 3) * 4;
    ps_gf32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NW; ++k)
      v += *(const ps_gf32x4*)(&s_sum[k][m * PN + n]);
    if constexpr (HALF) {
#pragma unroll
      for (int k = 0; k < NW; ++k)
        v += *(const ps_gf32x4*)(
            &s_sum[k][((m & 7) + 8) * PN + (n & 7) + 8]);
    }
    if constexpr (GATED) {
      // the quad of up columns is NO / 4 lanes on
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float gv = ps_bf16_to_f32(ps_f32_to_bf16(v[r]));
        const float uv = ps_bf16_to_f32(
            ps_f32_to_bf16(__shfl_down(v[r], NO / 4, 64)));
        v[r] = gv / (1.f + __expf(-gv)) * uv;
      }
    }
    if (m < M && n < NO)
      *(uint2*)(out + (long)m * (GATED ? N / 2 : N) + n0 + n) = make_uint2(
          (unsigned int)ps_f32_to_bf16(v[0]) |
              ((unsigned int)ps_f32_to_bf16(v[1]) << 16),
          (unsigned int)ps_f32_to_bf16(v[2]) |
              ((unsigned int)ps_f32_to_bf16(v[3]) << 16));
  }
}

// What skinny_lds_kernel reads and writes.
struct SlArgs {
  unsigned short* out;      // [M, N]; gated [M, N / 2]
  unsigned short* res_out;  // [M, K] = x + res, where there is a res
  const unsigned short *x, *res, *nw, *w;  // [M, K], [M, K], [K], [N, K]
  int M, N, K;
  int apart;                // rows between the two halves of a tile
  long x_stride;            // K with the norm
  float eps;
  // rotary form
  const int* positions;     // [M]
  const float* cos_sin;     // [.., HD]
  const long* slots;        // [M]
  void *kc, *vc;            // [blocks, KH, BS, HD]
  int QH, KH, HD, BS;
};

// Up to 16 rows of x that LDS holds, with what stands around the products that
// begin a layer's two halves:
//   NORM      x <- x + res,  y = x rsqrt(mean x^2 + eps) nw; else y = x
//             out = y W^T, then
//   SL_GATED  silu(gate) up
//   SL_ROPE   the rotary embedding of queries and keys, and keys and values into
//             the paged cache; W's rows are query heads, key heads, value heads
// A workgroup a CU reads (and normalises) all of x for itself while its first
// pieces of W are on their way, and walks tiles of 16 rows of W, every
// gridDim.x-th; its waves take every NW-th 128-byte piece of a tile, UC pieces in
// flight each across the tiles' ends. x costs a read from the caches a CU instead
// of one a tile, the norm and the rotary embedding no launches of their own
// (3.5 us each and up). The waves' sums of a tile are added by one of them while
// the others go on. Roundings are those of the separate kernels; x + res goes to
// a buffer of its own, since other workgroups still read res.
// Bound by the read of W. us, distinct weights, with the launches it replaces:
//   norm, 28672 x 4096, silu   1 row 41.3 (before 47.4), 4 rows 43.9 (50.1)
//   norm, 16384 x 2048, silu   1 row 14.1 (17.9), 8 rows 16.8 (20.1)
//   norm, 6144 x 4096, rotary  1 row 14.5 (20.6), 4 rows 16.7 (20.6)
//   norm, 3072 x 2048, rotary  1 row 6.9 (11.1), 8 rows 9.3 (12.4)
//   28672 x 4096, silu         8 rows 42.6 (52.1), 16 rows 44.9 (60.8; 5.3 TB/s)
//   6144 x 4096                8 rows 13.2 (15.0), 16 rows 14.4 (18.1)
// More workgroups a CU read and normalise x more often (28672 x 4096 with the norm,
// one row 41.3, two 40.7, four rows 43.9 and 46.1, all tiles at once 63), fewer
// pieces in flight do not cover a tile's end (one 42.3, four 42.0 at one row).
enum { SL_PLAIN, SL_GATED, SL_ROPE };
template <int EPI, bool NORM, typename KVT>
__global__ __launch_bounds__(SL_WAVES * 64) void skinny_lds_kernel(SlArgs a) {
  constexpr int UC = 2, NW = SL_WAVES;
  constexpr int PN = 20;  // pitch of a row of sums
  constexpr int NT = NW * 64;
  constexpr int VECS = NORM ? SL_NORM_X / 8 : SL_X / 8;
  constexpr int VP = VECS / NT;  // 16-byte pieces of x a thread has
  // sums of a tile: with two sets a tile has one barrier, if there is room
  constexpr int SETS = NORM ? 2 : 1;
  __shared__ __align__(16) float s_sum[SETS][NW][16 * PN];
  __shared__ float s_part[NORM ? VECS / 8 : 1], s_inv[16];
  __shared__ __align__(16) unsigned short s_x[VECS * 8 + 128];  // [M][K + 8]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rc = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, K = a.K, V = K / 8, total = M * V;

  // x first: loads land in the order in which they were asked for
  ps_bf16x8 xv[VP], rv[VP], nv[VP];
  int at[VP];  // where a piece goes in s_x
#pragma unroll
  for (int u = 0; u < VP; ++u) {
    const int i = u * NT + tid;
    if (i < total) {
      const int m = i / V;
      at[u] = i * 8 + m * 8;
      if constexpr (NORM) {
        xv[u] = *(const ps_bf16x8*)(a.x + i * 8);
        if (a.res) rv[u] = *(const ps_bf16x8*)(a.res + i * 8);
        nv[u] = *(const ps_bf16x8*)(a.nw + (i - m * V) * 8);
      } else {
        xv[u] = *(const ps_bf16x8*)(a.x + (long)m * a.x_stride +
                                    (i - m * V) * 8);
      }
    }
  }
  const int om = lane >> 2, on = (lane & 3) * 4;  // of the last step
  int pos = 0;
  long slot = -1;
  if constexpr (EPI == SL_ROPE) {
    if (om < M) {
      pos = a.positions[om];
      slot = a.slots[om];
    }
  }
  // a tile's rows of W: eight, and the eight that belong to them
  const int nc = K / 64;  // pieces of a row
  const int steps = (nc + NW - 1) / NW;
  const int per = EPI == SL_ROPE ? a.HD / 16 : 1;
  const int tiles = N / 16;
  const int apart = a.apart;
  auto row0 = [&](int tile) {
    return EPI == SL_ROPE ? tile / per * a.HD + tile % per * 8
                          : tile * (apart == 8 ? 16 : 8);
  };
  // what lies past the end reads as zero without an access
  const unsigned int off = 0x80000000u;
  const unsigned int wo =
      (unsigned int)(((rc & 7) + (rc >> 3) * apart) * K + g * 8) * 2;
  ps_gbf16x8 wf[UC][2];
  int lt = blockIdx.x, lj = 0;  // the next step to ask for
  auto load = [&](int u) {
    const int c = wave + NW * lj;
    const unsigned int o = c < nc && lt < tiles ? 0u : off;
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.w + (long)row0(min(lt, tiles - 1)) * K), 0, (int)off - 1,
        0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      wf[u][h] = __builtin_bit_cast(
          ps_gbf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                          wr, wo | o, c * 128 + 64 * h, 0));
    if (++lj == steps) lj = 0, lt += gridDim.x;
  };
#pragma unroll
  for (int u = 0; u < UC; ++u) load(u);
  __builtin_amdgcn_sched_barrier(0);

  if constexpr (!NORM) {
#pragma unroll
    for (int u = 0; u < VP; ++u)
      if (u * NT + tid < total) *(ps_bf16x8*)(s_x + at[u]) = xv[u];
  } else {
    float f[VP][8];
#pragma unroll
    for (int u = 0; u < VP; ++u) {
      const int i = u * NT + tid;
      float ss = 0.f;
      if (i < total) {
        ps_bf16x8 sv;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float y = ps_bf16_to_f32(xv[u][j]);
          if (a.res) y += ps_bf16_to_f32(rv[u][j]);
          f[u][j] = y;
          ss += y * y;
          sv[j] = ps_f32_to_bf16(y);
        }
        if (a.res && blockIdx.x == 0) *(ps_bf16x8*)(a.res_out + i * 8) = sv;
      }
      // eight lanes have 64 columns of one row
#pragma unroll
      for (int d = 1; d < 8; d <<= 1) ss += __shfl_xor(ss, d, 64);
      if ((lane & 7) == 0 && i < total) s_part[i / 8] = ss;
    }
    __syncthreads();
    for (int m = wave; m < M; m += NW) {
      float t = 0.f;
      for (int i = lane; i < nc; i += 64) t += s_part[m * nc + i];
      t = ps_group_sum<64>(t);
      if (lane == 0) s_inv[m] = rsqrtf(t / (float)K + a.eps);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < VP; ++u) {
      const int i = u * NT + tid;
      if (i < total) {
        const float inv = s_inv[i / V];
        ps_bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o[j] = ps_f32_to_bf16(f[u][j] * inv * ps_bf16_to_f32(nv[u][j]));
        *(ps_bf16x8*)(s_x + at[u]) = o;
      }
    }
  }
  // a tile's angles, on their way during its products
  ps_gf32x4 cs = {1.f, 1.f, 1.f, 1.f}, sn = {0.f, 0.f, 0.f, 0.f};
  auto angles = [&](int tile) {
    if constexpr (EPI == SL_ROPE) {
      if (om < M && tile / per < a.QH + a.KH) {
        const float* c =
            a.cos_sin + (long)pos * a.HD + tile % per * 8 + (on & 7);
        cs = *(const ps_gf32x4*)c;
        sn = *(const ps_gf32x4*)(c + a.HD / 2);
      }
    }
  };
  angles(blockIdx.x);
  __syncthreads();

  // rows past the last repeat it: their results are left out
  const unsigned short* xp = s_x + min(rc, M - 1) * (K + 8) + g * 8;
  ps_gf32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int tile = blockIdx.x, j = 0, set = 0, turn = 0;
  // The sums of a tile. acc[r]: row rc of x, row 4 g + r of the tile's.
  auto finish = [&] {
    if (SETS == 1 && tile != (int)blockIdx.x) __syncthreads();
    *(ps_gf32x4*)(&s_sum[set][wave][rc * PN + 4 * g]) = acc;
    __syncthreads();
    if (wave != turn) return;
    ps_gf32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NW; ++k)
      v += *(const ps_gf32x4*)(&s_sum[set][k][om * PN + on]);
    ps_gf32x4 z;  // the eight that belong to these
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = ps_bf16_to_f32(ps_f32_to_bf16(v[r]));
      z[r] = __shfl_xor(v[r], 2, 64);
    }
    const int head = tile / per;
    if constexpr (EPI == SL_GATED) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = v[r] / (1.f + __expf(-v[r])) * z[r];
    } else if constexpr (EPI == SL_ROPE) {
      if (head < a.QH + a.KH) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = on < 8 ? v[r] * cs[r] - z[r] * sn[r]
                        : v[r] * cs[r] + z[r] * sn[r];
      }
    }
    if (om >= M || (EPI == SL_GATED && on >= 8)) return;
    unsigned short e[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) e[r] = ps_f32_to_bf16(v[r]);
    const int col = row0(tile) + (on < 8 ? on : apart + on - 8);
    *(uint2*)(a.out + (long)om * (EPI == SL_GATED ? N / 2 : N) + col) =
        make_uint2((unsigned int)e[0] | ((unsigned int)e[1] << 16),
                   (unsigned int)e[2] | ((unsigned int)e[3] << 16));
    if constexpr (EPI == SL_ROPE) {
      const int h = head - a.QH;
      if (h < 0 || slot < 0) return;
      const bool isv = h >= a.KH;
      typename ps_kv_traits<KVT>::vec4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = ps_kv_traits<KVT>::from_f32(ps_bf16_to_f32(e[r]));
      const long row =
          (slot / a.BS * a.KH + (isv ? h - a.KH : h)) * a.BS + slot % a.BS;
      *(typename ps_kv_traits<KVT>::vec4*)((KVT*)(isv ? a.vc : a.kc) +
                                           row * a.HD + col - head * a.HD) = o;
    }
  };
  while (tile < tiles) {
#pragma unroll
    for (int u = 0; u < UC; ++u) {
      if (tile >= tiles) break;
      const int c = wave + NW * j;
      if (c < nc) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[u][h], *(const ps_gbf16x8*)(xp + c * 64 + 32 * h), acc, 0, 0,
              0);
      }
      load(u);
      if (++j == steps) {
        finish();
        acc = {0.f, 0.f, 0.f, 0.f};
        j = 0;
        tile += gridDim.x;
        set ^= SETS - 1;
        turn = turn + 1 == NW ? 0 : turn + 1;
        if (tile < tiles) angles(tile);
      }
    }
  }
}

// The short form: a workgroup owns 64 rows of W, all rows of x and a range of K,
// in steps of 64 columns: x passes through LDS between two barriers, W goes from
// memory straight into right operands. Nothing is ahead, so a step costs its
// latency, but there is nothing to fill either, and up to eight workgroups a CU
// hide one another: 17 rows of 2048 x 64 3.2 us (tiles 5.7), 17 rows of
// 128256 x 256 16 (25), 24 rows of 102400 x 4096 161 (175).
template <int M_TILES>
__global__ __launch_bounds__(256, 4) void skinny_gemm_kernel(
    unsigned short* __restrict__ out_bf16,  // [M, N] (splits == 1)
    float* __restrict__ ws,                 // [S, M, N] (splits > 1)
    const unsigned short* __restrict__ x,   // [M, K]
    const unsigned short* __restrict__ w,   // [N, K]
    int M, int N, int K, long x_stride /* row stride of x, elems */) {
  constexpr int MP = M_TILES * 16;  // padded M
  const int n0 = blockIdx.x * 64;
  const int splits = gridDim.y;
  const int kchunks = K / 64;
  const int per_split = (kchunks + splits - 1) / splits;
  const int kc_begin = blockIdx.y * per_split;
  const int kc_end = min(kchunks, kc_begin + per_split);
  if (kc_begin >= kc_end) return;

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int rc = lane & 15;
  const int nrow = n0 + wave * 16 + rc;  // this lane's W row (B col)

  // x chunk [MP][64] staged with 16-B slot XOR swizzle (slot ^= row&7)
  __shared__ __align__(16) unsigned short x_lds[MP][64];

  ps_gf32x4 acc[M_TILES];
#pragma unroll
  for (int mt = 0; mt < M_TILES; mt++) acc[mt] = {0.f, 0.f, 0.f, 0.f};

  for (int kc = kc_begin; kc < kc_end; kc++) {
    // ---- cooperative x staging: MP*8 16-B slots over 256 threads ----
    for (int u = tid; u < MP * 8; u += 256) {
      const int row = u >> 3;
      const int slot = u & 7;
      ps_bf16x8 v = {};
      if (row < M)
        v = *(const ps_bf16x8*)(x + (long)row * x_stride + kc * 64 +
                                slot * 8);
      *(ps_bf16x8*)(&x_lds[row][(slot ^ (row & 7)) * 8]) = v;
    }
    __syncthreads();
    // ---- B-frags: W rows streamed once ----
    const unsigned short* wr = w + (long)nrow * K + kc * 64;
    ps_gbf16x8 b0 = ps_as_gbf16(*(const ps_bf16x8*)(wr + g * 8));
    ps_gbf16x8 b1 = ps_as_gbf16(*(const ps_bf16x8*)(wr + 32 + g * 8));
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int mt = 0; mt < M_TILES; mt++) {
      const int row = mt * 16 + rc;
      ps_gbf16x8 a0 = ps_as_gbf16(
          *(const ps_bf16x8*)(&x_lds[row][(g ^ (row & 7)) * 8]));
      ps_gbf16x8 a1 = ps_as_gbf16(
          *(const ps_bf16x8*)(&x_lds[row][((4 + g) ^ (row & 7)) * 8]));
      acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc[mt],
                                                        0, 0, 0);
      acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc[mt],
                                                        0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
  }

  // ---- epilogue (C layout: row=(g*4+r), col=rc of each 16x16 tile).
  // splits==1 writes bf16 output directly; otherwise each split streams
  // its fp32 partial to ws[split][M][N] and a combine kernel reduces —
  // device atomicAdd RMW traffic (M*N*splits) was the measured 1/M
  // throughput wall of the earlier design.
#pragma unroll
  for (int mt = 0; mt < M_TILES; mt++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = mt * 16 + g * 4 + r;
      if (m >= M) continue;
      if (gridDim.y == 1) {
        out_bf16[(long)m * N + nrow] = ps_f32_to_bf16(acc[mt][r]);
      } else {
        ws[((long)blockIdx.y * M + m) * N + nrow] = acc[mt][r];
      }
    }
  }
}

// The tiled form, for 17 to 256 rows of x (and 9 to 16 of a W of more than 32768
// where LDS has no room for x): a workgroup owns 64 NC rows of W, all rows of x and a range of K, in
// steps of 128 columns. x passes through LDS, two steps' buffers with one barrier
// a step; W goes from memory straight into left operands, WD steps ahead. The
// eight waves are four by rows of W times two by halves of a step, which add up in
// LDS at the end. Partial sums of the ranges go to memory and are added by
// skinny_combine.
//
// Bound by the read of W while a range is long enough to hide its start, and by
// the reads of x from LDS with many rows (each wave reads all of x: 16 NC rows of
// W share a read). us, distinct weights, this / the short form / the library's
// kernel:
//   4096 x 14336   64 rows 32 / 48 / 40, 128 rows 39 / 65 / 74, 192 45 / 82 / 101
//   4096 x 4096    64 rows 16 / 22 / 14, 192 rows 24 / 40 / 31
//   28672 x 4096   64 rows 51 / 96 / 53, 192 rows 71 / 150 / 62
//   2048 x 8192    64 rows 17 / 25 / 21, 192 rows 25 / 40 / 25
// Waves split by rows of x as well read W twice: 10 to 40 % slower.
// GATED (one range): W holds N / 2 gate rows, then as many up rows; 16 rows of a
// tile are eight of each, which are two lane groups apart, and out [M, N / 2] is
// silu(gate) up, both rounded to bf16 first.
template <int MT, int NC, bool GATED>
__global__ __launch_bounds__(512, MT* NC <= 8 ? 4 : 2) void skinny_tile_kernel(
    unsigned short* __restrict__ out,      // [M, N] (one split)
    float* __restrict__ ws,                // [splits, M, N]
    const unsigned short* __restrict__ x,  // [M, K], rows x_stride apart
    const unsigned short* __restrict__ w,  // [N, K]
    int M, int N, int K, long x_stride, int splits) {
  constexpr int BN = 64 * NC;
  constexpr int WD = NC == 1 ? 4 : 3;       // steps of W in flight
  constexpr int XL = (MT + 1) / 2;          // pieces of x a thread stages
  constexpr int XB = (MT + MT % 2) * 2048;  // entries of one buffer
  constexpr int PN = BN + 4;                // pitch of a row of sums
  // sums in two halves of the rows where all are more than the buffers
  constexpr int MH = MT * 32 * PN > 2 * XB && MT > 1 ? MT / 2 : MT;
  constexpr int LDS = MH * 32 * PN > 2 * XB ? MH * 32 * PN : 2 * XB;
  __shared__ __align__(16) unsigned short lds[LDS];
  // the ranges of one tile side by side: an XCD reads few ranges of x
  const int split = blockIdx.x % splits, n0 = blockIdx.x / splits * BN;
  const int chunks = K / 64, per = (chunks + splits - 1) / splits;
  const int c0 = split * per, c1 = min(chunks, c0 + per);
  const int steps = (c1 - c0 + 1) / 2;
  // Every tile begins at another step of its range: rows of W a power of two
  // apart, read at the same columns by all workgroups, come from few channels of
  // memory. us, all at the first step / this / the short form: 17 rows of
  // 128256 x 4096 226 / 184 / 187, 128256 x 2048 116 / 102 / 129, 102400 x 8192
  // 419 / 333 / 311; 24 rows of 28672 x 4096 57 / 47 / 73, 4096 x 4096 12.8 / 13.6 /
  // 17.4.
  const int tile = blockIdx.x / splits;
  const int turn = steps > 0 ? (tile + tile / 8) % steps : 0;
  auto place = [&](int t) {
    const int s = min(t, steps - 1) + turn;
    return max(s >= steps ? s - steps : s, 0);
  };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave >> 2, wn = wave & 3;  // half of a step, rows of W
  const int rc = lane & 15, g = lane >> 4;

  const unsigned short* wp[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int row = n0 + (wn * NC + c) * 16;
    wp[c] = w + g * 8 +
            (long)(!GATED   ? row + rc
                   : rc < 8 ? row / 2 + rc
                            : (N + row) / 2 + rc - 8) *
                K;
  }
  ps_gbf16x8 wf[WD][NC][2];
  // steps past the end repeat the last chunk and are not multiplied
  auto load_w = [&](int u, int t) {
    const int k = min(c0 + 2 * place(t) + kg, c1 - 1) * 64;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wf[u][c][h] = *(const ps_gbf16x8*)(wp[c] + k + 32 * h);
  };
  // x: a thread takes one of a row's 16 slots of 16 bytes in XL rows, swizzled
  // by the row so that reads of 16 rows spread over the banks
  const int xs = tid & 15;
  ps_bf16x8 xf[2][XL];
  const unsigned short* xp[XL];
  int xd[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int row = i * 32 + (tid >> 4);
    xp[i] = x + (long)min(row, M - 1) * x_stride;
    xd[i] = row * 128 + (xs ^ (row & 7)) * 8;
  }
  auto load_x = [&](int u, int t) {
    const int k =
        min(c0 + 2 * place(t) + (xs >> 3), c1 - 1) * 64 + (xs & 7) * 8;
#pragma unroll
    for (int i = 0; i < XL; ++i) xf[u][i] = *(const ps_bf16x8*)(xp[i] + k);
  };
  auto put_x = [&](int u) {
#pragma unroll
    for (int i = 0; i < XL; ++i)
      *(ps_bf16x8*)(lds + u * XB + xd[i]) = xf[u][i];
  };
  ps_gf32x4 acc[NC][MT];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[c][i] = {0.f, 0.f, 0.f, 0.f};
  load_x(0, 0);
#pragma unroll
  for (int u = 0; u < WD; ++u) load_w(u, u);
  load_x(1, 1);
  put_x(0);
  load_x(0, 2);
  __syncthreads();
  const int xr0 = rc * 128 + ((kg * 8 + g) ^ (rc & 7)) * 8;
  const int xr1 = rc * 128 + ((kg * 8 + 4 + g) ^ (rc & 7)) * 8;
  constexpr int UN = WD % 2 == 0 ? WD : 2 * WD;
  for (int t = 0; t < steps; t += UN) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (t + u < steps) {
        const unsigned short* buf = lds + (u & 1) * XB;
        // the other buffer was read before the last barrier
        put_x((u + 1) & 1);
        load_x((u + 1) & 1, t + u + 3);
        if (c0 + 2 * place(t + u) + kg < c1) {
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            const ps_gbf16x8 b0 = *(const ps_gbf16x8*)(buf + i * 2048 + xr0);
            const ps_gbf16x8 b1 = *(const ps_gbf16x8*)(buf + i * 2048 + xr1);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
              acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  wf[u % WD][c][0], b0, acc[c][i], 0, 0, 0);
              acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  wf[u % WD][c][1], b1, acc[c][i], 0, 0, 0);
            }
          }
        }
        load_w(u % WD, t + u + WD);
        __syncthreads();
      }
    }
  }
  // acc[c][i][r]: row 16 i + rc of x, row n0 + (wn NC + c) 16 + 4 g + r of W
  float* sum = (float*)lds;
#pragma unroll
  for (int h = 0; h < MT; h += MH) {
    if (h > 0) __syncthreads();
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < MH; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          *(ps_gf32x4*)(sum + (i * 16 + rc) * PN + (wn * NC + c) * 16 +
                        4 * g) = acc[c][h + i];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int i = 0; i < MH; ++i) {
        const int m = (h + i) * 16 + rc;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int n = (wn * NC + c) * 16 + 4 * g;
          const ps_gf32x4 v =
              acc[c][h + i] +
              *(const ps_gf32x4*)(sum + (i * 16 + rc) * PN + n);
          if constexpr (GATED) {
            unsigned short e[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float gv = ps_bf16_to_f32(ps_f32_to_bf16(v[r]));
              const float uv = ps_bf16_to_f32(
                  ps_f32_to_bf16(__shfl_xor(v[r], 32, 64)));
              e[r] = ps_f32_to_bf16(gv / (1.f + __expf(-gv)) * uv);
            }
            if (m < M && g < 2)
              *(uint2*)(out + (long)m * (N / 2) +
                        (n0 + (wn * NC + c) * 16) / 2 + 4 * g) =
                  make_uint2((unsigned int)e[0] | ((unsigned int)e[1] << 16),
                             (unsigned int)e[2] | ((unsigned int)e[3] << 16));
            continue;
          }
          if (m >= M) continue;
          if (splits > 1)
            *(ps_gf32x4*)(ws + ((long)split * M + m) * N + n0 + n) = v;
          else
            *(uint2*)(out + (long)m * N + n0 + n) = make_uint2(
                (unsigned int)ps_f32_to_bf16(v[0]) |
                    ((unsigned int)ps_f32_to_bf16(v[1]) << 16),
                (unsigned int)ps_f32_to_bf16(v[2]) |
                    ((unsigned int)ps_f32_to_bf16(v[3]) << 16));
        }
      }
    }
  }
}

__global__ __launch_bounds__(256) void skinny_combine_kernel(
    unsigned short* __restrict__ out,  // [M, N] bf16
    const float* __restrict__ ws,      // [S, M, N] fp32
    long MN, int splits) {             // MN: a multiple of 64
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  ps_gf32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < splits; s++)
    a += *(const ps_gf32x4*)(ws + (long)s * MN + i);
  *(uint2*)(out + i) =
      make_uint2((unsigned int)ps_f32_to_bf16(a[0]) |
                     ((unsigned int)ps_f32_to_bf16(a[1]) << 16),
                 (unsigned int)ps_f32_to_bf16(a[2]) |
                     ((unsigned int)ps_f32_to_bf16(a[3]) << 16));
}

enum PsSkinnyForm { PS_NARROW, PS_WIDE, PS_SHORT };
struct PsSkinnyPlan {
  PsSkinnyForm form;
  int splits;
};

// Where the short form is the faster one. us, short / tiles:
// Few sums (up to 32768 rows of W): the tiles' ranges have four chunks at least
// and start with three or four steps of loads; the more sums, the more the short
// form pays for its splits. 17 x 512 x 1024 6.1 / 7.7, 17 x 512 x 2048 7.7 / 8.1,
// 64 x 1024 x 1024 8.7 / 8.8, 64 x 1024 x 1536 10.6 / 9.7, 32 x 4096 x 704 11.2 / 9.3,
// 64 x 4096 x 768 13.4 / 10.6.
// A W of more: no splits in either form. The tiles run in turns of the CUs, and
// what the busiest CU has beyond the mean, and the start of each turn, is the
// tiles' loss: the line follows the turns of wide tiles (up to one and a half,
// two, three, the first half of a fourth, all of it, more). 17 x 45056 x 512 15 / 17,
// x 1024 30 / 26; 17 x 78848 x 1536 54 / 57; 24 x 102400 x 4096 161 / 175; 24 x
// 128256 x 1536 84 / 90; 64 x 128256 x 1280 86 / 90; 128 x 128256 x 512 62 / 62;
// 192 x 95232 x 384 56 / 50; 256 x 61440 x 1024 81 / 85. Rows of 2048 columns come
// from few channels in the short form (17 x 128256 x 2048 129 / 102).
static bool ps_skinny_short(int M, int N, int K) {
  if (K < 128) return true;
  if (N <= 32768) {
    const long sums = (long)M * N;
    return K < (sums <= 32768    ? 2048
                : sums <= 65536  ? 1536
                : sums <= 131072 ? 640
                                 : 0);
  }
  static const int all = 1 << 30;
  static const int lines[5][6] = {{768, 896, 3264, all, 3648, 1088},
                                  {640, 640, 960, 2624, 1344, 704},
                                  {768, 640, 896, 1600, 640, 768},
                                  {512, 512, 384, 512, 512, 448},
                                  {768, 1088, 576, 1024, 1344, 896}};
  const int rows = M <= 32 ? 0 : M <= 64 ? 1 : M <= 128 ? 2 : M <= 192 ? 3 : 4;
  const int turn = N <= 49152    ? 0
                   : N <= 65536  ? 1
                   : N <= 98304  ? 2
                   : N <= 114688 ? 3
                   : N <= 131072 ? 4
                                 : 5;
  if (K == 2048 && rows == 0 && turn != 3) return false;
  return K < lines[rows][turn];
}

// Tiles of 64 or 128 rows of W and the ranges of K: as many workgroups as there
// are CUs, or as few more as one wave of narrow tiles takes. A range has four
// chunks at least, or its start is most of it. Of the two widths the one that
// fills more CUs, if that takes no partial sums of short rows (17 x 10240 x 896:
// three ranges of wide tiles 12.5, one of narrow ones 9.2; x 2048 16.6 / 15.8, x
// 3072 20.2 / 22.8); at as many the wide one for long rows (its reads of x from LDS
// go to twice the products), the narrow one for short ones (its partial sums are
// half). us at 192 rows, narrow / wide: 6144 x 4096 32 (192 workgroups) / 29
// (240), 4096 x 4096 23 / 24, 4096 x 14336 48 / 43, 2560 x 10240 33 (200) / 33
// (160), 18944 x 3584 82 (296) / 58 (148), 16384 x 2048 30 / 37. Up to 32 rows of a
// wide W are bound by its read alone: the narrow one where its busiest CU has an
// eighth fewer rows (17 rows, narrow / wide: 49152 x 4096 75 / 89, 65664 x 8192 212 /
// 239; 57344 x 4096 with as many rows 98 / 90, 32 of 136192 x 5120 with a tenth fewer
// 329 / 316). Above 192 rows the wide tile's sums do not fit in the registers.
static PsSkinnyPlan ps_skinny_plan(int M, int N, int K) {
  const int chunks = K / 64;
  // whole ranges of ceil(chunks / s) chunks are handed out: count those that
  // are not empty, since an empty one would write no partial sums
  auto ranges = [&](int s, int most) {
    if (s > most) s = most;
    if (s < 1) s = 1;
    const int per = (chunks + s - 1) / s;
    return (chunks + per - 1) / per;
  };
  if (ps_skinny_short(M, N, K))
    return {PS_SHORT, ranges(1024 / (N / 64), chunks)};
  int splits[2], used[2], busiest[2];
  for (int wide = 0; wide < 2; ++wide) {
    const int tiles = wide ? (N + 127) / 128 : N / 64;
    splits[wide] = ranges(256 / tiles, chunks / 4);
    // workgroups past the CUs wait for a second turn
    used[wide] = tiles > 256 ? 128 : tiles * splits[wide];
    busiest[wide] = (tiles + 255) / 256 * (wide ? 128 : 64);
  }
  bool wide;
  if (N > 32768 && M <= 32)
    wide = busiest[0] * 8 > busiest[1] * 7;
  else
    wide = (used[1] > used[0] &&
            (splits[1] == 1 || K > (M <= 64 ? 2048 : 1536))) ||
           (used[1] == used[0] && (K >= 8192 || N > 32768));
  wide = wide && N % 128 == 0 && M <= 192;
  return {wide ? PS_WIDE : PS_NARROW, splits[wide]};
}

// Whether skinny_lds_kernel has room for x and offsets for a tile of W.
static bool ps_skinny_lds_fits(int M, int N, int K, long x_stride,
                               const void* x, const void* w, bool norm) {
  return M >= 1 && M <= 16 && (long)M * K <= (norm ? SL_NORM_X : SL_X) &&
         N >= 64 && N % 64 == 0 && K >= 64 && K % 64 == 0 &&
         (long)(N + 32) * K < 1L << 31 && x_stride % 8 == 0 &&
         (((size_t)x | (size_t)w) & 15) == 0;
}

template <int EPI, bool NORM, typename KVT = unsigned short>
static void ps_skinny_lds_go(const SlArgs& a, hipStream_t stream) {
  skinny_lds_kernel<EPI, NORM, KVT>
      <<<std::min(a.N / 16, 256), SL_WAVES * 64, 0, stream>>>(a);
}

// Whether a kernel without splits takes it: up to 8 rows, up to 16 where W has no
// more than 32768 rows or LDS has room for x. More rows reread x too often where
// the other form needs no splits (N > 32768; us, rows kernel / tiles, distinct
// weights: 16 x 128256 x 4096 283 / 183, 16 x 51200 x 2560 82 / 66).
static bool ps_skinny_rows(int M, int N, int K, long x_stride, const void* x,
                           const void* w) {
  return (M <= 8 || (M <= 16 && N <= 32768) ||
          ps_skinny_lds_fits(M, N, K, x_stride, x, w, false)) &&
         x_stride >= 0 && (M - 1) * x_stride + K < (1L << 30);
}

template <bool GATED>
static void ps_skinny_rows_go(void* out, const void* x, const void* w, int M,
                              int N, int K, long x_stride,
                              hipStream_t stream) {
#define PS_SR(UC, NW, HALF, FAR)                                            \
  skinny_rows_kernel<UC, NW, GATED, HALF, FAR>                              \
      <<<N / (HALF ? 8 : 16), NW * 64, 0, stream>>>(                        \
          (unsigned short*)out, (const unsigned short*)x,                   \
          (const unsigned short*)w, M, N, K, (int)x_stride)
  // offsets from a tile's first row reach 15 rows on, gated those N / 2 behind
  if (((size_t)w & 15) != 0 || (GATED ? N + 32L : 32L) * K >= 1L << 31) {
    PS_SR(1, 16, false, true);
    return;
  }
  // 16 rows a workgroup leave half of the CUs without one: eight
  if (M <= 8 && N <= 2048 && K % 128 == 0) {
    // us at one row, a step in flight / two: 2048 x 2048 4.5 / 4.5, 512 x 1024
    // 3.2 / 3.5, 2048 x 4096 6.4 / 5.8, 2048 x 14336 13.5 / 12.7
    if (K <= 2048)
      PS_SR(1, 8, true, false);
    else
      PS_SR(2, 8, true, false);
    return;
  }
  // Reading x into LDS first takes longer than a short read of W beside it (us at
  // one row and 16, from memory / from LDS: 4096 x 1024 4.1 / 4.5 and 4.6 / 4.7, 8192
  // x 768 5.2 / 5.9 and 5.8 / 6.0, 12288 x 768 6.8 / 6.5 and 7.3 / 6.8, 3072 x 2048
  // 5.6 / 5.3 and 6.3 / 6.3)
  if ((K >= 2048 || N >= 12288) &&
      ps_skinny_lds_fits(M, N, K, x_stride, x, w, false)) {
    SlArgs a = {};
    a.out = (unsigned short*)out;
    a.x = (const unsigned short*)x;
    a.w = (const unsigned short*)w;
    a.M = M, a.N = N, a.K = K, a.x_stride = x_stride;
    // Tiles of 16 rows of W side by side, or 8 and the 8 that are N / 2 behind:
    // 16 rows a power of two apart and 16 KB or more long come from few channels
    // of memory (us at one row: 4096 x 8192 17.0 / 15.2, 28672 x 8192 89 / 81,
    // 12288 x 4096 19.8 / 19.9, 28672 x 4096 41.2 / 42.0)
    a.apart = GATED || (K >= 8192 && K % 4096 == 0) ? N / 2 : 8;
    ps_skinny_lds_go<GATED ? SL_GATED : SL_PLAIN, false>(a, stream);
    return;
  }
  // us, 8 waves / 16: 16 rows of 4096 x 8192 17.5 / 19.4, of 8192 x 8192 36.6 /
  // 34.0, 8 rows of 28672 x 8192 104 / 93, one row of 8192 x 1024 5.6 / 6.5
  if (K < 2048 || (M > 8 && N <= 4096))
    PS_SR(1, 8, false, false);
  else
    PS_SR(1, 16, false, false);
#undef PS_SR
}

extern "C" {

// out [M, N / 2] = silu(x Wg^T) * (x Wu^T), W = [Wg; Wu]; -1: not built. Of a W of
// more than 32768 rows only up to 8 rows of x: callers take the plain product and
// the activation for more.
int ps_skinny_gated(void* out, const void* x, const void* w, int M, int N,
                    int K, long x_stride, hipStream_t stream) {
  if (M < 1 || N < 64 || K < 64 || N % 64 != 0 || K % 64 != 0 ||
      (M > 8 && N > 32768) || !ps_skinny_rows(M, N, K, x_stride, x, w))
    return -1;
  ps_skinny_rows_go<true>(out, x, w, M, N, K, x_stride, stream);
  return 0;
}

// out [M, N / 2] = silu(y Wg^T) * (y Wu^T), y = rms_norm(x + res) nw, res_out =
// x + res (no res: y = rms_norm(x) nw); -1: not built
int ps_skinny_norm_gated(void* out, void* res_out, const void* x,
                         const void* res, const void* nw, const void* w,
                         int M, int N, int K, float eps, hipStream_t stream) {
  if (!ps_skinny_lds_fits(M, N, K, K, x, w, true)) return -1;
  SlArgs a = {};
  a.out = (unsigned short*)out;
  a.res_out = (unsigned short*)res_out;
  a.x = (const unsigned short*)x;
  a.res = (const unsigned short*)res;
  a.nw = (const unsigned short*)nw;
  a.w = (const unsigned short*)w;
  a.M = M, a.N = N, a.K = K, a.apart = N / 2, a.x_stride = K, a.eps = eps;
  ps_skinny_lds_go<SL_GATED, true>(a, stream);
  return 0;
}

// out [M, N]: query heads, key heads, value heads of y W^T, the first two rotated,
// the last two in the cache, y as above; without nw y is x. -1: not built
int ps_skinny_rope(void* out, void* res_out, const void* x, long x_stride,
                   const void* res, const void* nw, const void* w, int M,
                   int N, int K, float eps, const void* positions,
                   const void* cos_sin, const void* slots, void* k_cache,
                   void* v_cache, int QH, int KH, int HD, int BS, int kv_fp8,
                   hipStream_t stream) {
  if (HD < 16 || HD % 16 != 0 || N != (QH + 2 * KH) * HD ||
      !ps_skinny_lds_fits(M, N, K, x_stride, x, w, nw != nullptr))
    return -1;
  const SlArgs a = {(unsigned short*)out,
                    (unsigned short*)res_out,
                    (const unsigned short*)x,
                    (const unsigned short*)res,
                    (const unsigned short*)nw,
                    (const unsigned short*)w,
                    M,
                    N,
                    K,
                    HD / 2,
                    x_stride,
                    eps,
                    (const int*)positions,
                    (const float*)cos_sin,
                    (const long*)slots,
                    k_cache,
                    v_cache,
                    QH,
                    KH,
                    HD,
                    BS};
  if (nw != nullptr && kv_fp8)
    ps_skinny_lds_go<SL_ROPE, true, unsigned char>(a, stream);
  else if (nw != nullptr)
    ps_skinny_lds_go<SL_ROPE, true>(a, stream);
  else if (kv_fp8)
    ps_skinny_lds_go<SL_ROPE, false, unsigned char>(a, stream);
  else
    ps_skinny_lds_go<SL_ROPE, false>(a, stream);
  return 0;
}

// Most entries of x that LDS has room for, without the norm and with it.
void ps_skinny_limits(int* most) {
  most[0] = SL_X;
  most[1] = SL_NORM_X;
}

// ws == nullptr forces splits = 1. ps_skinny_gemm_splits reports the
// split depth the heuristic will pick for a shape so the caller can size
// the fp32 workspace.
int ps_skinny_gemm_splits(int M, int N, int K) {
  if (N < 64 || K < 64 || N % 64 != 0 || K % 64 != 0 || M > 256) return -1;
  if (M <= 16 && N <= 32768) return 1;
  return ps_skinny_plan(M, N, K).splits;
}

// The tiles or the short form; `parts`: the partial sums are the result.
static int ps_skinny_splits_go(void* out_bf16, void* ws, const void* x,
                               const void* w, int M, int N, int K,
                               long x_stride, bool parts, hipStream_t stream) {
  PsSkinnyPlan plan = ps_skinny_plan(M, N, K);
  if (ws == nullptr) plan.splits = 1;
#define PS_SG(MT)                                                           \
  skinny_gemm_kernel<MT><<<dim3(N / 64, plan.splits), 256, 0, stream>>>(    \
      (unsigned short*)out_bf16, (float*)ws, (const unsigned short*)x,      \
      (const unsigned short*)w, M, N, K, x_stride)
#define PS_ST(MT, NC)                                                       \
  skinny_tile_kernel<MT, NC, false>                                              \
      <<<dim3(N / (64 * NC) * plan.splits), dim3(512), 0, stream>>>(        \
          (unsigned short*)out_bf16, (float*)ws, (const unsigned short*)x,  \
          (const unsigned short*)w, M, N, K, x_stride, plan.splits)
#define PS_ST2(MT)                                                          \
  do {                                                                      \
    if (plan.form == PS_WIDE)                                               \
      PS_ST(MT, 2);                                                         \
    else                                                                    \
      PS_ST(MT, 1);                                                         \
  } while (0)
  if (plan.form == PS_SHORT) {
    if (M <= 16) PS_SG(1);
    else if (M <= 32) PS_SG(2);
    else if (M <= 64) PS_SG(4);
    else if (M <= 128) PS_SG(8);
    else PS_SG(16);
  } else {
    if (M <= 16) PS_ST2(1);
    else if (M <= 32) PS_ST2(2);
    else if (M <= 64) PS_ST2(4);
    else if (M <= 128) PS_ST2(8);
    else if (M <= 192) PS_ST2(12);
    else PS_ST(16, 1);
  }
#undef PS_ST2
#undef PS_ST
#undef PS_SG
  if (plan.splits > 1 && !parts) {
    const long MN = (long)M * N;
    skinny_combine_kernel<<<dim3((MN / 4 + 255) / 256), 256, 0, stream>>>(
        (unsigned short*)out_bf16, (const float*)ws, MN, plan.splits);
  }
  return 0;
}

int ps_skinny_gemm(void* out_bf16, void* ws, const void* x, const void* w,
                   int M, int N, int K, long x_stride, hipStream_t stream) {
  if (ps_skinny_gemm_splits(M, N, K) < 0) return -1;
  if (M < 1) return 0;  // no rows: their size in bytes would wrap below
  if (ps_skinny_rows(M, N, K, x_stride, x, w)) {
    ps_skinny_rows_go<false>(out_bf16, x, w, M, N, K, x_stride, stream);
    return 0;
  }
  return ps_skinny_splits_go(out_bf16, ws, x, w, M, N, K, x_stride, false,
                             stream);
}

// Partial sums [splits, M, N] in fp32 of more than 16 rows, for a kernel behind
// this one that adds them; -1: not built, or there is only one
int ps_skinny_parts(void* ws, const void* x, const void* w, int M, int N,
                    int K, long x_stride, hipStream_t stream) {
  if (M <= 16 || ps_skinny_gemm_splits(M, N, K) < 2) return -1;
  return ps_skinny_splits_go(nullptr, ws, x, w, M, N, K, x_stride, true,
                             stream);
}

// As ps_skinny_gated for 17 to 192 rows, in tiles that have all of K
int ps_skinny_gated_tiles(void* out, const void* x, const void* w, int M,
                          int N, int K, long x_stride, hipStream_t stream) {
  if (M <= 16 || M > 192 || ps_skinny_gemm_splits(M, N, K) != 1) return -1;
  const PsSkinnyPlan plan = ps_skinny_plan(M, N, K);
  if (plan.form == PS_SHORT) return -1;
#define PS_ST(MT, NC)                                                       \
  skinny_tile_kernel<MT, NC, true>                                          \
      <<<dim3(N / (64 * NC)), dim3(512), 0, stream>>>(                      \
          (unsigned short*)out, nullptr, (const unsigned short*)x,          \
          (const unsigned short*)w, M, N, K, x_stride, 1)
#define PS_ST2(MT)                                                          \
  do {                                                                      \
    if (plan.form == PS_WIDE)                                               \
      PS_ST(MT, 2);                                                         \
    else                                                                    \
      PS_ST(MT, 1);                                                         \
  } while (0)
  if (M <= 32) PS_ST2(2);
  else if (M <= 64) PS_ST2(4);
  else if (M <= 128) PS_ST2(8);
  else PS_ST2(12);
#undef PS_ST2
#undef PS_ST
  return 0;
}

}  // extern "C"
