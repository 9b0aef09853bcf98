// Skinny-batch GEMM for decode steps: out[M, N] = x[M, K] @ W[N, K]^T,
// bf16 inputs, fp32 accumulation, M <= 256.
//
// Why it exists: the library's tiles for the products of a decode batch leave
// the read of W, which bounds them, at a third to a half of the rate that memory
// gives. Up to 16 rows (8 of a W of more than 32768) go without splits; more go
// by the tiled form, or by the short form where a workgroup's range of K is
// short or the tiles leave CUs waiting. Figures stand at each.
// mfma_f32_16x16x32_bf16; operand k-pattern as verified in
// csrc/tools/mfma_probe.hip.
#include "ps_common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 ps_gbf16x8;
typedef __attribute__((ext_vector_type(4))) float ps_gf32x4;

PS_DEV ps_gbf16x8 ps_as_gbf16(ps_bf16x8 u) {
  union {
    ps_bf16x8 u16;
    ps_gbf16x8 bf;
  } v;
  v.u16 = u;
  return v.bf;
}

// Up to 16 rows of x (8 of a W of more than 32768): a workgroup owns 16 rows of W
// and all of K, its NW waves take every NW-th 128-byte piece of them, UC pieces
// in flight each, and add up in LDS at the end: no second kernel and no partial
// sums in memory. W goes from memory straight into left operands, x from the
// caches into right ones (rows past the last read as zeros without an access).
// Bound by the read of W, at few rows of W by its latency: 1 x 4096 x 4096 in
// 10.3 us (17.4 with the split kernel, its merge included), 1 x 28672 x 4096 in
// 46 (79; 5.1 TB/s), 1 x 2048 x 2048 in 5.0 (13.1). Reading x costs as many
// load instructions as reading W: 16 rows of it make the wide one 68 us.
// GATED: W holds N / 2 gate rows, then as many up rows; a workgroup takes eight
// of each and writes silu(gate) up, both rounded to bf16 first: [M, N / 2].
template <int UC, int NW, bool GATED>
__global__ __launch_bounds__(NW * 64) void skinny_rows_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, int M, int N, int K, int x_stride) {
  constexpr int PN = 20;  // pitch of a row of sums
  __shared__ __align__(16) float s_sum[NW][16 * PN];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rc = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (GATED ? 8 : 16);
  const int nc = K / 64;  // pieces
  const int wrow = GATED && rc >= 8 ? N / 2 + n0 + rc - 8 : n0 + rc;
  const unsigned short* wp = w + (long)wrow * K + g * 8;
  const auto xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)x, 0, ((M - 1) * x_stride + K) * 2, 0x00020000);
  const unsigned int xo =
      rc < M ? (unsigned int)(rc * x_stride + g * 8) * 2 : 0x80000000u;
  ps_gf32x4 acc = {0.f, 0.f, 0.f, 0.f};
  ps_gbf16x8 wf[UC][2], xf[UC][2];
  // pieces past the end repeat the last one and are not multiplied
  auto load = [&](int u, int c) {
    const int k = min(c, nc - 1) * 64;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wf[u][h] = *(const ps_gbf16x8*)(wp + k + 32 * h);
      xf[u][h] = __builtin_bit_cast(
          ps_gbf16x8,
          __builtin_amdgcn_raw_buffer_load_b128(xr, xo, k * 2 + 64 * h, 0));
    }
  };
  const int w0 = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
  for (int u = 0; u < UC; ++u) load(u, w0 + NW * u);
  for (int c = w0; c < nc; c += NW * UC) {
#pragma unroll
    for (int u = 0; u < UC; ++u) {
      if (c + NW * u < nc) {
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
    if constexpr (GATED) {
      // the quad of up columns is two lanes on
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float gv = ps_bf16_to_f32(ps_f32_to_bf16(v[r]));
        const float uv = ps_bf16_to_f32(
            ps_f32_to_bf16(__shfl_down(v[r], 2, 64)));
        v[r] = gv / (1.f + __expf(-gv)) * uv;
      }
    }
    if (m < M && (!GATED || n < 8))
      *(uint2*)(out + (long)m * (GATED ? N / 2 : N) + n0 + n) = make_uint2(
          (unsigned int)ps_f32_to_bf16(v[0]) |
              ((unsigned int)ps_f32_to_bf16(v[1]) << 16),
          (unsigned int)ps_f32_to_bf16(v[2]) |
              ((unsigned int)ps_f32_to_bf16(v[3]) << 16));
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

// The tiled form, for 17 to 256 rows of x (and 9 to 16 of a W of more than
// 32768): a workgroup owns 64 NC rows of W, all rows of x and a range of K, in
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
template <int MT, int NC>
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
  for (int c = 0; c < NC; ++c)
    wp[c] = w + (long)(n0 + (wn * NC + c) * 16 + rc) * K + g * 8;
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
// 192 x 95232 x 384 56 / 50; 256 x 61440 x 1024 81 / 85. Rows of 2048 columns come from few
// channels in the short form (17 x 128256 x 2048 129 / 102).
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

// Whether the kernel without splits takes it; its byte offsets are 31 bits.
// More than 8 rows reread x too often where the other form needs no splits
// (N > 32768; us, this / the tiles, distinct weights: 16 x 128256 x 4096 283 / 183,
// 16 x 128256 x 2048 151 / 101, 16 x 51200 x 2560 82 / 66).
static bool ps_skinny_rows(int M, int N, int K, long x_stride) {
  return (M <= 8 || (M <= 16 && N <= 32768)) && x_stride >= 0 &&
         (M - 1) * x_stride + K < (1L << 30);
}

template <bool GATED>
static void ps_skinny_rows_go(void* out, const void* x, const void* w, int M,
                              int N, int K, long x_stride,
                              hipStream_t stream) {
#define PS_SR(UC, NW)                                                       \
  skinny_rows_kernel<UC, NW, GATED><<<N / 16, NW * 64, 0, stream>>>(        \
      (unsigned short*)out, (const unsigned short*)x,                       \
      (const unsigned short*)w, M, N, K, (int)x_stride)
  // long rows: four pieces in flight a wave, else a piece and more waves (us
  // at one row, 16 waves of one piece against 8 of four: 2048 x 2048 5.0 /
  // 6.3, 16384 x 2048 16.5 / 20.8, 28672 x 4096 46.2 / 51.6, 4096 x 14336
  // 28.0 / 25.2). Enough workgroups to fill the chip on short rows want smaller
  // ones, the more so where 16 waves do not share out the pieces evenly (16 / 8
  // waves of one piece: 50304 x 768 22.4 / 18.3, 65536 x 1024 33.8 / 27.3, 51200 x
  // 2560 53.3 / 50.4, 16384 x 2048 17.1 / 16.8; 28672 x 4096 47.0 / 48.8, 18944 x
  // 3584 29.8 / 31.2, 8192 x 1024 5.7 / 6.2)
  if (K > 4096)
    PS_SR(4, 8);
  else if (N >= 12288 && K <= 3072)
    PS_SR(1, 8);
  else
    PS_SR(1, 16);
#undef PS_SR
}

extern "C" {


// out [M, N / 2] = silu(x Wg^T) * (x Wu^T), W = [Wg; Wu]; -1: not built
int ps_skinny_gated(void* out, const void* x, const void* w, int M, int N,
                    int K, long x_stride, hipStream_t stream) {
  if (M < 1 || N < 64 || K < 64 || N % 64 != 0 || K % 64 != 0 ||
      !ps_skinny_rows(M, N, K, x_stride))
    return -1;
  ps_skinny_rows_go<true>(out, x, w, M, N, K, x_stride, stream);
  return 0;
}

// ws == nullptr forces splits = 1. ps_skinny_gemm_splits reports the
// split depth the heuristic will pick for a shape so the caller can size
// the fp32 workspace.
int ps_skinny_gemm_splits(int M, int N, int K) {
  if (N < 64 || K < 64 || N % 64 != 0 || K % 64 != 0 || M > 256) return -1;
  if (M <= 16 && N <= 32768) return 1;
  return ps_skinny_plan(M, N, K).splits;
}

int ps_skinny_gemm(void* out_bf16, void* ws, const void* x, const void* w,
                   int M, int N, int K, long x_stride, hipStream_t stream) {
  if (ps_skinny_gemm_splits(M, N, K) < 0) return -1;
  if (M < 1) return 0;  // no rows: their size in bytes would wrap below
  if (ps_skinny_rows(M, N, K, x_stride)) {
    ps_skinny_rows_go<false>(out_bf16, x, w, M, N, K, x_stride, stream);
    return 0;
  }
  PsSkinnyPlan plan = ps_skinny_plan(M, N, K);
  if (ws == nullptr) plan.splits = 1;
#define PS_SG(MT)                                                           \
  skinny_gemm_kernel<MT><<<dim3(N / 64, plan.splits), 256, 0, stream>>>(    \
      (unsigned short*)out_bf16, (float*)ws, (const unsigned short*)x,      \
      (const unsigned short*)w, M, N, K, x_stride)
#define PS_ST(MT, NC)                                                       \
  skinny_tile_kernel<MT, NC>                                                \
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
  if (plan.splits > 1) {
    const long MN = (long)M * N;
    skinny_combine_kernel<<<dim3((MN / 4 + 255) / 256), 256, 0, stream>>>(
        (unsigned short*)out_bf16, (const float*)ws, MN, plan.splits);
  }
  return 0;
}

}  // extern "C"
