// Skinny-batch GEMM for decode steps: out[M, N] = x[M, K] @ W[N, K]^T,
// bf16 inputs, fp32 accumulation, M <= 256.
//
// Why it exists: hipBLASLt's tile selection for the decode-shaped GEMMs
// (qkv [M,4096]x[6144,4096], o, down) streams weights at only 1.4-2 TB/s at
// M in 16..128 (profiles/gemm_plain.log) when the op is purely
// weight-bandwidth-bound (~6 TB/s available). This kernel is built around
// streaming W exactly once:
//   grid = (N/64, SPLITS): workgroup owns 64 N-rows x a K-range.
//   4 waves x 16 N-rows each; B-frags are direct 16-B lane loads from W
//   (lane's col = its N-row, contiguous dims) -- W bytes are read once
//   across the whole grid.
//   x (tiny) is staged per 64-wide K-chunk in XOR-swizzled LDS and consumed
//   as A-frags for ceil(M/16) m-tiles; per-k-chunk MFMA count scales with
//   m-tiles while W traffic stays fixed.
//   Split-K partials go to an fp32 workspace that a second kernel adds up.
// That is the form for 17 to 256 rows, and for 9 to 16 where W has more than
// 32768; fewer have one of their own, below.
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

__global__ __launch_bounds__(256) void skinny_combine_kernel(
    unsigned short* __restrict__ out,  // [M, N] bf16
    const float* __restrict__ ws,      // [S, M, N] fp32
    long MN, int splits) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= MN) return;
  float acc = 0.f;
  for (int s = 0; s < splits; s++) acc += ws[(long)s * MN + i];
  out[i] = ps_f32_to_bf16(acc);
}



// Whether the kernel without splits takes it; its byte offsets are 31 bits.
// More than 8 rows reread x too often where the other form needs no splits
// (N > 32768; us, this / split, distinct weights: 16 x 128256 x 4096 283 / 213,
// 16 x 128256 x 2048 151 / 126, 16 x 51200 x 2560 82 / 79; 8 x 128256 x 4096 222 /
// 236; with splits 16 x 28672 x 4096 68 / 71).
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
  if (M <= 16) return 1;
  const int kchunks = K / 64;
  const int target_wgs = 1024;
  int splits = target_wgs / (N / 64);
  if (splits < 1) splits = 1;
  if (splits > kchunks) splits = kchunks;
  // the kernel hands out whole ranges of ceil(kchunks / splits) chunks: count
  // the ranges that are not empty, since an empty one writes no partial and
  // the combine pass would add what its workspace happened to hold
  const int per_split = (kchunks + splits - 1) / splits;
  return (kchunks + per_split - 1) / per_split;
}

int ps_skinny_gemm(void* out_bf16, void* ws, const void* x, const void* w,
                   int M, int N, int K, long x_stride, hipStream_t stream) {
  int splits = ps_skinny_gemm_splits(M, N, K);
  if (splits < 0) return -1;
  if (M < 1) return 0;  // no rows: their size in bytes would wrap below
  if (ps_skinny_rows(M, N, K, x_stride)) {
    ps_skinny_rows_go<false>(out_bf16, x, w, M, N, K, x_stride, stream);
    return 0;
  }
  if (ws == nullptr) splits = 1;
  dim3 grid(N / 64, splits);
  dim3 block(256);
#define PS_SG(MT)                                                           \
  skinny_gemm_kernel<MT><<<grid, block, 0, stream>>>(                       \
      (unsigned short*)out_bf16, (float*)ws, (const unsigned short*)x,      \
      (const unsigned short*)w, M, N, K, x_stride)
  if (M <= 16) PS_SG(1);
  else if (M <= 32) PS_SG(2);
  else if (M <= 64) PS_SG(4);
  else if (M <= 128) PS_SG(8);
  else PS_SG(16);
#undef PS_SG
  if (splits > 1) {
    const long MN = (long)M * N;
    skinny_combine_kernel<<<dim3((MN + 255) / 256), 256, 0, stream>>>(
        (unsigned short*)out_bf16, (const float*)ws, MN, splits);
  }
  return 0;
}

}  // extern "C"
