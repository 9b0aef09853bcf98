// The recurrences of chunk_scan.hip one token at a time, for segments shorter
// than a chunk: single decode tokens most of all.
//
// One workgroup per (segment, head). What bounds a decode batch is the state,
// read and written once per token (64 sequences x 32 heads x 128 x 128 fp32:
// 268 MB), so the mapping follows its rows in memory: a thread holds four
// neighbouring columns of every RG-th row in registers, 16-byte accesses that
// are contiguous over a wave, all loads of the state in flight before the
// token's vectors are prepared. Sums over rows go through LDS, one partial per
// row group and column. Measured there: 40 us, 6.7 TB/s (general delta; channel
// delta 41, mlstm 42, gla 16 x 128 x 256 42, ssd 128 x 128 x 64 80 us).
//
// A thread per column and lane quarter (the sequential kernels' mapping, which
// remains for widths not built here) touches 64 bytes of a row at a time; at
// the size above it measured 131 us, 2.0 TB/s.
#include "scan_common.h"

// NR: rows of the state per thread; the block has RG row groups of C4 = DV / 4
// threads. RGC: RG where it is one of the usual ones, known ahead: its offsets
// are then immediates, where they would cost 50 registers (0: taken from RG).
template <typename T, int MODE, int NR, int RGC>
__global__ __launch_bounds__(256, RGC && NR <= 16 ? 4 : 2)
void token_scan_kernel(
    void* __restrict__ outv, int ldo, CkIn in,
    const float* __restrict__ p2, const float* __restrict__ normw,
    float* __restrict__ state, float* __restrict__ aux,
    const int* __restrict__ seq_rows, int H, int G, int D, int DVr, int C4r,
    int RGr, float eps, float scale, float c0f, int nmax) {
  constexpr bool DELTA = MODE == CK_GD || MODE == CK_CD;
  constexpr int RG1 = RGC ? RGC : 1;
  const int RG = RGC ? RGC : RGr, C4 = RGC ? 256 / RG1 : C4r;
  const int DV = RGC ? 1024 / RG1 : DVr;
  constexpr bool PERCH = MODE <= CK_GLA;  // a decay per channel
  // per channel: what reads the state for the removal term, for the read-out;
  // decay, removal and write coefficients. Rows past D stay zero
  __shared__ float lz[512], lr[512];
  __shared__ __align__(16) ck_f32x4 lv[512];
  __shared__ __align__(16) float part[1024];  // [RG][DV]
  __shared__ __align__(16) float zv[256];
  __shared__ float red[2][4], red2[2][4];

  const int seg = blockIdx.x / H, hd = blockIdx.x % H;
  const int t0 = seq_rows[4 * seg], n = seq_rows[4 * seg + 1];
  const int p0 = seq_rows[4 * seg + 2], slot = seq_rows[4 * seg + 3];
  if (n >= nmax) return;  // the chunk kernels' segments
  const int tid = threadIdx.x;
  // threads past the last row group go along with it and write nothing
  const int cg = tid % C4, rg = min(tid / C4, RG - 1);
  const bool live = tid < C4 * RG;
  // a uniform base and 32-bit offsets: row rg + r * RG, past D the last one
  // (whose coefficients are then zero)
  char* Sg = (char*)(state + ((size_t)slot * H + hd) * (size_t)D * DV);
  const unsigned off = (unsigned)(rg * DV + cg * 4) * 4;
  const unsigned step = (unsigned)(RG * DV) * 4;
  const unsigned last = (unsigned)((D - 1) * DV + cg * 4) * 4;
  ck_f32x4 S[NR];
  if (p0 != 0) {
#pragma unroll
    for (int r = 0; r < NR; ++r)
      S[r] = *(const ck_f32x4*)(Sg + min(off + r * step, last));
  } else {
#pragma unroll
    for (int r = 0; r < NR; ++r) S[r] = ck_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int i = D + tid; i < 512; i += 256) {
    lz[i] = lr[i] = 0.f;
    lv[i] = ck_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float nrm = 0.f, mrun = 0.f;  // normaliser entry, running maximum
  float* Ng = MODE == CK_MLSTM ? aux + ((size_t)slot * H + hd) * (D + 1)
                               : nullptr;
  if (MODE == CK_MLSTM && p0 != 0) {
    nrm = Ng[min(tid, D - 1)];
    mrun = Ng[D];
  }
  const int grp = hd / (H / G);

  for (int tt = 0; tt < n; ++tt) {
    // row and thread as values the compiler cannot see through: it would keep
    // an address per operand and lane, and every LDS address, beside the state
    int tr = t0 + tt, tid = threadIdx.x;
    asm volatile("" : "+s"(tr));
    asm volatile("" : "+v"(tid));
    const size_t row = (size_t)tr;
    const int lane = tid & 63, wave = tid >> 6;
    const int cg = tid % C4, rg = min(tid / C4, RG - 1);
    const bool live = tid < C4 * RG;
    const int d = tid;
    const bool chan = d < D;
    const int dc = chan ? d : 0;
    const unsigned hk = grp * D + dc, hz = hd * D + dc, hv = hd * DV;
    const int j = tid;  // this thread's column in the read-out
    const bool col = j < DV;
    const unsigned vc = hv + (col ? j : 0);
    const float b0 = PERCH ? in.p0[hz] : in.p0[hd];
    float b1 = 0.f;
    if (MODE == CK_GD) b1 = in.p1[hz];
    if (MODE != CK_GD && MODE != CK_GLA) b1 = in.p1[hd];
    float kv = MxElem<T>::ld((const T*)in.k + row * in.ldk + hk);
    float rv = MxElem<T>::ld((const T*)in.q + row * in.ldq + hk);
    const float dec = MxElem<T>::ld((const T*)in.dec + row * in.lddec +
                                    (PERCH ? hz : (unsigned)hd));
    float av = 0.f;
    if (MODE == CK_GD)
      av = MxElem<T>::ld((const T*)in.a + row * in.lda + hz);
    if (MODE == CK_CD || MODE == CK_MLSTM)
      av = MxElem<T>::ld((const T*)in.a + row * in.lda + hd);
    const float vj = MxElem<T>::ld((const T*)in.v + row * in.ldv + vc);
    const float gj = MxElem<T>::ld((const T*)in.gate + row * in.ldg + vc);
    if (!chan) kv = rv = 0.f;

    // decay, write scale, norms
    float w = 1.f, wr = 1.f, em = 0.f;
    if (MODE == CK_GD) {
      w = expf(-scale * mx_sigmoid(dec + b0));
      av = mx_sigmoid(av + b1);
    } else if (MODE == CK_CD) {
      w = expf(-expf(b1) * ck_softplus(dec + b0));
      av = mx_sigmoid(av);
    } else if (MODE == CK_GLA) {
      w = expf(ck_log_sigmoid(dec + b0) * c0f);
    } else if (MODE == CK_SSD) {
      wr = ck_softplus(dec + b0);
      w = expf(-expf(b1) * wr);
    } else {
      const float ig = c0f * tanhf((av + b0) / c0f);
      const float fg = ck_log_sigmoid(c0f * tanhf((dec + b1) / c0f));
      const float mn = fmaxf(fg + mrun, ig);
      w = expf(fg + mrun - mn);
      wr = expf(ig - mn);
      em = expf(-mn);
      mrun = mn;
    }
    float s0 = 0.f, s1 = 0.f;
    if (DELTA) s0 = kv * kv;
    if (MODE == CK_CD) s1 = rv * rv;
    if (MODE == CK_MLSTM) {
      rv *= scale;
      nrm = w * nrm + wr * kv;
      s0 = chan ? nrm * rv : 0.f;
    }
    if (DELTA || MODE == CK_MLSTM) {
      s0 = mx_wave_sum(s0);
      if (MODE == CK_CD) s1 = mx_wave_sum(s1);
      if (lane == 0) {
        red[0][wave] = s0;
        red[1][wave] = s1;
      }
    }
    if (col) zv[j] = vj;
    __syncthreads();
    float sum0 = 0.f, sum1 = 0.f;
    if (DELTA || MODE == CK_MLSTM) {
      sum0 = red[0][0] + red[0][1] + red[0][2] + red[0][3];
      sum1 = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
    if (chan) {
      ck_f32x4 c = {w, 0.f, 0.f, 0.f};
      if (MODE == CK_GD) {
        const float u = kv * (1.0f / sqrtf(sum0 + 1e-6f));
        lz[d] = u;
        c[1] = -av * u;
        c[2] = kv;
        lr[d] = rv;
      } else if (MODE == CK_CD) {
        const float u = kv * (1.0f / sqrtf(sum0 + 1e-6f));
        lz[d] = w * u;
        c[2] = u;
        lr[d] = rv * (scale / sqrtf(sum1 + 1e-6f));
      } else {
        c[2] = wr * kv;
        lr[d] = MODE == CK_MLSTM ? rv : rv * scale;
      }
      lv[d] = c;
    }
    __syncthreads();
    ck_f32x4 v4 = {0.f, 0.f, 0.f, 0.f}, z4 = v4;
    v4 = *(const ck_f32x4*)(zv + cg * 4);
    if (DELTA) {
      ck_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        acc += lz[rg + r * RG] * S[r];
        // a few rows' coefficients at a time: all of them would spill
        if (r % 8 == 7) __builtin_amdgcn_sched_barrier(0);
      }
      if (live) *(ck_f32x4*)(part + rg * DV + cg * 4) = acc;
      __syncthreads();
      if (col) {
        float z = 0.f;
        for (int x = 0; x < RG; ++x) z += part[x * DV + j];
        // what is written: the general delta's two terms stay apart
        zv[j] = MODE == CK_CD ? av * (vj - z) : z;
      }
      __syncthreads();
      z4 = *(const ck_f32x4*)(zv + cg * 4);
    }
    ck_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const ck_f32x4 c = lv[rg + r * RG];
      ck_f32x4 s = c[0] * S[r];
      if (MODE == CK_GD) s += c[1] * z4;
      s += c[2] * (MODE == CK_CD ? z4 : v4);
      S[r] = s;
      if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      acc += lr[rg + r * RG] * S[r];
      if (r % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    }
    if (live) *(ck_f32x4*)(part + rg * DV + cg * 4) = acc;
    __syncthreads();
    float o = 0.f;
    if (col)
      for (int x = 0; x < RG; ++x) o += part[x * DV + j];
    if (MODE == CK_SSD) {
      if (col)
        ((float*)outv + row * ldo)[vc] =
            (o + p2[hd] * vj) * gj * mx_sigmoid(gj);
    } else {
      if (MODE == CK_MLSTM) o /= fmaxf(fabsf(sum0), em) + 1e-6f;
      const float ss = mx_wave_sum(col ? o * o : 0.f);
      if (lane == 0) red2[0][wave] = ss;
      __syncthreads();
      if (col) {
        const float tot = red2[0][0] + red2[0][1] + red2[0][2] + red2[0][3];
        const float inv = 1.0f / sqrtf(tot / (float)DV + eps);
        const float nw =
            normw[MODE == CK_GD || MODE == CK_MLSTM ? vc : (unsigned)j];
        float g = mx_sigmoid(gj);
        if (MODE == CK_GLA) g *= gj;
        MxElem<T>::st((T*)outv + row * ldo + vc, o * inv * nw * g);
      }
    }
    if (tt + 1 < n) __syncthreads();  // LDS is written anew
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (rg + r * RG < D) *(ck_f32x4*)(Sg + (off + r * step)) = S[r];
  }
  if (MODE == CK_MLSTM) {
    if (tid < D) Ng[tid] = nrm;
    if (tid == 0) Ng[D] = mrun;
  }
}

#define TK_ARGS                                                              \
  void *out, int ldo, CkIn in, const void *p2, const void *normw,            \
      void *state, void *aux, const void *seq_rows, int S_, int H, int G,    \
      int D, int DV, float eps, float scale, float c0, int nmax,             \
      hipStream_t stream
#define TK_PASS                                                              \
  out, ldo, in, p2, normw, state, aux, seq_rows, S_, H, G, D, DV, eps,       \
      scale, c0, nmax, stream

template <typename T, int MODE>
static int tk_launch(TK_ARGS) {
  // 16-byte columns, 256 threads for a token's vectors and read-out, the
  // partial sums' LDS
  if (D > 128 || DV > 256 || DV % 4 || (uintptr_t)state % 16) return 1;
  const int C4 = DV / 4;
  int RG = 256 / C4;
  if (RG > D) RG = D;
  const int rows = (D + RG - 1) / RG;
#define TK_CASE(NR, RGC)                                                     \
  if (rows <= NR && (RGC == 0 || (RGC == RG && RG * C4 == 256))) {           \
    hipLaunchKernelGGL((token_scan_kernel<T, MODE, NR, RGC>), dim3(S_ * H),  \
                       dim3(256), 0, stream, out, ldo, in,                   \
                       (const float*)p2, (const float*)normw, (float*)state, \
                       (float*)aux, (const int*)seq_rows, H, G, D, DV, C4,   \
                       RG, eps, scale, c0, nmax);                            \
    return 0;                                                                \
  }
  TK_CASE(4, 16)
  TK_CASE(8, 16)
  TK_CASE(8, 8)
  TK_CASE(16, 8)
  TK_CASE(32, 4)
  TK_CASE(1, 0)
  TK_CASE(4, 0)
  TK_CASE(16, 0)
  TK_CASE(32, 0)
#undef TK_CASE
  return 1;
}

// mode 0 general delta, 1 channel delta, 2 gla, 3 ssd, 4 mlstm; scale: the
// general delta's decay scale, else the queries'. Segments of fewer than nmax
// rows. Returns 1 where the widths are not built.
extern "C" int mx_token_scan(
    int mode, void* out, int ldo, const void* q, int ldq, const void* k,
    int ldk, const void* v, int ldv, const void* dec, int lddec,
    const void* a, int lda, const void* gate, int ldg, const void* p0,
    const void* p1, const void* p2, const void* normw, void* state, void* aux,
    const void* seq_rows, int S_, int H, int G, int D, int DV, float eps,
    float scale, float c0, int nmax, int dtype, void* stream_) {
  if (S_ <= 0) return 0;
  hipStream_t stream = (hipStream_t)stream_;
  CkIn in = {q, k, v, dec, a, gate, ldq, ldk, ldv, lddec, lda, ldg,
             (const float*)p0, (const float*)p1};
#define TK_MODE(M)                                                          \
  case M:                                                                   \
    return dtype == MX_BF16 ? tk_launch<mx_bf16, M>(TK_PASS)                \
                            : tk_launch<float, M>(TK_PASS);
  switch (mode) {
    TK_MODE(CK_GD)
    TK_MODE(CK_CD)
    TK_MODE(CK_GLA)
    TK_MODE(CK_SSD)
    TK_MODE(CK_MLSTM)
  }
  return 1;
}
