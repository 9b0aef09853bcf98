// Fused normalisation / activation / rotary kernels for the MI355X engine.
//
// Parity targets (behavioural, not code): the external vLLM engine's
// rms_norm / fused_add_rms_norm / silu_and_mul / rotary_embedding op surface
// that /root/reference drives through its helm engine flags
// (see SURVEY.md section 2.8).  All kernels are memory-bound: the design
// point is HBM3E bandwidth (~6.3 TB/s achievable), so every bf16 access is a
// 16-byte ushort8 vector and each tensor element is touched exactly once
// where possible.
#include "ps_common.h"

// Eight columns of partial sums that lie `apart` entries apart, added in order.
PS_DEV void ps_sum_parts(const float* p, int S, long apart, float* sum) {
  ps_f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll 8
  for (int s = 0; s < S; ++s) {
    a += *(const ps_f32x4*)(p + s * apart);
    b += *(const ps_f32x4*)(p + s * apart + 4);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sum[j] = a[j];
    sum[4 + j] = b[j];
  }
}

// ---------------------------------------------------------------------------
// RMSNorm:  out[t, :] = x[t, :] * rsqrt(mean(x^2) + eps) * w
// with ADD (the per-layer hot path)
//   residual[t,:] += x[t,:];  x[t,:] = rmsnorm(residual[t,:]) * w
// One workgroup per token row, the row and the weights in registers: 2 reads
// and 2 writes per element. A decode batch is bound by the latency of the
// chain, so the weights are asked for with the row and the waves' sums cross
// one barrier (before: the weights after the second of two).
// ---------------------------------------------------------------------------
template <int BLOCK, int VPT, bool ADD>  // VPT ushort8 vectors per thread
__global__ __launch_bounds__(BLOCK) void rms_norm_kernel(
    unsigned short* __restrict__ out,      // [T, D]; with ADD in and out
    const unsigned short* __restrict__ x,  // [T, D]
    unsigned short* __restrict__ residual, // [T, D], with ADD
    const unsigned short* __restrict__ w,  // [D]
    float eps, int D) {
  const long row = blockIdx.x * (long)D;
  unsigned short* orow = out + row;
  const unsigned short* xr = ADD ? orow : x + row;
  unsigned short* rr = ADD ? residual + row : nullptr;

  ps_bf16x8 xv[VPT], rv[VPT], wv[VPT];
#pragma unroll
  for (int u = 0; u < VPT; u++) {
    const int i = (u * BLOCK + (int)threadIdx.x) * 8;
    if (i < D) {
      xv[u] = *(const ps_bf16x8*)(xr + i);
      if constexpr (ADD) rv[u] = *(const ps_bf16x8*)(rr + i);
      wv[u] = *(const ps_bf16x8*)(w + i);
    }
  }
  float vals[VPT][8];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < VPT; u++) {
    const int i = (u * BLOCK + (int)threadIdx.x) * 8;
    if (i < D) {
      ps_bf16x8 sv;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float f = ps_bf16_to_f32(xv[u][j]);
        if constexpr (ADD) f += ps_bf16_to_f32(rv[u][j]);
        vals[u][j] = f;
        ss += f * f;
        sv[j] = ps_f32_to_bf16(f);
      }
      if constexpr (ADD) *(ps_bf16x8*)(rr + i) = sv;
    }
  }
  // reduce ss across the block
  __shared__ float red[BLOCK / 64];
  ss = ps_group_sum<64>(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int k = 0; k < BLOCK / 64; k++) tot += red[k];
  const float inv = rsqrtf(tot / (float)D + eps);

#pragma unroll
  for (int u = 0; u < VPT; u++) {
    const int i = (u * BLOCK + (int)threadIdx.x) * 8;
    if (i < D) {
      ps_bf16x8 ov;
#pragma unroll
      for (int j = 0; j < 8; j++)
        ov[j] = ps_f32_to_bf16(vals[u][j] * inv * ps_bf16_to_f32(wv[u][j]));
      *(ps_bf16x8*)(orow + i) = ov;
    }
  }
}

// The same where x comes as partial sums of a product, [S, T, D] in fp32: their
// sum, rounded as the product's own last step does, is what the norm adds to the
// residual. That step has no launch of its own then (4.8 to 5.4 us a product of a
// decode batch). More threads a row than above, since each has S times the loads.
template <int BLOCK, int VPT>
__global__ __launch_bounds__(BLOCK) void rms_norm_parts_kernel(
    unsigned short* __restrict__ out,       // [T, D]
    const float* __restrict__ parts,        // [S, T, D]
    int S, unsigned short* __restrict__ residual,  // [T, D]
    const unsigned short* __restrict__ w,   // [D]
    float eps, int D) {
  const long row = blockIdx.x * (long)D, TD = gridDim.x * (long)D;
  ps_bf16x8 rv[VPT], wv[VPT];
  float vals[VPT][8];
#pragma unroll
  for (int u = 0; u < VPT; u++) {
    const int i = (u * BLOCK + (int)threadIdx.x) * 8;
    if (i < D) {
      rv[u] = *(const ps_bf16x8*)(residual + row + i);
      wv[u] = *(const ps_bf16x8*)(w + i);
      ps_sum_parts(parts + row + i, S, TD, vals[u]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < VPT; u++) {
    const int i = (u * BLOCK + (int)threadIdx.x) * 8;
    if (i < D) {
      ps_bf16x8 sv;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float f = ps_bf16_to_f32(ps_f32_to_bf16(vals[u][j])) +
                        ps_bf16_to_f32(rv[u][j]);
        vals[u][j] = f;
        ss += f * f;
        sv[j] = ps_f32_to_bf16(f);
      }
      *(ps_bf16x8*)(residual + row + i) = sv;
    }
  }
  __shared__ float red[BLOCK / 64];
  ss = ps_group_sum<64>(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int k = 0; k < BLOCK / 64; k++) tot += red[k];
  const float inv = rsqrtf(tot / (float)D + eps);
#pragma unroll
  for (int u = 0; u < VPT; u++) {
    const int i = (u * BLOCK + (int)threadIdx.x) * 8;
    if (i < D) {
      ps_bf16x8 ov;
#pragma unroll
      for (int j = 0; j < 8; j++)
        ov[j] = ps_f32_to_bf16(vals[u][j] * inv * ps_bf16_to_f32(wv[u][j]));
      *(ps_bf16x8*)(out + row + i) = ov;
    }
  }
}

// ---------------------------------------------------------------------------
// SiLU-and-mul: out[t, d] = silu(x[t, d]) * x[t, D + d], D = out feature dim.
// ---------------------------------------------------------------------------
__global__ void silu_and_mul_kernel(unsigned short* __restrict__ out,
                                    const unsigned short* __restrict__ x,
                                    int D, long total /* = T * D / 8 */) {
  const long stride = (long)gridDim.x * blockDim.x;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += stride) {
    const long elem = idx * 8;
    const long t = elem / D;
    const long d = elem % D;
    ps_bf16x8 g = *(const ps_bf16x8*)(x + t * 2 * (long)D + d);
    ps_bf16x8 u = *(const ps_bf16x8*)(x + t * 2 * (long)D + D + d);
    ps_bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float gf = ps_bf16_to_f32(g[j]);
      float s = gf / (1.f + __expf(-gf));
      o[j] = ps_f32_to_bf16(s * ps_bf16_to_f32(u[j]));
    }
    *(ps_bf16x8*)(out + elem) = o;
  }
}

// ---------------------------------------------------------------------------
// Rotary embedding, GPT-NeoX style (Llama): rotate (r, r + D/2) pairs in the
// leading rot_dim dims of every q / k head.  cos/sin are precomputed on the
// host (guide App. B: never evaluate trig on-device for RoPE).
// cos_sin layout: [max_pos, rot_dim]  (cos[rot/2] || sin[rot/2]), fp32.
// ---------------------------------------------------------------------------
__global__ void rope_kernel(const int* __restrict__ positions,  // [T]
                            unsigned short* __restrict__ q,     // [T, QH*HD]
                            unsigned short* __restrict__ k,     // [T, KH*HD]
                            const float* __restrict__ cos_sin,
                            int QH, int KH, int HD, int ROT) {
  const long t = blockIdx.x;
  const float* cs = cos_sin + (long)positions[t] * ROT;
  const int half = ROT / 2;
  const int total = (QH + KH) * half;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int h = idx / half;
    const int r = idx % half;
    unsigned short* base = (h < QH) ? (q + t * (long)QH * HD + (long)h * HD)
                                    : (k + t * (long)KH * HD + (long)(h - QH) * HD);
    const float c = cs[r];
    const float s = cs[half + r];
    const float x1 = ps_bf16_to_f32(base[r]);
    const float x2 = ps_bf16_to_f32(base[r + half]);
    base[r] = ps_f32_to_bf16(x1 * c - x2 * s);
    base[r + half] = ps_f32_to_bf16(x2 * c + x1 * s);
  }
}

// ---------------------------------------------------------------------------
// C launchers
// ---------------------------------------------------------------------------
extern "C" {

#define PS_NORM(VPT, ADD)                                                    \
  rms_norm_kernel<256, VPT, ADD><<<dim3((unsigned)T), 256, 0, stream>>>(     \
      (unsigned short*)out, (const unsigned short*)x,                        \
      (unsigned short*)residual, (const unsigned short*)w, eps, D)
#define PS_NORM_WIDTH(ADD)                                                   \
  do {                                                                       \
    if (D <= 2048)                                                           \
      PS_NORM(1, ADD);                                                       \
    else if (D <= 4096)                                                      \
      PS_NORM(2, ADD);                                                       \
    else if (D <= 8192)                                                      \
      PS_NORM(4, ADD);                                                       \
    else                                                                     \
      PS_NORM(16, ADD);                                                      \
  } while (0)

void ps_rms_norm(void* out, const void* x, const void* w, float eps, long T,
                 int D, hipStream_t stream) {
  void* residual = nullptr;
  PS_NORM_WIDTH(false);
}

void ps_fused_add_rms_norm(void* out, void* residual, const void* w,
                           float eps, long T, int D, hipStream_t stream) {
  const void* x = nullptr;  // in place
  PS_NORM_WIDTH(true);
}
#undef PS_NORM_WIDTH
#undef PS_NORM

void ps_rms_norm_parts(void* out, const void* parts, int S, void* residual,
                       const void* w, float eps, long T, int D,
                       hipStream_t stream) {
#define PS_NORM(VPT)                                                         \
  rms_norm_parts_kernel<512, VPT><<<dim3((unsigned)T), 512, 0, stream>>>(    \
      (unsigned short*)out, (const float*)parts, S,                          \
      (unsigned short*)residual, (const unsigned short*)w, eps, D)
  if (D <= 4096)
    PS_NORM(1);
  else if (D <= 8192)
    PS_NORM(2);
  else
    PS_NORM(8);
#undef PS_NORM
}

void ps_silu_and_mul(void* out, const void* x, long T, int D,
                     hipStream_t stream) {
  const long total = T * (long)D / 8;
  const int block = 256;
  const long want = (total + block - 1) / block;
  const int grid = (int)(want < 2048 ? (want > 0 ? want : 1) : 2048);
  silu_and_mul_kernel<<<grid, block, 0, stream>>>(
      (unsigned short*)out, (const unsigned short*)x, D, total);
}

void ps_rope(const void* positions, void* q, void* k, const void* cos_sin,
             long T, int QH, int KH, int HD, int ROT, hipStream_t stream) {
  const int block = 256;
  rope_kernel<<<dim3((unsigned)T), block, 0, stream>>>(
      (const int*)positions, (unsigned short*)q, (unsigned short*)k,
      (const float*)cos_sin, QH, KH, HD, ROT);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Fused RoPE + KV append operating IN-PLACE on the packed qkv tensor
// ([T, (QH+2*KH)*HD] with arbitrary row stride): rotates q and k, then
// scatters the rotated k and v rows into the paged cache. Replaces
// rope_kernel + reshape_and_cache_kernel + three .contiguous() copies.
// ---------------------------------------------------------------------------
template <typename KVT>
__global__ void fused_rope_cache_kernel(
    unsigned short* __restrict__ qkv, const int* __restrict__ positions,
    const float* __restrict__ cos_sin, const long* __restrict__ slot_mapping,
    KVT* __restrict__ k_cache, KVT* __restrict__ v_cache,
    int QH, int KH, int HD, int ROT, long qkv_stride, int BS) {
  using KVTr = ps_kv_traits<KVT>;
  using kvec8 = typename KVTr::vec8;
  const long t = blockIdx.x;
  unsigned short* base = qkv + t * qkv_stride;
  const float* cs = cos_sin + (long)positions[t] * ROT;
  const int half = ROT / 2;
  const int total = (QH + KH) * half;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int h = idx / half;
    const int r = idx % half;
    unsigned short* hp = base + (long)h * HD;  // q heads then k heads
    const float c = cs[r];
    const float s = cs[half + r];
    const float x1 = ps_bf16_to_f32(hp[r]);
    const float x2 = ps_bf16_to_f32(hp[r + half]);
    hp[r] = ps_f32_to_bf16(x1 * c - x2 * s);
    hp[r + half] = ps_f32_to_bf16(x2 * c + x1 * s);
  }
  __syncthreads();
  const long slot = slot_mapping[t];
  if (slot < 0) return;
  const long blk = slot / BS;
  const int off = (int)(slot % BS);
  const int kvelems = KH * HD;
  const unsigned short* ksrc = base + (long)QH * HD;
  const unsigned short* vsrc = ksrc + kvelems;
  for (int i = threadIdx.x * 8; i < 2 * kvelems; i += blockDim.x * 8) {
    const bool isv = i >= kvelems;
    const int r = isv ? i - kvelems : i;
    const int h = r / HD;
    const int d = r % HD;
    const long dst = ((blk * KH + h) * BS + off) * (long)HD + d;
    KVT* cache = isv ? v_cache : k_cache;
    const unsigned short* src = (isv ? vsrc : ksrc) + r;
    ps_bf16x8 sv = *(const ps_bf16x8*)src;
    kvec8 ov;
#pragma unroll
    for (int j = 0; j < 8; j++)
      ov[j] = KVTr::from_f32(ps_bf16_to_f32(sv[j]));
    *(kvec8*)(cache + dst) = ov;
  }
}

// The same where half a rotary width and what is left of a head are whole
// 16-byte vectors: a thread rotates a pair of vectors or copies one, straight
// from the packed row to where it belongs, with nothing read back and no
// barrier. A token's vectors are shared by gridDim.y workgroups.
template <typename KVT>
__global__ __launch_bounds__(256) void fused_rope_cache_vec_kernel(
    unsigned short* __restrict__ qkv, const int* __restrict__ positions,
    const float* __restrict__ cos_sin, const long* __restrict__ slot_mapping,
    KVT* __restrict__ k_cache, KVT* __restrict__ v_cache, int QH, int KH,
    int HD, int ROT, long qkv_stride, int BS) {
  using KVTr = ps_kv_traits<KVT>;
  using kvec8 = typename KVTr::vec8;
  const long t = blockIdx.x;
  unsigned short* base = qkv + t * qkv_stride;
  const float* cs = cos_sin + (long)positions[t] * ROT;
  const long slot = slot_mapping[t];
  const int half = ROT / 2, nr = half / 8, np = (HD - ROT) / 8, nv = HD / 8;
  const int rot = (QH + KH) * nr;       // pairs of vectors to rotate
  const int rest = rot + KH * np;       // then what of a key is not rotated
  const int total = rest + KH * nv;     // then the values
  // a cache row of a key or value head
  auto row = [&](int h) {
    return ((slot / BS * KH + h) * BS + slot % BS) * HD;
  };
  auto put = [&](KVT* cache, long at, ps_bf16x8 v) {
    kvec8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = KVTr::from_f32(ps_bf16_to_f32(v[j]));
    *(kvec8*)(cache + at) = o;
  };
  for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < total;
       i += gridDim.y * blockDim.x) {
    if (i < rot) {
      const int h = i / nr, r = i % nr * 8;
      unsigned short* hp = base + (long)h * HD + r;  // q heads then k heads
      const ps_bf16x8 a = *(const ps_bf16x8*)hp;
      const ps_bf16x8 b = *(const ps_bf16x8*)(hp + half);
      float c[8], s[8];
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        *(float4*)(c + j) = *(const float4*)(cs + r + j);
        *(float4*)(s + j) = *(const float4*)(cs + half + r + j);
      }
      ps_bf16x8 x, y;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float x1 = ps_bf16_to_f32(a[j]), x2 = ps_bf16_to_f32(b[j]);
        x[j] = ps_f32_to_bf16(x1 * c[j] - x2 * s[j]);
        y[j] = ps_f32_to_bf16(x2 * c[j] + x1 * s[j]);
      }
      *(ps_bf16x8*)hp = x;
      *(ps_bf16x8*)(hp + half) = y;
      if (h >= QH && slot >= 0) {
        put(k_cache, row(h - QH) + r, x);
        put(k_cache, row(h - QH) + r + half, y);
      }
    } else if (slot >= 0) {
      const bool isv = i >= rest;
      const int k = isv ? i - rest : i - rot, n = isv ? nv : np;
      const int h = k / n, d = k % n * 8 + (isv ? 0 : ROT);
      const ps_bf16x8 v = *(const ps_bf16x8*)(
          base + (long)(QH + (isv ? KH : 0) + h) * HD + d);
      put(isv ? v_cache : k_cache, row(h) + d, v);
    }
  }
}

// The same from partial sums of a product, [S, T, (QH + 2 KH) HD] in fp32, each
// column's sum rounded as the product's own last step does: queries to rows of
// their own, keys and values to the cache. Four columns of each half a thread, all
// splits' loads on their way at once: bound by their latency. us with the product
// before it, 32/8 heads of 128 of 4096: 192 rows 32.0 (the library's product and
// the kernel above 37.0), 128 rows 27.0 (28.6), 64 rows 22.9 (20.9).
template <typename KVT>
__global__ __launch_bounds__(256) void rope_parts_kernel(
    unsigned short* __restrict__ q, const float* __restrict__ parts, int S,
    const int* __restrict__ positions, const float* __restrict__ cos_sin,
    const long* __restrict__ slot_mapping, KVT* __restrict__ k_cache,
    KVT* __restrict__ v_cache, int QH, int KH, int HD, int BS) {
  const long t = blockIdx.x;
  const long N = (long)(QH + 2 * KH) * HD, TN = gridDim.x * N;
  const long slot = slot_mapping[t];
  const int half = HD / 2, nr = half / 4;
  const int rot = (QH + KH) * nr;  // pairs to rotate, then the values
  const int i = blockIdx.y * blockDim.x + threadIdx.x;
  auto sum = [&](long col) {
    const float* p = parts + t * N + col;
    ps_f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < S; ++s) a += *(const ps_f32x4*)(p + s * TN);
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = ps_bf16_to_f32(ps_f32_to_bf16(a[j]));
    return a;
  };
  auto put = [&](KVT* cache, int h, int d, const unsigned short(&v)[4]) {
    typename ps_kv_traits<KVT>::vec4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = ps_kv_traits<KVT>::from_f32(ps_bf16_to_f32(v[j]));
    *(typename ps_kv_traits<KVT>::vec4*)(
        cache + ((slot / BS * KH + h) * BS + slot % BS) * HD + d) = o;
  };
  if (i < rot) {
    const int h = i / nr, r = i % nr * 4;
    const float* cs = cos_sin + (long)positions[t] * HD;
    const ps_f32x4 c = *(const ps_f32x4*)(cs + r);
    const ps_f32x4 s = *(const ps_f32x4*)(cs + half + r);
    const ps_f32x4 a = sum((long)h * HD + r), b = sum((long)h * HD + half + r);
    unsigned short x[4], y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[j] = ps_f32_to_bf16(a[j] * c[j] - b[j] * s[j]);
      y[j] = ps_f32_to_bf16(b[j] * c[j] + a[j] * s[j]);
    }
    if (h < QH) {
      unsigned short* out = q + (t * QH + h) * HD + r;
      *(ps_bf16x4*)out = ps_bf16x4{x[0], x[1], x[2], x[3]};
      *(ps_bf16x4*)(out + half) = ps_bf16x4{y[0], y[1], y[2], y[3]};
    } else if (slot >= 0) {
      put(k_cache, h - QH, r, x);
      put(k_cache, h - QH, r + half, y);
    }
  } else if (i < rot + KH * HD / 4 && slot >= 0) {
    const int col = (i - rot) * 4;
    const ps_f32x4 a = sum((long)(QH + KH) * HD + col);
    unsigned short x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = ps_f32_to_bf16(a[j]);
    put(v_cache, col / HD, col % HD, x);
  }
}

extern "C" void ps_fused_rope_cache(void* qkv, const void* positions,
                                    const void* cos_sin,
                                    const void* slot_mapping, void* k_cache,
                                    void* v_cache, long T, int QH, int KH,
                                    int HD, int ROT, long qkv_stride, int BS,
                                    int kv_fp8, hipStream_t stream) {
  if (ROT % 16 == 0 && HD % 8 == 0 && ROT <= HD && qkv_stride % 8 == 0 &&
      (((size_t)qkv | (size_t)cos_sin | (size_t)k_cache | (size_t)v_cache) &
       15) == 0) {
    // few tokens: a vector a thread, many: a workgroup a token
    const int work = (QH + KH) * (ROT / 16) + KH * (2 * HD - ROT) / 8;
    const dim3 grid((unsigned)T, T < 512 ? (work + 255) / 256 : 1);
    // no more waves than vectors: 4096 tokens of 8/1 heads of 64 5.9 us, 6.5 with
    // four waves
    const int block = work < 256 ? (work + 63) / 64 * 64 : 256;
#define PS_ROPE(KVT)                                                         \
  fused_rope_cache_vec_kernel<KVT><<<grid, block, 0, stream>>>(              \
      (unsigned short*)qkv, (const int*)positions, (const float*)cos_sin,    \
      (const long*)slot_mapping, (KVT*)k_cache, (KVT*)v_cache, QH, KH, HD,   \
      ROT, qkv_stride, BS)
    if (kv_fp8)
      PS_ROPE(unsigned char);
    else
      PS_ROPE(unsigned short);
#undef PS_ROPE
    return;
  }
  if (kv_fp8)
    fused_rope_cache_kernel<unsigned char>
        <<<dim3((unsigned)T), 256, 0, stream>>>(
            (unsigned short*)qkv, (const int*)positions,
            (const float*)cos_sin, (const long*)slot_mapping,
            (unsigned char*)k_cache, (unsigned char*)v_cache, QH, KH, HD,
            ROT, qkv_stride, BS);
  else
    fused_rope_cache_kernel<unsigned short>
        <<<dim3((unsigned)T), 256, 0, stream>>>(
            (unsigned short*)qkv, (const int*)positions,
            (const float*)cos_sin, (const long*)slot_mapping,
            (unsigned short*)k_cache, (unsigned short*)v_cache, QH, KH, HD,
            ROT, qkv_stride, BS);
}

// From partial sums [S, T, (QH + 2 KH) HD]: queries to q [T, QH HD], keys and
// values to the cache; whole heads are rotated. -1: not built
extern "C" int ps_rope_cache_parts(void* q, const void* parts, int S,
                                   const void* positions, const void* cos_sin,
                                   const void* slot_mapping, void* k_cache,
                                   void* v_cache, long T, int QH, int KH,
                                   int HD, int BS, int kv_fp8,
                                   hipStream_t stream) {
  if (HD % 8 != 0 || S < 1 ||
      (((size_t)q | (size_t)parts | (size_t)cos_sin | (size_t)k_cache |
        (size_t)v_cache) &
       15) != 0)
    return -1;
  const int work = (QH + KH) * (HD / 8) + KH * HD / 4;
  const dim3 grid((unsigned)T, (work + 255) / 256);
#define PS_ROPE(KVT)                                                         \
  rope_parts_kernel<KVT><<<grid, 256, 0, stream>>>(                          \
      (unsigned short*)q, (const float*)parts, S, (const int*)positions,     \
      (const float*)cos_sin, (const long*)slot_mapping, (KVT*)k_cache,       \
      (KVT*)v_cache, QH, KH, HD, BS)
  if (kv_fp8)
    PS_ROPE(unsigned char);
  else
    PS_ROPE(unsigned short);
#undef PS_ROPE
  return 0;
}

// ---------------------------------------------------------------------------
// Row-wise int8 KV quantization (CacheGen-style serde for the offload /
// transfer tiers): each row of `hd` elements gets one fp32 scale
// (max|x| / 127). Halves PCIe/host-pool traffic vs bf16 at ~0.4% RMS error.
// ---------------------------------------------------------------------------
__global__ void kv_quant_kernel(signed char* __restrict__ out,
                                float* __restrict__ scales,
                                const unsigned short* __restrict__ in,
                                int hd, long rows) {
  const long r = (long)blockIdx.x * blockDim.y + threadIdx.y;
  if (r >= rows) return;
  const unsigned short* row = in + r * hd;
  signed char* orow = out + r * hd;
  const int lane = threadIdx.x;  // 64 lanes per row
  float amax = 0.f;
  for (int i = lane * 8; i < hd; i += 64 * 8) {
    ps_bf16x8 v = *(const ps_bf16x8*)(row + i);
#pragma unroll
    for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(ps_bf16_to_f32(v[j])));
  }
  amax = ps_group_max<64>(amax);
  const float scale = amax > 0.f ? amax / 127.f : 1.f;
  const float inv = 1.f / scale;
  if (lane == 0) scales[r] = scale;
  for (int i = lane * 8; i < hd; i += 64 * 8) {
    ps_bf16x8 v = *(const ps_bf16x8*)(row + i);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float f = ps_bf16_to_f32(v[j]) * inv;
      orow[i + j] = (signed char)lrintf(fminf(fmaxf(f, -127.f), 127.f));
    }
  }
}

__global__ void kv_dequant_kernel(unsigned short* __restrict__ out,
                                  const signed char* __restrict__ in,
                                  const float* __restrict__ scales,
                                  int hd, long rows) {
  const long r = (long)blockIdx.x * blockDim.y + threadIdx.y;
  if (r >= rows) return;
  const signed char* row = in + r * hd;
  unsigned short* orow = out + r * hd;
  const float scale = scales[r];
  for (int i = threadIdx.x * 8; i < hd; i += 64 * 8) {
    ps_bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; j++)
      v[j] = ps_f32_to_bf16((float)row[i + j] * scale);
    *(ps_bf16x8*)(orow + i) = v;
  }
}

extern "C" {
void ps_kv_quant(void* out, void* scales, const void* in, long rows, int hd,
                 hipStream_t stream) {
  dim3 block(64, 4);
  dim3 grid((unsigned)((rows + 3) / 4));
  kv_quant_kernel<<<grid, block, 0, stream>>>(
      (signed char*)out, (float*)scales, (const unsigned short*)in, hd, rows);
}
void ps_kv_dequant(void* out, const void* in, const void* scales, long rows,
                   int hd, hipStream_t stream) {
  dim3 block(64, 4);
  dim3 grid((unsigned)((rows + 3) / 4));
  kv_dequant_kernel<<<grid, block, 0, stream>>>(
      (unsigned short*)out, (const signed char*)in, (const float*)scales, hd,
      rows);
}
}

// ---------------------------------------------------------------------------
// fp8 activation-quantizing variants (fuse the dynamic
// activation quantization into the producing kernel instead of a separate
// amax + cast pass). Each emits OCP fp8-e4m3 rows plus a per-ROW scale
// (amax/448) for rowwise-scaled fp8 GEMMs. Three phases per row: reduce
// sum-of-squares; compute normed values in registers + reduce row amax;
// quantize + store fp8.
// ---------------------------------------------------------------------------
template <int BLOCK, int MAX_VPT, bool FUSED_ADD>
__global__ __launch_bounds__(BLOCK) void rms_norm_fp8_kernel(
    unsigned char* __restrict__ out_q,      // [T, D] fp8
    float* __restrict__ out_scale,          // [T]
    unsigned short* __restrict__ x,         // [T, D] (delta when fused)
    unsigned short* __restrict__ residual,  // [T, D] in/out (fused only)
    const unsigned short* __restrict__ w,   // [D]
    float eps, int D) {
  const long t = blockIdx.x;
  unsigned short* xr = x + t * (long)D;
  unsigned short* rr = FUSED_ADD ? residual + t * (long)D : nullptr;
  unsigned char* orow = out_q + t * (long)D;

  float vals[MAX_VPT][8];
  int nvec = 0;
  float ss = 0.f;
  for (int i = threadIdx.x * 8; i < D; i += BLOCK * 8) {
    ps_bf16x8 xv = *(const ps_bf16x8*)(xr + i);
    ps_bf16x8 sv;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float f = ps_bf16_to_f32(xv[j]);
      if (FUSED_ADD) {
        f += ps_bf16_to_f32(((const ps_bf16x8*)(rr + i))[0][j]);
        sv[j] = ps_f32_to_bf16(f);
      }
      vals[nvec][j] = f;
      ss += f * f;
    }
    if (FUSED_ADD) *(ps_bf16x8*)(rr + i) = sv;
    nvec++;
  }
  __shared__ float red[BLOCK / 64];
  ss = ps_group_sum<64>(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0) {
    float tot = 0.f;
#pragma unroll
    for (int wv = 0; wv < BLOCK / 64; wv++) tot += red[wv];
    red[0] = rsqrtf(tot / (float)D + eps);
  }
  __syncthreads();
  const float inv = red[0];

  // normed values + row amax
  float amax = 1e-6f;
  nvec = 0;
  for (int i = threadIdx.x * 8; i < D; i += BLOCK * 8) {
    ps_bf16x8 wv = *(const ps_bf16x8*)(w + i);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float f = vals[nvec][j] * inv * ps_bf16_to_f32(wv[j]);
      vals[nvec][j] = f;
      amax = fmaxf(amax, fabsf(f));
    }
    nvec++;
  }
  __shared__ float reda[BLOCK / 64];
  amax = ps_group_max<64>(amax);
  if ((threadIdx.x & 63) == 0) reda[threadIdx.x >> 6] = amax;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = 0.f;
#pragma unroll
    for (int wv = 0; wv < BLOCK / 64; wv++) m = fmaxf(m, reda[wv]);
    reda[0] = m / 448.0f;
    out_scale[t] = m / 448.0f;
  }
  __syncthreads();
  const float rs = 1.0f / reda[0];

  nvec = 0;
  for (int i = threadIdx.x * 8; i < D; i += BLOCK * 8) {
    ps_fp8x8 qv;
#pragma unroll
    for (int j = 0; j < 8; j++)
      qv[j] = ps_f32_to_fp8(vals[nvec][j] * rs);
    *(ps_fp8x8*)(orow + i) = qv;
    nvec++;
  }
}

template <int BLOCK, int MAX_VPT>
__global__ __launch_bounds__(BLOCK) void silu_and_mul_fp8_kernel(
    unsigned char* __restrict__ out_q,  // [T, D] fp8
    float* __restrict__ out_scale,      // [T]
    const unsigned short* __restrict__ x,  // [T, 2D]
    int D) {
  const long t = blockIdx.x;
  const unsigned short* g = x + t * (long)(2 * D);
  const unsigned short* u = g + D;
  unsigned char* orow = out_q + t * (long)D;

  float vals[MAX_VPT][8];
  int nvec = 0;
  float amax = 1e-6f;
  for (int i = threadIdx.x * 8; i < D; i += BLOCK * 8) {
    ps_bf16x8 gv = *(const ps_bf16x8*)(g + i);
    ps_bf16x8 uv = *(const ps_bf16x8*)(u + i);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float a = ps_bf16_to_f32(gv[j]);
      float f = a / (1.0f + __expf(-a)) * ps_bf16_to_f32(uv[j]);
      vals[nvec][j] = f;
      amax = fmaxf(amax, fabsf(f));
    }
    nvec++;
  }
  __shared__ float reda[BLOCK / 64];
  amax = ps_group_max<64>(amax);
  if ((threadIdx.x & 63) == 0) reda[threadIdx.x >> 6] = amax;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = 0.f;
#pragma unroll
    for (int wv = 0; wv < BLOCK / 64; wv++) m = fmaxf(m, reda[wv]);
    reda[0] = m / 448.0f;
    out_scale[t] = m / 448.0f;
  }
  __syncthreads();
  const float rs = 1.0f / reda[0];
  nvec = 0;
  for (int i = threadIdx.x * 8; i < D; i += BLOCK * 8) {
    ps_fp8x8 qv;
#pragma unroll
    for (int j = 0; j < 8; j++)
      qv[j] = ps_f32_to_fp8(vals[nvec][j] * rs);
    *(ps_fp8x8*)(orow + i) = qv;
    nvec++;
  }
}

extern "C" {

void ps_rms_norm_fp8(void* out_q, void* out_scale, void* x, void* residual,
                     const void* w, float eps, long T, int D, int fused,
                     hipStream_t stream) {
  dim3 grid((unsigned)T);
#define PS_RNF(B, V, F)                                                   \
  rms_norm_fp8_kernel<B, V, F><<<grid, B, 0, stream>>>(                    \
      (unsigned char*)out_q, (float*)out_scale, (unsigned short*)x,       \
      (unsigned short*)residual, (const unsigned short*)w, eps, D)
  if (fused) {
    if (D <= 4096) PS_RNF(512, 1, true);
    else PS_RNF(1024, 2, true);
  } else {
    if (D <= 4096) PS_RNF(512, 1, false);
    else PS_RNF(1024, 2, false);
  }
#undef PS_RNF
}

void ps_silu_and_mul_fp8(void* out_q, void* out_scale, const void* x, long T,
                         int D, hipStream_t stream) {
  dim3 grid((unsigned)T);
  if (D <= 4096)
    silu_and_mul_fp8_kernel<512, 1><<<grid, 512, 0, stream>>>(
        (unsigned char*)out_q, (float*)out_scale,
        (const unsigned short*)x, D);
  else
    silu_and_mul_fp8_kernel<1024, 4><<<grid, 1024, 0, stream>>>(
        (unsigned char*)out_q, (float*)out_scale,
        (const unsigned short*)x, D);
}

}  // extern "C"
