// Shared by the matrix-core attention kernels that keep the softmax in
// registers: operand types, the exact three-term cut of fp32 weights, the online
// softmax step.
#pragma once

#include "mix_common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 kv_bf16x8;
typedef __attribute__((ext_vector_type(16))) float kv_f32x16;
typedef __attribute__((ext_vector_type(4))) float kv_f32x4;
typedef __attribute__((ext_vector_type(4))) short kv_s4;
typedef __attribute__((ext_vector_type(4))) unsigned int kv_u4;
typedef __attribute__((address_space(3))) kv_s4 kv_lds_s4;

#define KV_LOG2E 1.44269504f
#define KV_LOW (-3.0e38f)
// Powers of two by which a tile's scores may exceed those that set the reference of
// the weights before it moves: what moves it, in a tile where any of a wave's rows
// does, is a product per accumulated number (96 of 560 instructions of the prompt
// form of window_attention.hip, in most tiles, as a sequence's 32nd tile still holds
// the largest score so far of one of 32 rows with 60 %). The reference is as much
// above the score that set it, so that no weight is above 1 and sums of weighted
// values have the range that they have with the maximum itself as reference.
#define KV_FAR 4.f

union KvPack {
  kv_bf16x8 v;
  kv_s4 h[2];
  unsigned int w[4];
  uint4 q;
};

// Two weights (the first one low) cut into three bf16 terms of 8 mantissa bits
// each (truncation; both remainders are exact).
PS_DEV void kv_split(float p0, float p1, unsigned int* a, unsigned int* b,
                     unsigned int* c) {
  const unsigned int x0 = __float_as_uint(p0) & 0xffff0000u;
  const unsigned int x1 = __float_as_uint(p1) & 0xffff0000u;
  const float r0 = p0 - __uint_as_float(x0), r1 = p1 - __uint_as_float(x1);
  const unsigned int y0 = __float_as_uint(r0) & 0xffff0000u;
  const unsigned int y1 = __float_as_uint(r1) & 0xffff0000u;
  const unsigned int z0 = __float_as_uint(r0 - __uint_as_float(y0));
  const unsigned int z1 = __float_as_uint(r1 - __uint_as_float(y1));
  *a = __builtin_amdgcn_perm(x1, x0, 0x07060302u);
  *b = __builtin_amdgcn_perm(y1, y0, 0x07060302u);
  *c = __builtin_amdgcn_perm(z1, z0, 0x07060302u);
}

// One online-softmax step of a lane's N scores v (relative to the reference m, which
// was KV_FAR above the largest score when it last moved, or absolute while m is
// KV_LOW): weights into v, their sum into l, a new reference into m; returns the
// factor for what was accumulated before. mx: the largest v over all lanes of the
// row. The factor is 1 for every lane (and *moved false) when no reference of the
// wave moves. sink2: a sink in powers of two that joins with the row's first
// maximum, of which this lane has `share` (the alternative to kv_sink where what
// lives past the walk costs).
template <int N>
PS_DEV float kv_softmax(float* v, float mx, float* m, float* l, bool* moved,
                        float sink2 = -INFINITY, float share = 0.f) {
  const bool fresh = *m == KV_LOW;
  *moved = __any(mx > 0.f || (fresh && mx > -INFINITY));
  float alpha = 1.f;
  if (*moved) {
    const float top = share != 0.f ? fmaxf(mx, sink2) : mx;
    const float d =
        fresh ? (mx > -INFINITY ? top + KV_FAR : 0.f) : fmaxf(mx + KV_FAR, 0.f);
    if (!fresh) {
      alpha = __builtin_amdgcn_exp2f(-d);
      *m += d;
    } else if (mx > -INFINITY) {
      *m = d;
      if (share != 0.f) *l = share * __builtin_amdgcn_exp2f(sink2 - d);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] -= d;
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = __builtin_amdgcn_exp2f(v[i]);
    s += v[i];
  }
  *l = *l * alpha + s;
  return alpha;
}

// A sink (natural log units) joins a finished row of reference m and denominator
// l; returns the factor for the row's sums. It comes last: scores relative to
// a sink far below them would lose their digits, and to one of minus infinity
// be no numbers.
PS_DEV float kv_sink(float sink, float* m, float* l) {
  const float d = fmaf(sink, KV_LOG2E, -*m);
  if (!(d > 0.f)) {
    *l += __builtin_amdgcn_exp2f(d);
    return 1.f;
  }
  const float f = __builtin_amdgcn_exp2f(-d);
  *l = *l * f + 1.f;
  *m = fminf(*m + d, -KV_LOW);  // the product may be past the largest float
  return f;
}

// LDS written by some lanes of a wave is read by others of the same wave: the
// wave's LDS accesses complete in order, this keeps the compiler to it.
PS_DEV void kv_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Which of `count` sequences a workgroup at place `pos` of as many has: the longest
// ones first, so that none starts late, but the second of two rounds of the CUs
// (`half` places each) from the shortest on, as its workgroups join the first
// round's on their CUs: every CU then has about as many keys to read, and all of
// them stay busy to the end. As sequences come, a CU has two long ones while another
// is done with two short ones. Where the second round is not full, the first places,
// which it joins, have the shortest ones of the first (us, as they come / the longest
// ones there / so: 33 of 2000 to 4000 keys 91 / 101 / 83, fp8 40 / 46 / 40; 40 of 300
// to 4000 93 / 71 / 68).
// Found without a sort: the tile count (at most `most`) that `rank` sequences exceed,
// bit by bit, among counts that the lanes hold. All keep their places where none has
// more than KV_SHORT tiles, every one as many as the first, within an eighth, or one
// more than `whole` tiles, which are several workgroups' (counts say nothing of their
// work then). In more than four rounds, where workgroups start as others end, those
// of up to KV_SHORT tiles keep theirs (`mine` is the place's own count) and do not
// wait for the others' lengths (32/8 heads, 256 x 20 to 300 keys 37 us, 41
// otherwise); in few they have to pair with long ones (61 of 300 to 4000 98 us, 109
// otherwise).
#define KV_ORDER 320  // sequences at most
#define KV_SHORT 16
template <typename F>
PS_DEV int kv_order(F tiles_of, int count, int pos, int lane, int half,
                    int mine, int most, int whole = 0x7fffffff) {
  const int skip = count > 4 * half ? KV_SHORT : 0;
  if (mine <= skip) return pos;
  int tiles[KV_ORDER / 64];
#pragma unroll
  for (int j = 0; j < KV_ORDER / 64; ++j) {
    const int s = j * 64 + lane;
    tiles[j] = s < count ? tiles_of(s) : -1;
  }
  auto above = [&](int t) {  // sequences of more than t tiles
    int n = 0;
#pragma unroll
    for (int j = 0; j < KV_ORDER / 64; ++j)
      if (j * 64 < count) n += __popcll(__ballot(tiles[j] > t));
    return n;
  };
  const int first = __builtin_amdgcn_readfirstlane(tiles[0]);
  bool even = true;  // all within an eighth of the first one
#pragma unroll
  for (int j = 0; j < KV_ORDER / 64; ++j)
    if (j * 64 < count)
      even &= __all(tiles[j] < 0 || abs(tiles[j] - first) <= first / 8);
  int seq = pos;
  if (!even && above(KV_SHORT) > 0 && above(whole) == 0) {
    int rank = 0;  // of this place among those of longer ones
#pragma unroll
    for (int j = 0; j < KV_ORDER / 64; ++j) {
      const int at = min(pos - 64 * j, 64);
      if (at > 0)
        rank += __popcll(__ballot(tiles[j] > skip && lane < at));
    }
    const int end = min(2 * half, above(skip));
    const int pairs = skip > 0 ? half : end - half;  // CUs that get a second one
    if (rank >= half && rank < end)
      rank = half + end - 1 - rank;
    else if (rank < half && pairs > 0)
      rank += rank < pairs ? half - pairs : -pairs;
    int t = 0;
    for (int b = 31 - __clz(most | 1); b >= 0; --b)
      if (above(t + (1 << b) - 1) > rank) t += 1 << b;
    int left = rank - above(t);  // which of those of t tiles
#pragma unroll
    for (int j = 0; j < KV_ORDER / 64; ++j) {
      const unsigned long long m = __ballot(tiles[j] == t);
      const int n = __popcll(m);
      if (left >= 0 && left < n) {
        const int before = __builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        seq = j * 64 + __ffsll((unsigned long long)__ballot(
                           tiles[j] == t && before == left)) - 1;
      }
      left -= n;
    }
    seq = __builtin_amdgcn_readfirstlane(seq);
  }
  return seq;
}
