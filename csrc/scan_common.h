// Shared by the recurrence kernels (chunk_scan.hip, token_scan.hip): forms,
// operands, and the exponential family with errors of an ulp or two.
#pragma once

#include "mix_common.h"

#define CK_GD 0
#define CK_CD 1
#define CK_GLA 2
#define CK_SSD 3
#define CK_MLSTM 4

typedef __attribute__((ext_vector_type(4))) float ck_f32x4;

// Operands of a recurrence: rows of one step, strides in elements. q is the
// general delta's receptance; a is its removal gate, the channel delta's write
// strength, the matrix LSTM's input gate. p0, p1 in the order of the forms:
// w0, ab | dt_bias, a_log | p0, - | dt_bias, a_log | p0, p1.
struct CkIn {
  const void *q, *k, *v, *dec, *a, *gate;
  int ldq, ldk, ldv, lddec, lda, ldg;
  const float *p0, *p1;  // GD: w0, ab; CD: dt_bias, a_log; GLA: p0
};

// exp(x) for x up to 88, within 2 ulp: the product with log2(e) in two parts,
// the second one applied to the result. Not-a-numbers pass through.
PS_DEV float ck_exp(float x) {
  x = x < -200.f ? -200.f : x;
  const float t = x * 1.44269502f;
  const float lo = fmaf(x, 1.44269502f, -t) + x * 1.92596299e-8f;
  const float y = __builtin_amdgcn_exp2f(t);
  return fmaf(y, lo * 0.693147181f, y);
}

// 1 / y by one Newton step on the hardware's reciprocal; y finite, not 0
PS_DEV float ck_rcp(float y) {
  const float r = __builtin_amdgcn_rcpf(y);
  return fmaf(fmaf(-y, r, 1.f), r, r);
}

// 1 / sqrt(y) likewise; 0 for an infinite y, where the step's correction (far
// below 1 otherwise) is no number and the minimum takes the other argument. A
// choice between the two results cost the operands' kernel 6 %.
PS_DEV float ck_rsqrt(float y) {
  const float r = __builtin_amdgcn_rsqf(y);
  return fmaf(fminf(fmaf(-y * r, r, 1.f), 1.f), 0.5f * r, r);
}

PS_DEV float ck_sigmoid(float x) {
  return ck_rcp(1.f + ck_exp(x < -80.f ? 80.f : -x));
}

// log(1 + exp(-|z|)) as 2 artanh(s), s = e / (2 + e) <= 1 / 3, by its series up to
// s^13 (what is left is below 2e-8 of it), s with its rounding error beside it. Its
// errors are those of log1pf(expf()) (softplus: 2.24 units of 2^-24 at most, 0.42 in
// the mean), in a third of the instructions; they were half of those that laid down
// the channel delta's operands (6007 rows of 32 x 128x128: 531 -> 495 us in all).
PS_DEV float ck_log1p_exp(float z) {
  const float e = expf(-fabsf(z));
  const float d = 2.f + e, de = (2.f - d) + e;  // d + de = 2 + e
  const float r = __builtin_amdgcn_rcpf(d);
  float s = e * r;
  s = fmaf(fmaf(-s, de, fmaf(-d, s, e)), r, s);
  const float lo = fmaf(-s, de, fmaf(-d, s, e)) * r;
  const float q = s * s;
  float p = fmaf(q, 1.f / 13.f, 1.f / 11.f);
  p = fmaf(q, p, 1.f / 9.f);
  p = fmaf(q, p, 1.f / 7.f);
  p = fmaf(q, p, 1.f / 5.f);
  p = fmaf(q, p, 1.f / 3.f);
  return 2.f * (fmaf(s * q, p, lo) + s);
}

PS_DEV float ck_softplus(float z) { return fmaxf(z, 0.f) + ck_log1p_exp(z); }

PS_DEV float ck_log_sigmoid(float z) {
  return fminf(z, 0.f) - ck_log1p_exp(z);
}

// fp32 numbers on the bf16 matrix unit: each finite one is exactly the sum of
// three bf16 terms (h, m, l: 8 bits each; the first one is cut off and not
// rounded, so that the largest numbers stay finite); of an infinity, or what is
// no number, m and l are no numbers. Beside an operand that is bf16 already
// every product is exact, and the unit takes 3 / 16 of the fp32 unit's time.
typedef __attribute__((ext_vector_type(2))) unsigned ck_u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned ck_u32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 ck_bf16x8;

struct CkTerms4 {  // of four numbers
  ck_u32x2 h, m, l;
};
struct CkTerms8 {
  ck_u32x4 h, m, l;
};

PS_DEV unsigned ck_pack_high(float a, float b) {  // upper halves, a the low one
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a),
                               0x07060302u);
}

PS_DEV void ck_split2(float a, float b, unsigned* h, unsigned* m,
                      unsigned* l) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  const unsigned top = 0xffff0000u;
  *h = ck_pack_high(a, b);
  const f32x2 r = {a - __uint_as_float(__float_as_uint(a) & top),
                   b - __uint_as_float(__float_as_uint(b) & top)};
  *m = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
  const f32x2 q = {r[0] - __uint_as_float(*m << 16),
                   r[1] - __uint_as_float(*m & top)};
  *l = __builtin_bit_cast(unsigned, __builtin_convertvector(q, bf16x2));
}

PS_DEV CkTerms4 ck_split(ck_f32x4 x) {
  unsigned h[2], m[2], l[2];
  ck_split2(x[0], x[1], &h[0], &m[0], &l[0]);
  ck_split2(x[2], x[3], &h[1], &m[1], &l[1]);
  return {{h[0], h[1]}, {m[0], m[1]}, {l[0], l[1]}};
}

PS_DEV ck_u32x4 ck_join(ck_u32x2 a, ck_u32x2 b) {
  return {a[0], a[1], b[0], b[1]};
}

PS_DEV CkTerms8 ck_split(ck_f32x4 a, ck_f32x4 b) {
  const CkTerms4 x = ck_split(a), y = ck_split(b);
  return {ck_join(x.h, y.h), ck_join(x.m, y.m), ck_join(x.l, y.l)};
}

// Number j of eight bf16.
PS_DEV float ck_bf16(ck_u32x4 x, int j) {
  return __uint_as_float(j & 1 ? x[j >> 1] & 0xffff0000u : x[j >> 1] << 16);
}

PS_DEV ck_f32x4 ck_mfma(ck_u32x4 a, ck_u32x4 b, ck_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(ck_bf16x8, a), __builtin_bit_cast(ck_bf16x8, b), c, 0,
      0, 0);
}
