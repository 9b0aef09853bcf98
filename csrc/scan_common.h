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

PS_DEV float ck_softplus(float z) { return z > 20.f ? z : log1pf(expf(z)); }

PS_DEV float ck_log_sigmoid(float z) {
  return fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
}
