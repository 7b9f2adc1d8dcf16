// Shared device/host helpers for the gfx950 BPM and Debye-Wolf kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#define BPMH_DEV __device__ __forceinline__
#define BPMH_HD __host__ __device__ __forceinline__

// Complex helpers on float2 (x = real, y = imag).
BPMH_HD float2 c_add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
BPMH_HD float2 c_sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
BPMH_HD float2 c_scale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// a*b with the component formula (a.x b.x - a.y b.y, a.x b.y + a.y b.x)
BPMH_HD float2 c_mul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a*conj(b)
BPMH_HD float2 c_mulc(float2 a, float2 b) {
  return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
// multiply by -i (forward) or +i (inverse)
template <bool INV>
BPMH_HD float2 c_rot90(float2 a) {
  return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

// IEEE float32 arithmetic that is never fused into an FMA with a neighbouring
// operation, used where a formula of the reference has to be reproduced
// operation by operation (HIP's __fmul_rn / __fadd_rn are plain operators
// that the compiler contracts; the pragma marks these operations as not
// contractible, so each rounds on its own in every kernel that inlines
// them).
BPMH_DEV float f_mul(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
BPMH_DEV float f_add(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}
BPMH_DEV float f_sub(float a, float b) {
#pragma clang fp contract(off)
  return a - b;
}
BPMH_DEV float f_div(float a, float b) {
#pragma clang fp contract(off)
  return a / b;
}
BPMH_DEV double d_mul(double a, double b) {
#pragma clang fp contract(off)
  return a * b;
}
BPMH_DEV double d_add(double a, double b) {
#pragma clang fp contract(off)
  return a + b;
}
BPMH_DEV double d_sub(double a, double b) {
#pragma clang fp contract(off)
  return a - b;
}

// cos/sin of a float32 angle, evaluated in float64 and rounded to float32.
// The angle less its nearest multiple of pi/2 (two FMAs with pi/2 split into
// two float64 parts, exact to 2^-54 for |x| < 2^31) goes through the Taylor
// series of sin to r^13 and cos to r^14 on [-pi/4, pi/4]; the first omitted
// terms are below 2.1e-14 and 1.1e-15 (no rounded result differed from the
// exact values' over 4 million arguments up to 2000).  27 float64 operations
// and no branch, against the library's sincos with its reduction for
// arguments of any size: weighted pass B at 1024^2, whose time after the mean
// is known is this evaluation, 13.64 -> 13.24 us (kernel trace).
BPMH_DEV float2 sincos_f32_via_f64(float ph) {
  const double x = (double)ph;
  const double n = rint(x * 0.63661977236758134308);       // 2/pi
  double r = fma(-n, 1.57079632679489655800, x);            // pi/2, high part
  r = fma(-n, 6.12323399573676603587e-17, r);               // low part
  const double r2 = r * r;
  double s = fma(r2, 1.60590438368216145994e-10, -2.50521083854417187751e-8);  // 1/13!, -1/11!
  s = fma(r2, s, 2.75573192239858906526e-6);                // 1/9!
  s = fma(r2, s, -1.98412698412698412698e-4);               // -1/7!
  s = fma(r2, s, 8.33333333333333333333e-3);                // 1/5!
  s = fma(r2, s, -1.66666666666666666667e-1);               // -1/3!
  s = fma(r * r2, s, r);
  double c = fma(r2, -1.14707455977297247139e-11, 2.08767569878680989792e-9);  // -1/14!, 1/12!
  c = fma(r2, c, -2.75573192239858906526e-7);               // -1/10!
  c = fma(r2, c, 2.48015873015873015873e-5);                // 1/8!
  c = fma(r2, c, -1.38888888888888888889e-3);               // -1/6!
  c = fma(r2, c, 4.16666666666666666667e-2);                // 1/4!
  c = fma(r2, c, -0.5);
  c = fma(r2, c, 1.0);
  const float sf = (float)s, cf = (float)c;
  // quarter turns: n mod 4
  const int q = (int)(n - 4. * floor(n * 0.25));
  const float a = (q & 1) ? sf : cf, b = (q & 1) ? cf : sf;
  return make_float2((q == 1 || q == 2) ? -a : a, (q & 2) ? -b : b);
}

// sin and cos of |x| <= pi/4 by the Taylor series of sin to x^9 and cos to
// x^10, in Horner form with FMA; the first omitted terms are below 2.5e-9
// relative, so the result is within about 1 ulp.
constexpr float kSincosNear = 0.78539816f;
BPMH_DEV void sincos_near(float x, float* s, float* c) {
  const float x2 = x * x;
  float ps = fmaf(x2, 2.75573192e-6f, -1.98412698e-4f);  // 1/9!, -1/7!
  ps = fmaf(x2, ps, 8.33333333e-3f);                      // 1/5!
  ps = fmaf(x2, ps, -1.66666667e-1f);                     // -1/3!
  *s = fmaf(x * x2, ps, x);
  float pc = fmaf(x2, -2.75573192e-7f, 2.48015873e-5f);   // -1/10!, 1/8!
  pc = fmaf(x2, pc, -1.38888889e-3f);                     // -1/6!
  pc = fmaf(x2, pc, 4.16666667e-2f);                      // 1/4!
  pc = fmaf(x2, pc, -0.5f);
  *c = fmaf(x2, pc, 1.f);
}

// sin and cos of a float32 angle: the series up to pi/4 (every phase screen
// of a physical index contrast: |k0 dz dn| is far below that), the
// range-reduced library sincosf beyond.
BPMH_DEV void sincos_fast(float x, float* s, float* c) {
  if (fabsf(x) <= kSincosNear) sincos_near(x, s, c);
  else sincosf(x, s, c);
}

// Streaming (nontemporal) global accesses.  Used where measurement favours
// them: the row pass's plane loads and stores (the column tiles that read and
// write the plane next run on other XCDs, so the lines are not reused from
// this XCD's L2) and the write-once per-plane output volumes.  The column
// pass keeps ordinary accesses: neighbouring tiles share 128-B lines in L2.
typedef float bpmh_f2v __attribute__((ext_vector_type(2)));
BPMH_DEV float2 ld_stream(const float2* q) {
  const bpmh_f2v w = __builtin_nontemporal_load((const bpmh_f2v*)q);
  return make_float2(w.x, w.y);
}
BPMH_DEV float ld_stream(const float* q) { return __builtin_nontemporal_load(q); }
BPMH_DEV void st_stream(float2* q, float2 v) {
  const bpmh_f2v w = {v.x, v.y};
  __builtin_nontemporal_store(w, (bpmh_f2v*)q);
}
BPMH_DEV void st_stream(float* q, float v) { __builtin_nontemporal_store(v, q); }

// The reference's M_PI in bpm_3d_kernels.cl:3 (a float literal).
#define BPMH_PI_F 3.14159265358979f
