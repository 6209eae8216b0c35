// fx_fft.h — the transform passes of the F stage on a shifted frequency grid.
//
// A block's samples times the linear fringe rotator, transformed, are the
// samples' transform at the bins k + d (d = the rotator's turns per block):
//     sum_n x[n] e^{-2 pi i (k + d) n/L}.
// In a decimation-in-time FFT only the twiddles know the bin, so the rotation
// costs nothing: every pass of radix R over N finished bins multiplies input r
// by w^r with w = e^{-2 pi i (k + d)/(N R)} instead of e^{-2 pi i k/(N R)}.
// Inside a pass the products w^r never appear either: a radix-2 butterfly
// with its own twiddle t is six FMAs,
//     p = a + t b,  m = 2 a - p,
// and the 32 butterflies of a radix-16 pass need w^8, w^4, w^2, w and four
// fixed multiples of them (e^{-i pi/4} w^2; e^{-i pi q/8} w, q = 1..3; the
// remaining ones are -i times these).
#pragma once
#include <hip/hip_runtime.h>

namespace fxg {

// complex product as two multiplies and two FMAs
__device__ __forceinline__ float2 cmulx(float2 a, float2 b) {
  return make_float2(__builtin_fmaf(-a.y, b.y, a.x * b.x), __builtin_fmaf(a.y, b.x, a.x * b.y));
}

// e^{2 pi i t} of an FP64 angle in turns to FP32 rounding: the nearest quarter
// turn taken off in FP64, then the Taylor polynomials of sine and cosine on an
// eighth of a turn either side (truncation below 3e-9).  The hardware sine and
// cosine are off by up to 1.2e-7 besides their argument's rounding, which in
// the twiddles of every pass would set the spectrum's error.
__device__ __forceinline__ float2 exact_rotator(double t) {
  const double q = rint(4.0 * t);
  const float r = (float)__builtin_fma(-0.25, q, t);
  const int n = (int)q;
  const float z = r * r;
  // (2 pi)^n / n!; 2 pi itself in two parts
  const float ps = __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, 42.0586939f, -76.7058598f), 81.6052493f), -41.3417022f);
  const float s = __builtin_fmaf(r, 6.2831855f, r * __builtin_fmaf(z, ps, -1.7484555e-7f));
  const float c = __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, -26.4262568f, 60.2446414f),
                                 -85.4568172f), 64.9393940f), -19.7392088f), 1.0f);
  const float x = n & 1 ? -s : c, y = n & 1 ? c : s;
  return n & 2 ? make_float2(-x, -y) : make_float2(x, y);
}

// (a, b) -> (a + w b, a - w b)
__device__ __forceinline__ void bfly(float2& a, float2& b, float2 w) {
  const float px = __builtin_fmaf(-w.y, b.y, __builtin_fmaf(w.x, b.x, a.x));
  const float py = __builtin_fmaf(w.y, b.x, __builtin_fmaf(w.x, b.y, a.y));
  b = make_float2(__builtin_fmaf(2.0f, a.x, -px), __builtin_fmaf(2.0f, a.y, -py));
  a = make_float2(px, py);
}
// a + w b alone
__device__ __forceinline__ float2 bfly_plus(float2 a, float2 b, float2 w) {
  return make_float2(__builtin_fmaf(-w.y, b.y, __builtin_fmaf(w.x, b.x, a.x)),
                     __builtin_fmaf(w.y, b.x, __builtin_fmaf(w.x, b.y, a.y)));
}
// -i w
__device__ __forceinline__ float2 rot_mi(float2 w) { return make_float2(w.y, -w.x); }

// The twiddles of a radix-16 pass: w^8, w^4, w^2, e^{-i pi/4} w^2 and
// e^{-i pi q/8} w for q = 0..3.
struct Tw16 {
  float2 w8, w4, w2, w2h, w1, w1a, w1b, w1c;
};
constexpr float kC1 = 0.92387953251128675613f, kS1 = 0.38268343236508977173f, kH = 0.70710678118654752440f;
// e^{-i pi/4} w
__device__ __forceinline__ float2 turn8(float2 w) { return make_float2(kH * (w.x + w.y), kH * (w.y - w.x)); }
// the four fixed multiples from w^2 and w
__device__ __forceinline__ void tw16_multiples(Tw16& t) {
  t.w2h = turn8(t.w2);
  t.w1a = cmulx(t.w1, make_float2(kC1, -kS1));
  t.w1b = turn8(t.w1);
  t.w1c = cmulx(t.w1, make_float2(kS1, -kC1));
}

constexpr int bitrev2(int i) { return ((i & 1) << 1) | ((i & 2) >> 1); }
constexpr int bitrev4(int i) { return ((i & 1) << 3) | ((i & 2) << 1) | ((i & 4) >> 1) | ((i & 8) >> 3); }
constexpr int bitrev3(int i) { return ((i & 1) << 2) | (i & 2) | ((i & 4) >> 2); }

// Stages 2..4 of the radix-16 pass over v, whose stage 1 (butterflies of
// w^8 between r and r + 8) is done: output q is left in v[bitrev4(q)].  With
// HALF only the outputs q < 8 are formed, in v[bitrev4(q)] (even places).
__device__ __forceinline__ void dft16_stage2(float2* v, const Tw16& t) {
#pragma unroll
  for (int r = 0; r < 4; r++) bfly(v[r], v[r + 4], t.w4);
#pragma unroll
  for (int r = 8; r < 12; r++) bfly(v[r], v[r + 4], rot_mi(t.w4));
}
__device__ __forceinline__ void dft16_stage3(float2* v, const Tw16& t) {
#pragma unroll
  for (int r = 0; r < 2; r++) {
    bfly(v[r], v[r + 2], t.w2);
    bfly(v[r + 4], v[r + 6], rot_mi(t.w2));
    bfly(v[r + 8], v[r + 10], t.w2h);
    bfly(v[r + 12], v[r + 14], rot_mi(t.w2h));
  }
}
// twiddle of the last stage's butterfly over places 2 h, 2 h + 1 (h < 8)
__device__ __forceinline__ float2 dft16_last_tw(const Tw16& t, int h) {
  const int q0 = bitrev3(h);
  const float2 w = (q0 & 3) == 0 ? t.w1 : (q0 & 3) == 1 ? t.w1a : (q0 & 3) == 2 ? t.w1b : t.w1c;
  return q0 & 4 ? rot_mi(w) : w;
}
template <bool HALF>
__device__ __forceinline__ void dft16_stage4(float2* v, const Tw16& t) {
#pragma unroll
  for (int h = 0; h < 8; h++) {
    if (HALF) v[2 * h] = bfly_plus(v[2 * h], v[2 * h + 1], dft16_last_tw(t, h));
    else bfly(v[2 * h], v[2 * h + 1], dft16_last_tw(t, h));
  }
}
template <bool HALF>
__device__ __forceinline__ void dft16_tw(float2* v, const Tw16& t) {
#pragma unroll
  for (int r = 0; r < 8; r++) bfly(v[r], v[r + 8], t.w8);
  dft16_stage2(v, t);
  dft16_stage3(v, t);
  dft16_stage4<HALF>(v, t);
}

// Radix 8 likewise, from w^4, w^2 and w: output q in v[bitrev3(q)]
// (HALF: q < 4 only, in the even places)
template <bool HALF>
__device__ __forceinline__ void dft8_tw(float2* v, float2 w4, float2 w2, float2 w1) {
#pragma unroll
  for (int r = 0; r < 4; r++) bfly(v[r], v[r + 4], w4);
#pragma unroll
  for (int r = 0; r < 2; r++) {
    bfly(v[r], v[r + 2], w2);
    bfly(v[r + 4], v[r + 6], rot_mi(w2));
  }
  const float2 w1h = turn8(w1);
#pragma unroll
  for (int h = 0; h < 4; h++) {
    const int q0 = bitrev2(h);
    const float2 w = q0 & 1 ? w1h : w1;
    const float2 tw = q0 & 2 ? rot_mi(w) : w;
    if (HALF) v[2 * h] = bfly_plus(v[2 * h], v[2 * h + 1], tw);
    else bfly(v[2 * h], v[2 * h + 1], tw);
  }
}

}  // namespace fxg
