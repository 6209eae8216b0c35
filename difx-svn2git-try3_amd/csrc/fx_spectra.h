// fx_spectra.h — stores of spectrum values in the job's spectrum type, shared
// by the F-stage kernels (fx_fstage.hip, fx_station.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include "fx_kernels.h"

namespace fxg {

// fp8 e4m3 pair (re low byte, im high byte) of y * 2^e, saturated at the
// largest finite value 448
__device__ __forceinline__ unsigned short fp8_pair(float2 y, int e) {
  const float a = fminf(fmaxf(ldexpf(y.x, e), -448.0f), 448.0f);
  const float b = fminf(fmaxf(ldexpf(y.y, e), -448.0f), 448.0f);
  return (unsigned short)(__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false) & 0xFFFF);
}
struct Fp8Out {
  unsigned short* p;          // the band's spectrum of this block
  const signed char* e;       // the band's channel exponents
};

// channel c's value y stored at element i of the spectrum (i = cidx(c))
__device__ __forceinline__ void put_spec(float2* o, long long i, int c, float2 y) { o[i] = y; }
__device__ __forceinline__ void put_spec(__half2* o, long long i, int c, float2 y) { o[i] = __floats2half2_rn(y.x, y.y); }
__device__ __forceinline__ void put_spec(__hip_bfloat162* o, long long i, int c, float2 y) { o[i] = __float22bfloat162_rn(y); }
__device__ __forceinline__ void put_spec(const Fp8Out& o, long long i, int c, float2 y) { o.p[i] = fp8_pair(y, o.e[c]); }

// zero spectrum of one (band, block): C values of the job's spectrum type
__device__ __forceinline__ void zero_spec(void* spectra, int prec, long long outbase, int C, long long gs, int tid,
                                          int nt) {
  if (prec == FXG_XMAC_FP32) {
    float2* o = (float2*)spectra + outbase;
    for (int c = tid; c < C; c += nt) o[cidx(c, gs)] = make_float2(0.f, 0.f);
  } else if (prec == FXG_XMAC_FP8) {
    unsigned short* o = (unsigned short*)spectra + outbase;
    for (int c = tid; c < C; c += nt) o[cidx(c, gs)] = 0;
  } else {
    unsigned* o = (unsigned*)spectra + outbase;
    for (int c = tid; c < C; c += nt) o[cidx(c, gs)] = 0u;
  }
}

}  // namespace fxg
