// fx_mux.hip — the corner turn of VDIF thread multiplexing for gfx950
// (stage 2 of vdifmux, libraries/vdifio/src/vdifmux.c:878-1000, with the
// data rule every corner turner of cornerturners.c implements): output
// sample-time t carries, in thread order, one unit per thread (its channels
// at t, unitbits bits), padded with zero units to a power of two.
#include <hip/hip_runtime.h>
#include "fx_kernels.h"

namespace fxg {

// An incomplete frame is zero, or (validity propagation) keeps the threads it
// has, the missing threads' units zero; the first lanes of a frame's first row
// write its header.
// Units of U bits from N (a power of two) threads: a lane loads one word of
// every thread, 32/U sample-times, and writes the N output words they fill, so
// that every byte is read and written once; the units move between registers
// by shifts known at compile time, two operations each.  Bound by HBM.  8
// threads of 2 bits, 4000 frames of 8000 bytes each (512 MB moved): 1645 us with
// 16 loads an output word -> 115 (4.5 TB/s).
// VEC: output words of one store, N or 4 (aligned frames) or 1.
template <int U, int N, int VEC>
__global__ __launch_bounds__(256) void k_vdifmux_u(MuxArgs A) {
  constexpr int PER = 32 / U;
  constexpr unsigned UM = U == 32 ? 0xFFFFFFFFu : (1u << (U & 31)) - 1u;
  const int f = blockIdx.x;
  const int w = blockIdx.y * 256 + threadIdx.x;
  unsigned* frame = (unsigned*)(A.dest + (long long)f * A.framebytes);
  if (blockIdx.y == 0 && threadIdx.x < 8) frame[threadIdx.x] = A.headers[(long long)f * 8 + threadIdx.x];
  if (w >= A.outwords / N) return;
  const unsigned long long m = A.mask[f];
  const bool keep = m == A.goodmask || A.partial;    // else the frame is zero
  const long long* const off = A.srcoff + (long long)f * A.nthreads;
  unsigned in[N], out[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    in[k] = 0u;
    if (keep && k < A.nthreads && ((m >> k) & 1ull)) in[k] = ((const unsigned*)(A.src + off[k]))[w];
  }
#pragma unroll
  for (int j = 0; j < N; j++) {
    unsigned v = 0u;
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int u = j * PER + q;
      v |= ((in[u & (N - 1)] >> (u / N * U)) & UM) << (q * U);
    }
    out[j] = v;
  }
  unsigned* const o = frame + 8 + (long long)w * N;
#pragma unroll
  for (int j = 0; j < N; j += VEC) {
    if constexpr (VEC == 4) *(uint4*)(o + j) = make_uint4(out[j], out[j + 1], out[j + 2], out[j + 3]);
    else if constexpr (VEC == 2) *(uint2*)(o + j) = make_uint2(out[j], out[j + 1]);
    else o[j] = out[j];
  }
}

template <int U, int N>
static void launch_vdifmux_un(const MuxArgs& a, hipStream_t stream) {
  constexpr int VEC = N >= 4 ? 4 : N;
  const dim3 grid((unsigned)a.nframes, (unsigned)((a.outwords / N + 255) / 256));
  if ((((uintptr_t)a.dest | (uintptr_t)a.framebytes) & (4 * VEC - 1)) == 0)
    hipLaunchKernelGGL((k_vdifmux_u<U, N, VEC>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((k_vdifmux_u<U, N, 1>), grid, dim3(256), 0, stream, a);
}

template <int U>
static void launch_vdifmux_n(const MuxArgs& a, hipStream_t stream) {
  switch (a.unitsper) {
    case 1: return launch_vdifmux_un<U, 1>(a, stream);
    case 2: return launch_vdifmux_un<U, 2>(a, stream);
    case 4: return launch_vdifmux_un<U, 4>(a, stream);
    case 8: return launch_vdifmux_un<U, 8>(a, stream);
    case 16: return launch_vdifmux_un<U, 16>(a, stream);
    default: return launch_vdifmux_un<U, 32>(a, stream);      // FXG_MUX_MAX_THREADS is below
  }
}

hipError_t launch_vdifmux(const MuxArgs& a, hipStream_t stream) {
  if (a.nframes <= 0) return hipSuccess;
  switch (a.unitbits) {
    case 1: launch_vdifmux_n<1>(a, stream); break;
    case 2: launch_vdifmux_n<2>(a, stream); break;
    case 4: launch_vdifmux_n<4>(a, stream); break;
    case 8: launch_vdifmux_n<8>(a, stream); break;
    case 16: launch_vdifmux_n<16>(a, stream); break;
    case 32: launch_vdifmux_n<32>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace fxg
