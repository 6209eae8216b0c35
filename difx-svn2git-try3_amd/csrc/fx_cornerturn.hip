// fx_cornerturn.hip — the corner turn for gfx950: frame payloads (sample-time
// major, channel minor) to one contiguous sample stream per band, which the F
// stage and the phase cal read.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "fx_kernels.h"
#include "fx_bits.h"

namespace fxg {

// ---------------------------------------------------------------------------
// k_cornerturn: one workgroup per (frame, datastream), for jobs whose
// datastreams differ in shape or are not aligned.  De-interleaves the
// frame payload (sample-time major, channel minor) into one contiguous
// sample stream per band, unitbits per sample (nbits, or 2 nbits for complex
// samples), LSB first, so that the F-stage of one band reads L*unitbits/8
// contiguous bytes per FFT block.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_cornerturn(const DevStation* __restrict__ st,
                                                    const DevStationSub* __restrict__ ss,
                                                    unsigned char* __restrict__ ct) {
  extern __shared__ unsigned char pay[];
  const int s = blockIdx.y;
  const DevStation S = st[s];
  const DevStationSub Q = ss[s];
  const long long f = blockIdx.x;
  if (f >= Q.nframes) return;
  const unsigned char* src = Q.data + f * S.framebytes + S.headerbytes;
  if ((((unsigned long long)Q.data | (unsigned long long)S.framebytes | (unsigned long long)S.headerbytes) & 3) == 0) {
    // eight words per thread in flight before their LDS stores
    const unsigned* s32 = (const unsigned*)src;
    unsigned* p32 = (unsigned*)pay;
    const int nw = S.databytes / 4;
    for (int i0 = threadIdx.x; i0 < nw; i0 += 8 * blockDim.x) {
      unsigned w[8];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int i = i0 + q * blockDim.x;
        if (i < nw) w[q] = s32[i];
      }
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int i = i0 + q * blockDim.x;
        if (i < nw) p32[i] = w[q];
      }
    }
  } else {
    for (int i = threadIdx.x; i < S.databytes; i += blockDim.x) pay[i] = src[i];
  }
  __syncthreads();
  const int nbits = S.unitbits, nchan = S.nchan, bpf = S.bpf;
  if (nbits >= 8) {
    // units of whole bytes (complex 8-bit: two bytes per unit)
    const int bpu = nbits / 8;
    for (int ob = threadIdx.x; ob < nchan * bpf; ob += blockDim.x) {
      const int c = ob / bpf, i = ob - c * bpf;
      const int u = i / bpu;
      ct[Q.ctbase + (long long)c * Q.ctstride + f * bpf + i] = pay[(u * nchan + c) * bpu + (i - u * bpu)];
    }
    return;
  }
  const int per = 8 / nbits;                   // samples per output byte
  const unsigned mask = (1u << nbits) - 1u;
  for (int ob = threadIdx.x; ob < nchan * bpf; ob += blockDim.x) {
    const int c = ob / bpf, i = ob - c * bpf;
    unsigned v = 0;
    for (int k = 0; k < per; k++) {
      const int bit = ((i * per + k) * nchan + c) * nbits;
      v |= ((pay[bit >> 3] >> (bit & 7)) & mask) << (k * nbits);
    }
    ct[Q.ctbase + (long long)c * Q.ctstride + f * bpf + i] = (unsigned char)v;
  }
}

// ---------------------------------------------------------------------------
// k_cornerturn2<W>: the same corner turn for 2-bit frames whose sample-times
// are W whole 32-bit words (16 W bands), used when every datastream has that
// shape and 4W-byte aligned frames.  A workgroup stages 4096 consecutive
// sample-times through LDS with coalesced loads; each thread then turns 16
// of them for all bands with a 2-bit transpose in registers and stores one
// coalesced word per band.
// ---------------------------------------------------------------------------
template <int W>
__global__ __launch_bounds__(256) void k_cornerturn2(const DevStation* __restrict__ st,
                                                     const DevStationSub* __restrict__ ss,
                                                     unsigned char* __restrict__ ct) {
  using VW = typename std::conditional<W == 1, unsigned, typename std::conditional<W == 2, uint2, uint4>::type>::type;
  constexpr int TPW = 16 * 256;                        // sample-times per workgroup
  __shared__ VW buf[TPW + TPW / 16];                   // element i at i + i/16
  const int s = blockIdx.y;
  const DevStation S = st[s];
  const DevStationSub Q = ss[s];
  const long long spf = S.databytes / (4 * W);          // sample-times per frame
  const long long total = Q.nframes * spf;
  const long long base = (long long)blockIdx.x * TPW;
  if (base >= total) return;                            // the whole workgroup
  // frame f and sample-time r within it of this thread's sample-time, kept
  // up to date as it steps by 256 (one division per workgroup)
  const long long fw = base / spf;
  long long f = fw;
  long long r = base - fw * spf + threadIdx.x;
  while (r >= spf) { r -= spf; f++; }
  // all 16 loads in flight before the first LDS store
  VW v[16];
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const long long tau = base + threadIdx.x + k * 256;
    if (tau < total) {
      v[k] = ((const VW*)(Q.data + f * S.framebytes + S.headerbytes))[r];
    } else {
      memset(&v[k], 0, sizeof v[k]);
    }
    r += 256;
    while (r >= spf) { r -= spf; f++; }
  }
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const int i = threadIdx.x + k * 256;
    buf[i + (i >> 4)] = v[k];
  }
  __syncthreads();
  const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
  if (g * 16 >= total) return;
  uint32_t w[W][16];
#pragma unroll
  for (int t = 0; t < 16; t++) {
    const VW v = buf[threadIdx.x * 17 + t];
    const uint32_t* pv = (const uint32_t*)&v;
#pragma unroll
    for (int c = 0; c < W; c++) w[c][t] = pv[c];
  }
#pragma unroll
  for (int c = 0; c < W; c++) {
    transpose16x2(w[c]);
#pragma unroll
    for (int k = 0; k < 16; k++)
      ((uint32_t*)(ct + Q.ctbase + (long long)(16 * c + k) * Q.ctstride))[g] = w[c][k];
  }
}

// ---------------------------------------------------------------------------
// k_cornerturn_u<U, N, VEC>: the corner turn in registers for units of U bits
// and 2^N bands, used when every datastream has that shape and frames aligned
// to loads of VEC words (2-bit frames of 16 bands and more take
// k_cornerturn2, whose staged loads are whole lines).  The payloads are one
// stream of words that skips the headers; 2^N of them are 32/U sample-times of
// every band, which a thread loads, turns (turn_units) and stores as one word
// per band, coalesced over the threads.  A copy bound by HBM, against a
// workgroup per frame that gathered every output byte from LDS: 30 stations x
// 8 bands, 2-bit, 2 GB 2.76 -> 0.84 ms; 7 stations x 16 bands, 8-bit, 0.95 GB
// 1.24 -> 0.41 ms; 3 stations x 4 bands, 75 KB 14.6 -> 5.7 us.
// ---------------------------------------------------------------------------
constexpr int ct_groups(int N) { return N >= 4 ? 1 : 16 >> N; }   // groups per thread: 16 words in flight or more

template <int U, int N, int VEC>
__global__ __launch_bounds__(256) void k_cornerturn_u(const DevStation* __restrict__ st,
                                                      const DevStationSub* __restrict__ ss,
                                                      unsigned char* __restrict__ ct) {
  using VW = typename std::conditional<VEC == 1, unsigned, typename std::conditional<VEC == 2, uint2, uint4>::type>::type;
  constexpr int NC = 1 << N, K = ct_groups(N), NV = NC / VEC;
  const int s = blockIdx.y;
  const DevStation& S = st[s];
  const DevStationSub& Q = ss[s];
  const int wpf = S.databytes / 4;                      // payload words per frame, a multiple of VEC
  const long long total = Q.nframes * (long long)wpf;
  const long long groups = (total + NC - 1) / NC, g0 = (long long)blockIdx.x * 256 * K;
  if (g0 >= groups) return;                             // the whole workgroup
  const long long fw = g0 * NC / wpf;                   // frame and word of the workgroup's first word
  const int rw = (int)(g0 * NC - fw * wpf);
  // and of this thread's first group, and its step of 256 groups, by division:
  // one frame at a time a workgroup's last group of a payload of 8 bytes is 2048
  // steps off (the stage for 8 blocks of 512 samples, two 8-bit bands: 288 -> 9 us)
  const unsigned r0 = (unsigned)rw + threadIdx.x * NC, step = 256 * NC / (unsigned)wpf;
  long long fg = fw + r0 / (unsigned)wpf;
  int rg = (int)(r0 % (unsigned)wpf);
  union { uint32_t w[NC]; VW v[NV]; } x[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int o = (threadIdx.x + k * 256) * NC;
    long long f = fg;
    int r = rg;
    fg += step;
    rg += 256 * NC - (int)step * wpf;
    if (rg >= wpf) { rg -= wpf; fg++; }
    const long long left = total - g0 * NC - o;         // words from this group's first to the stream's end
#pragma unroll
    for (int i = 0; i < NV; i++) {
      if (i * VEC < left) x[k].v[i] = *(const VW*)(Q.data + f * S.framebytes + S.headerbytes + 4LL * r);
      else memset(&x[k].v[i], 0, sizeof(VW));
      r += VEC;
      if (r >= wpf) { r -= wpf; f++; }
    }
  }
#pragma unroll
  for (int k = 0; k < K; k++) {
    const long long g = g0 + threadIdx.x + k * 256;
    if (g >= groups) break;
    turn_units<U, N>(x[k].w);
#pragma unroll
    for (int i = 0; i < NC; i++)
      ((uint32_t*)(ct + Q.ctbase + (long long)turned_channel<U, N>(i) * Q.ctstride))[g] = x[k].w[i];
  }
}

template <int U>
static bool launch_ct_u(const CornerTurn& c, const DevStation* st, const DevStationSub* ss, unsigned char* ct, int nst,
                        hipStream_t stream) {
  const long long per = 256LL * ct_groups(c.logn);
  const dim3 grid((unsigned)((c.maxgroups + per - 1) / per), nst), block(256);
#define X(Nv, Vv) \
  if (c.logn == Nv && c.vec == Vv) { hipLaunchKernelGGL((k_cornerturn_u<U, Nv, Vv>), grid, block, 0, stream, st, ss, ct); return true; }
  X(0, 1) X(1, 2) X(2, 2) X(2, 4) X(3, 2) X(3, 4) X(4, 2) X(4, 4) X(5, 2) X(5, 4) X(6, 2)
#undef X
  return false;
}

hipError_t launch_cornerturn(const DevStation* st, const DevStationSub* ss, unsigned char* ct, int nst,
                             const CornerTurn& c, hipStream_t stream) {
  if (c.maxframes <= 0) return hipSuccess;
  if (c.fastW) {
    const long long groups = (c.maxsamples + 15) / 16;
    dim3 grid((unsigned)((groups + 255) / 256), nst);
    if (c.fastW == 1) hipLaunchKernelGGL(k_cornerturn2<1>, grid, dim3(256), 0, stream, st, ss, ct);
    else if (c.fastW == 2) hipLaunchKernelGGL(k_cornerturn2<2>, grid, dim3(256), 0, stream, st, ss, ct);
    else hipLaunchKernelGGL(k_cornerturn2<4>, grid, dim3(256), 0, stream, st, ss, ct);
    return hipGetLastError();
  }
  if (c.unit == 2 ? launch_ct_u<2>(c, st, ss, ct, nst, stream) : c.unit == 4 ? launch_ct_u<4>(c, st, ss, ct, nst, stream)
      : c.unit == 8 ? launch_ct_u<8>(c, st, ss, ct, nst, stream) : c.unit == 16 && launch_ct_u<16>(c, st, ss, ct, nst, stream))
    return hipGetLastError();
  dim3 grid((unsigned)c.maxframes, nst);
  hipLaunchKernelGGL(k_cornerturn, grid, dim3(256), (size_t)c.maxdatabytes, stream, st, ss, ct);
  return hipGetLastError();
}

}  // namespace fxg
