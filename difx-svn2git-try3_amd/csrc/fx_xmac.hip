// fx_xmac.hip — baseline-based (X-engine) kernels for gfx950:
//   k_xmac_f32   dense Hermitian cross-multiply-accumulate over every input
//                (datastream band) of one frequency, FP32 FMA: the plain
//                drop-in for Core::processdata's vectorAddProduct_cf32
//                (core.cpp:826-975) and Mode's autocorrelations
//                (mode.cpp:1292-1375)
//   k_weights    baseline and autocorrelation weights (core.cpp:998-1045,
//                mode.cpp:1299-1307)
//   k_scatter    copy into the core result layout (core.cpp:1781-1787,
//                1299-1366)
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include "fx_kernels.h"

namespace fxg {

// ---------------------------------------------------------------------------
// FP32 XMAC.  One workgroup = one channel tile of CT channels of one
// frequency; every thread owns one channel and one 8x8 tile (ta <= tb) of
// the input-by-input product matrix, accumulating
//     V[a][b][c] += X_a[c] * conj(X_b[c])
// over every block of the chunk.  Input spectra are staged through LDS, TB
// blocks at a time.
// ---------------------------------------------------------------------------


__device__ __forceinline__ float2 load_spec(const float2* p, long long i) { return p[i]; }
__device__ __forceinline__ float2 load_spec(const __half2* p, long long i) { return __half22float2(p[i]); }
__device__ __forceinline__ float2 load_spec(const __hip_bfloat162* p, long long i) {
  __hip_bfloat162 v = p[i];
  return make_float2(__bfloat162float(v.x), __bfloat162float(v.y));
}

template <typename TS>
__global__ __launch_bounds__(576) void k_xmac_f32(XmacArgs A) {
  const TS* spec = (const TS*)A.spec;
  extern __shared__ float2 sh[];              // [TB][G*8][CT]
  const int tid = threadIdx.x;
  const int nthreads = blockDim.x;
  const int CT = A.CT, TB = A.TB, NP = A.G * 8;
  const int c0 = blockIdx.x * CT;
  const int sb0 = blockIdx.y * A.split_blocks;               // this row's blocks
  const int nb = min(A.nblocks - sb0, A.split_blocks);
  float2* const Vout = A.V + (long long)blockIdx.y * A.vsplit;
  const int cl = tid % CT;
  const int tile = tid / CT;
  int ta = 0, tb = 0;
  {
    int t = tile, row = 0;
    while (row < A.G && t >= A.G - row) { t -= A.G - row; row++; }
    ta = row; tb = row + t;
  }
  const bool active = tile < A.ntiles;
  float2 acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int k = 0; k < 8; k++) acc[i][k] = make_float2(0.f, 0.f);

  for (int t0 = 0; t0 < nb; t0 += TB) {
    const int nstage = TB * NP * CT;
    for (int e = tid; e < nstage; e += nthreads) {
      int c = e % CT;
      int a = (e / CT) % NP;
      int tt = e / (CT * NP);
      float2 v = make_float2(0.f, 0.f);
      if (a < A.nin && t0 + tt < nb && c0 + c < A.nchan)
        v = load_spec(spec, A.in_off[a] + (long long)(sb0 + t0 + tt) * A.block_stride + cidx(c0 + c, A.gstride));
      sh[e] = v;
    }
    __syncthreads();
    if (active) {
      const int nt = min(TB, nb - t0);
      for (int tt = 0; tt < nt; tt++) {
        const float2* row = sh + (long long)tt * NP * CT;
        float2 xb[8];
#pragma unroll
        for (int k = 0; k < 8; k++) xb[k] = row[(tb * 8 + k) * CT + cl];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          float2 xa = row[(ta * 8 + i) * CT + cl];
#pragma unroll
          for (int k = 0; k < 8; k++) {
            acc[i][k].x += xa.x * xb[k].x + xa.y * xb[k].y;
            acc[i][k].y += xa.y * xb[k].x - xa.x * xb[k].y;
          }
        }
      }
    }
    __syncthreads();
  }
  if (!active || c0 + cl >= A.nchan) return;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    int a = ta * 8 + i;
    if (a >= A.nin) continue;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      int b = tb * 8 + k;
      if (b >= A.nin) continue;
      float2* p = Vout + ((long long)a * A.nin + b) * A.nchan + c0 + cl;
      if (A.accumulate) { float2 o = *p; o.x += acc[i][k].x; o.y += acc[i][k].y; *p = o; }
      else *p = acc[i][k];
    }
  }
}

// ---------------------------------------------------------------------------
// weights: per weight table entry the sum over blocks of w1*w2 (a baseline
// product) or of w1 (an autocorrelation), each added in block order; w is a
// recorded band's weight on INTERLACEDVDIF datastreams, else the block's
// data weight
// ---------------------------------------------------------------------------
// acc + 1 + ... + 1 (n ones) in FP32, each addition rounded.  One addition of m
// of them rounds the same where acc is whole, or at least m, and the sum stays
// below 2^22: then at most one binade is crossed, and an integer added after its
// rounding moves no tie, a spacing there being a quarter or less.
__device__ __forceinline__ float add_ones(float acc, int n) {
  while (n > 0) {
    int m = 1;
    if (acc + (float)n < 4194304.0f) m = acc == truncf(acc) ? n : min(n, max(1, (int)acc));
    acc += (float)m;
    n -= m;
  }
  return acc;
}

// An entry's terms of N blocks a thread, STEP apart: both sides' weights are loaded
// together (bw, negative where a block was not processed, and the band's own in
// its place) and multiplied when they are used.  The weights come from their own
// array: out of the 80-byte block records the lines alone took a CU 100 us.
template <int N, int STEP>
struct WeightTerms {
  static constexpr bool few = STEP == 64;          // loads wholly past the last block are left out
  const DevWTerm T;
  const float *bw1, *bw2, *own1, *own2;
  int nchan1, nchan2;
  const int nblocks, at;
  float w1[N], w2[N], o1[N], o2[N];
  __device__ __forceinline__ WeightTerms(const DevStation* st, const DevStationSub* ss, const float* bw, int nblocks,
                                         const DevWTerm& T, int at)
      : T(T), nblocks(nblocks), at(at) {
    bw1 = bw + (long long)T.d1 * nblocks;
    if (T.b1 >= 0) { own1 = ss[T.d1].pbw + T.b1; nchan1 = st[T.d1].nchan; }
    if (T.d2 < 0) return;
    bw2 = bw + (long long)T.d2 * nblocks;
    if (T.b2 >= 0) { own2 = ss[T.d2].pbw + T.b2; nchan2 = st[T.d2].nchan; }
  }
  __device__ __forceinline__ void side(int t0, const float* src, bool band, const float* own, int nchan, float (&w)[N],
                                       float (&o)[N]) {
#pragma unroll
    for (int q = 0; q < N; q++)
      if (!few || t0 + q * STEP < nblocks) w[q] = src[min(t0 + q * STEP + at, nblocks - 1)];
    if (!band) return;
#pragma unroll
    for (int q = 0; q < N; q++)
      if (!few || t0 + q * STEP < nblocks) o[q] = own[(long long)min(t0 + q * STEP + at, nblocks - 1) * nchan];
  }
  __device__ __forceinline__ void load(int t0) {
    side(t0, bw1, T.b1 >= 0, own1, nchan1, w1, o1);
    if (T.d2 >= 0) side(t0, bw2, T.b2 >= 0, own2, nchan2, w2, o2);
  }
  __device__ __forceinline__ float term(int t0, int q) const {
    if (t0 + q * STEP + at >= nblocks) return 0.0f;
    const float x = w1[q] < 0.0f ? 0.0f : T.b1 >= 0 ? o1[q] : w1[q];
    if (T.d2 < 0) return x;
    return x * (w2[q] < 0.0f ? 0.0f : T.b2 >= 0 ? o2[q] : w2[q]);
  }
};

// acc + 64 terms in order, read together beforehand
struct Terms64 {
  float4 t[16];
  __device__ __forceinline__ explicit Terms64(const float* p) {
#pragma unroll
    for (int j = 0; j < 16; j++) t[j] = ((const float4*)p)[j];
  }
  __device__ __forceinline__ float add(float acc) const {
#pragma unroll
    for (int j = 0; j < 16; j++) {
      acc += t[j].x;
      acc += t[j].y;
      acc += t[j].z;
      acc += t[j].w;
    }
    return acc;
  }
};

// The sums are FP32 in block order, a serial chain (the reference's rounding), but
// in most streams nearly every term is 0 or 1: terms are sorted into masks by 64,
// the ones of many groups are added at once, and a group with any other term is
// added in order (odd term by odd term took twice as long as one addition at a
// time where most are odd).  The next terms load meanwhile.
//   k_weights: a workgroup an entry, 4096 terms at a time, for long sums of few
// entries; bound by the one wavefront that adds.  20000 blocks, against one
// addition at a time: all ones 144 -> 15 us, a fifth of short frames lost 140 ->
// 75, bands blanked in every third (INTERLACEDVDIF) 150 -> 80.
//   k_weights_w: a wavefront an entry, 512 terms at a time, for up to 1024 blocks,
// where the other's barriers and empty wavefronts cost more (9 stations of 16
// bands, INTERLACEDVDIF, 300 blocks 18 us, this 9), and for more than 1024
// entries, where four times as many fit the chip (2000 blocks 36 and 23; 9
// stations of 4 bands 15 and 18).
__global__ __launch_bounds__(256) void k_weights(const DevStation* __restrict__ st,
                                                 const DevStationSub* __restrict__ ss,
                                                 const float* __restrict__ bw, int nblocks,
                                                 const DevWTerm* __restrict__ terms, int nterms,
                                                 float* __restrict__ wout) {
  constexpr int CH = 4096, PER = CH / 256;
  __shared__ __align__(16) float term[CH];
  __shared__ unsigned long long ones[CH / 64], odd[CH / 64];
  const int i = blockIdx.x;
  if (i >= nterms) return;
  const int lane = threadIdx.x & 63;
  WeightTerms<PER, 256> W(st, ss, bw, nblocks, terms[i], threadIdx.x);
  float acc = 0.0f;
  W.load(0);
  for (int t0 = 0; t0 < nblocks; t0 += CH) {
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int k = q * 256 + threadIdx.x;
      const float x = W.term(t0, q);
      term[k] = x;
      const unsigned long long o = __ballot(x == 1.0f), z = __ballot(x != 0.0f) & ~o;
      if (lane == 0) { ones[k >> 6] = o; odd[k >> 6] = z; }
    }
    __syncthreads();
    if (t0 + CH < nblocks) W.load(t0 + CH);
    if (threadIdx.x < 64) {
      const int own = __popcll(ones[lane]);
      int n = own;
      unsigned long long mixed = __ballot(odd[lane] != 0ull);
      // the ones before group g are added together, then its terms in order
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(n, d);
        if (lane >= d) n += u;
      }
      int done = 0;
      while (mixed) {
        const int g = __builtin_ctzll(mixed);
        mixed &= mixed - 1ull;
        const Terms64 t(term + 64 * g);
        const int upto = __builtin_amdgcn_readlane(n, g);
        acc = t.add(add_ones(acc, upto - __builtin_amdgcn_readlane(own, g) - done));
        done = upto;
      }
      acc = add_ones(acc, __builtin_amdgcn_readlane(n, 63) - done);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) wout[i] = acc;
}

constexpr int kWeightWaves = 4;                    // entries of a workgroup of k_weights_w

__global__ __launch_bounds__(64 * kWeightWaves) void k_weights_w(const DevStation* __restrict__ st,
                                                                 const DevStationSub* __restrict__ ss,
                                                                 const float* __restrict__ bw, int nblocks,
                                                                 const DevWTerm* __restrict__ terms, int nterms,
                                                                 float* __restrict__ wout) {
  constexpr int NG = 8;
  __shared__ __align__(16) float lds[kWeightWaves][64 * NG];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = blockIdx.x * kWeightWaves + wave;
  if (i >= nterms) return;                         // the whole wavefront; no barrier below
  WeightTerms<NG, 64> W(st, ss, bw, nblocks, terms[i], lane);
  float* const term = lds[wave];
  float acc = 0.0f;
  W.load(0);
  for (int t0 = 0; t0 < nblocks; t0 += 64 * NG) {
    unsigned long long one[NG], odd[NG], any = 0ull;
#pragma unroll
    for (int q = 0; q < NG; q++) {
      const float x = W.term(t0, q);
      term[q * 64 + lane] = x;
      one[q] = __ballot(x == 1.0f);
      odd[q] = __ballot(x != 0.0f) & ~one[q];
      any |= odd[q];
    }
    if (t0 + 64 * NG < nblocks) W.load(t0 + 64 * NG);
    // a wavefront's own LDS accesses complete in order: this orders the compiler's
    auto order = [] {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    int n = 0;                                     // ones not yet added
    if (any != 0ull) order();
#pragma unroll
    for (int q = 0; q < NG; q++) {
      if (odd[q] == 0ull) {
        n += __popcll(one[q]);
        continue;
      }
      const Terms64 t(term + 64 * q);
      acc = t.add(add_ones(acc, n));
      n = 0;
    }
    if (any != 0ull) order();
    acc = add_ones(acc, n);
  }
  if (lane == 0) wout[i] = acc;
}

// ---------------------------------------------------------------------------
// scatter: result[seg.resoff + c] = mean of V[seg.voff + c avg + i], i < avg
// (conjugated if flagged), scaled by vscale; float segments copy one weight;
// zero segments clear what nothing else writes
// ---------------------------------------------------------------------------
constexpr int kScatterPer = 4;   // channels per thread (their loads in flight together)

__global__ __launch_bounds__(256) void k_scatter(const DevSeg* __restrict__ segs, int nseg,
                                                 const float2* __restrict__ V, const float* __restrict__ w,
                                                 float vscale, float* __restrict__ res) {
  int sidx = blockIdx.y;
  if (sidx >= nseg) return;
  const DevSeg g = segs[sidx];
  const int cb = blockIdx.x * (256 * kScatterPer) + threadIdx.x;
  if (g.kind == SEG_FLOATS) {
    if (cb == 0) res[g.resoff] = w[g.voff];
    return;
  }
  if (g.kind == SEG_ZERO) {
#pragma unroll
    for (int q = 0; q < kScatterPer; q++)
      if (cb + q * 256 < g.nchan) res[g.resoff + cb + q * 256] = 0.0f;
    return;
  }
  if (cb >= g.nchan) return;
  float2 v[kScatterPer];
  if (g.avg == 1) {
#pragma unroll
    for (int q = 0; q < kScatterPer; q++) {
      const int c = cb + q * 256;
      v[q] = c < g.nchan ? V[g.voff + c] : make_float2(0.0f, 0.0f);
    }
  } else {
    // vectorMean_cf32 of the group: sum in channel order, then divide
#pragma unroll
    for (int q = 0; q < kScatterPer; q++) {
      const int c = cb + q * 256;
      v[q] = make_float2(0.0f, 0.0f);
      if (c >= g.nchan) continue;
      const float2* p = V + g.voff + (long long)c * g.avg;
      for (int i = 0; i < g.avg; i++) { v[q].x += p[i].x; v[q].y += p[i].y; }
      v[q].x /= (float)g.avg;
      v[q].y /= (float)g.avg;
    }
  }
  const bool al8 = (reinterpret_cast<unsigned long long>(res) & 7) == 0;
#pragma unroll
  for (int q = 0; q < kScatterPer; q++) {
    const int c = cb + q * 256;
    if (c >= g.nchan) break;
    float2 y = v[q];
    if (g.conj) y.y = -y.y;
    if (al8) {
      reinterpret_cast<float2*>(res)[g.resoff + c] = make_float2(y.x * vscale, y.y * vscale);   // one 8-byte store
    } else {
      res[2 * (g.resoff + c)] = y.x * vscale;
      res[2 * (g.resoff + c) + 1] = y.y * vscale;
    }
  }
}

hipError_t launch_xmac_f32(const XmacArgs& a, int prec, hipStream_t stream) {
  size_t shmem = (size_t)a.TB * a.G * 8 * a.CT * sizeof(float2);
  dim3 grid((unsigned)((a.nchan + a.CT - 1) / a.CT), (unsigned)((a.nblocks + a.split_blocks - 1) / a.split_blocks));
  int threads = a.CT * a.ntiles;
  threads = ((threads + 63) / 64) * 64;
  if (threads > 576) return hipErrorInvalidValue;
  if (prec == FXG_XMAC_FP32) hipLaunchKernelGGL(k_xmac_f32<float2>, grid, dim3(threads), shmem, stream, a);
  else if (prec == FXG_XMAC_FP16) hipLaunchKernelGGL(k_xmac_f32<__half2>, grid, dim3(threads), shmem, stream, a);
  else hipLaunchKernelGGL(k_xmac_f32<__hip_bfloat162>, grid, dim3(threads), shmem, stream, a);
  return hipGetLastError();
}

// V (+)= sum_s P[s*vsplit + .], V [nin][nin][nchan]: the partial sums
// of block ranges, of the input pairs a <= b that are read, added in
// split order so that the result does not depend on scheduling, eight loads in
// flight.  14 inputs, 256 channels, 32 rows 33 us -> 11.
__global__ __launch_bounds__(256) void k_xmac_reduce(const float2* __restrict__ P, int nsplit, long long vsplit,
                                                     float2* __restrict__ V, unsigned nin, unsigned nchan, long long n,
                                                     int accumulate) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const unsigned q = (unsigned)(i / nchan);
  if (q / nin > q % nin) return;
  float2 acc = accumulate ? V[i] : make_float2(0.f, 0.f);
  for (int s0 = 0; s0 < nsplit; s0 += 8) {
    float2 p[8];
#pragma unroll
    for (int s = 0; s < 8; s++) p[s] = s0 + s < nsplit ? P[(long long)(s0 + s) * vsplit + i] : make_float2(0.f, 0.f);
#pragma unroll
    for (int s = 0; s < 8; s++) {
      acc.x += p[s].x;
      acc.y += p[s].y;
    }
  }
  V[i] = acc;
}

hipError_t launch_xmac_reduce(const float2* P, int nsplit, long long vsplit, float2* V, int nin, int nchan,
                              int accumulate, hipStream_t stream) {
  const long long n = (long long)nin * nin * nchan;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_xmac_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, P, nsplit, vsplit, V,
                     (unsigned)nin, (unsigned)nchan, n, accumulate);
  return hipGetLastError();
}

// p[i] = 0 for i < n: four floats per thread where aligned
__global__ __launch_bounds__(256) void k_zero(float* __restrict__ p, long long n) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 3 < n && ((uintptr_t)(p + i) & 15) == 0) {
    *(float4*)(p + i) = make_float4(0.f, 0.f, 0.f, 0.f);
  } else {
    for (long long k = i; k < n && k < i + 4; k++) p[k] = 0.0f;
  }
}

hipError_t launch_zero(float* p, long long n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  const long long blocks = (n + 1023) / 1024;
  hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, stream, p, n);
  return hipGetLastError();
}

hipError_t launch_weights(const DevStation* st, const DevStationSub* ss, const float* bw, int nblocks,
                          const DevWTerm* terms, int nterms, float* w, hipStream_t stream) {
  if (nterms == 0) return hipSuccess;
  if (nblocks > 1024 && nterms <= 1024)
    hipLaunchKernelGGL(k_weights, dim3(nterms), dim3(256), 0, stream, st, ss, bw, nblocks, terms, nterms, w);
  else
    hipLaunchKernelGGL(k_weights_w, dim3((nterms + kWeightWaves - 1) / kWeightWaves), dim3(64 * kWeightWaves), 0, stream, st,
                       ss, bw, nblocks, terms, nterms, w);
  return hipGetLastError();
}

hipError_t launch_scatter(const DevSeg* segs, int nseg, int maxlen, const float2* V, const float* w, float vscale,
                          float* res, hipStream_t stream) {
  if (nseg == 0) return hipSuccess;
  int blocks = (maxlen + 256 * kScatterPer - 1) / (256 * kScatterPer);
  if (blocks < 1) blocks = 1;
  // grid.y is limited to 65535: launch in slices
  for (int s0 = 0; s0 < nseg; s0 += 65535) {
    int n = nseg - s0 < 65535 ? nseg - s0 : 65535;
    hipLaunchKernelGGL(k_scatter, dim3(blocks, n), dim3(256), 0, stream, segs + s0, n, V, w, vscale, res);
  }
  return hipGetLastError();
}

}  // namespace fxg
