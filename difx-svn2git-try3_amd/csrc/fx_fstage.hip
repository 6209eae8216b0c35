// fx_fstage.hip — the F stage with linear (real samples: or post-F) fringe
// rotation (mode.cpp:909-1310): level decoding, fringe rotation, FFT, sideband
// select, fractional-sample rotation.
#include <hip/hip_runtime.h>
#include "fx_kernels.h"
#include "fx_device.h"
#include "fx_fft.h"
#include "fx_place.h"
#include "fx_spectra.h"
#include <cmath>
#include <vector>

namespace fxg {

// The passes of one length L = PW x M: PW workgroups share a block above 8192
// points, each transforming M points to the bins k = PW k' + pw.  M = R1 x
// (16) x RL: R1 = 16 P in the first pass, 16 in a middle one from 2048 points
// on, RL = 16 or 8 in the last; NTF threads a block and NB blocks per
// workgroup of NT threads; the per-block table (pass 1: CP entries for each of
// the P thread sets; the last pass's four powers and the eight channel steps;
// eight twiddles for each bin of the middle pass).
template <int L> struct FsShape {
  static constexpr int M = L > 8192 ? 8192 : L, PW = L / M;
  static constexpr int LOG = M == 128 ? 7 : M == 256 ? 8 : M == 512 ? 9 : M == 1024 ? 10 : M == 2048 ? 11
                           : M == 4096 ? 12 : 13;
  static constexpr int P = LOG % 4 == 1 ? 2 : LOG % 4 == 2 ? 4 : 1;
  static constexpr int R1 = 16 * P, J1 = M / R1, RL = LOG % 4 == 3 ? 8 : 16;
  static constexpr bool MID = LOG >= 11;
  static constexpr int J2 = MID ? J1 / 16 : 16;
  static constexpr int NTF = M / 16, NB = NTF >= 128 ? 1 : 256 / NTF, NT = NTF * NB;
  static constexpr int CP = PW > 1 || P == 4 ? 12 : P == 2 ? 10 : 8, LAST = P * CP, MIDOFF = LAST + 12;
  static constexpr int NE = MIDOFF + (MID ? 8 * R1 : 0);
  static constexpr bool TWO = MID && PW == 1;                  // takes two bands of one rotation
  // PW > 1: quads of one first-pass input, and tables of quad sums
  static constexpr int QSUM = P * PW / 4, NSUM = PW == 1 ? 0 : PW == 2 ? 2 : 1;
};

// Validity of the 32 / BITS consecutive samples from t of one band, one bit
// each (the rule of sample_value: frames by their valid byte range, blanked
// bands, validend, the end of the data)
template <int COUNT>
__device__ __forceinline__ unsigned valid_samples(const DevStation& S, const DevStationSub& Q,
                                                  const int2* __restrict__ ftab, long long t, long long validend,
                                                  int band) {
  // sample numbers are below 2^31 + L, so 32-bit divisions do (3 bands of 65536 8-bit
  // points, five blocks of a lossy stream 49 -> 45 us)
  unsigned m = 0u;
  if (t < 0 || t >= validend) return m;
  const unsigned first = (unsigned)t, end = (unsigned)min(t + COUNT, validend), fs = (unsigned)S.framesamples;
  for (unsigned u = first; u < end;) {
    const unsigned f = u / fs, base = f * fs, fe = min(end, base + fs);
    if ((long long)f >= Q.nframes) break;
    const int2 z = ftab[Q.fbase + f];
    const bool blank = Q.fblank && ((Q.fblank[f] >> band) & 1ull);
    if (z.x < z.y && !blank) {
      const unsigned gb = (unsigned)S.groupbytes, gs = (unsigned)S.groupsamples;
      const unsigned g0 = ((unsigned)min(z.x, S.databytes) + gb - 1) / gb;
      const unsigned g1 = ((unsigned)min(z.y, S.databytes) + gb - 1) / gb;
      const unsigned a = max(u, base + g0 * gs), b = min(fe, base + g1 * gs);
      if (b > a) m |= ((1u << (b - a)) - 1u) << (a - first);
    }
    u = fe;
  }
  return m;
}

// 16 bits to 16 two-bit fields (each bit doubled)
__device__ __forceinline__ unsigned double_bits16(unsigned m) {
  m = (m | (m << 8)) & 0x00FF00FFu;
  m = (m | (m << 4)) & 0x0F0F0F0Fu;
  m = (m | (m << 2)) & 0x33333333u;
  m = (m | (m << 1)) & 0x55555555u;
  return m * 3u;
}

// Four rows of 16 two-bit samples to quads: byte m of a[t] becomes the four
// rows' sample 4 m + t, row 0 in the low bits.
__device__ __forceinline__ void quads2(unsigned* a) {
  unsigned t;
  t = ((a[0] >> 2) ^ a[1]) & 0x33333333u; a[1] ^= t; a[0] ^= t << 2;
  t = ((a[2] >> 2) ^ a[3]) & 0x33333333u; a[3] ^= t; a[2] ^= t << 2;
  t = ((a[0] >> 4) ^ a[2]) & 0x0F0F0F0Fu; a[2] ^= t; a[0] ^= t << 4;
  t = ((a[1] >> 4) ^ a[3]) & 0x0F0F0F0Fu; a[3] ^= t; a[1] ^= t << 4;
}
// Four rows of four bytes to quads: byte i of a[t] becomes row i's byte t.
__device__ __forceinline__ void quads8(unsigned* a) {
  const unsigned lo01 = __builtin_amdgcn_perm(a[1], a[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(a[1], a[0], 0x07030602u);
  const unsigned lo23 = __builtin_amdgcn_perm(a[3], a[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(a[3], a[2], 0x07030602u);
  a[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
  a[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
  a[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
  a[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
}

// x0 + g1 x1 + g2 x2 + g3 x3
__device__ __forceinline__ float2 quad_sum(const float4& x, float2 g1, float2 g2, float2 g3) {
  return make_float2(__builtin_fmaf(g3.x, x.w, __builtin_fmaf(g2.x, x.z, __builtin_fmaf(g1.x, x.y, x.x))),
                     __builtin_fmaf(g3.y, x.w, __builtin_fmaf(g2.y, x.z, g1.y * x.y)));
}

// ---------------------------------------------------------------------------
// k_fstage_lin<L, NBITS>: 16 points per thread in every pass.
//
// What bounds it: FP32 VALU issue (wave64, four cycles an instruction; 73 to 89 %
// of the cycles, at 65536 points 77 % beside 60 % of LDS), so it is built for few
// instructions:
//   - the fringe rotation is in the twiddles (fx_fft.h), whose per-block
//     values are two dozen to 60 sines of FP64 phases, one per thread;
//   - the first pass reads samples as quads, the four samples a quarter of
//     the block apart, whose first two butterfly stages have real inputs: one
//     LDS byte and one 16-byte lookup decode four samples;
//   - R1 = 16 P: pass 1 has radix 32 or 64 where L is an odd power of two or
//     four times a power of 16, P threads sharing one input set (each forms
//     the outputs q = P q' + p), so that no length but 8 x 16^n needs a pass
//     of smaller radix: two LDS exchanges at 2048 points and more, one below;
//   - the last pass forms only the sideband's half of the outputs (the lower
//     sideband's sign rides on w);
//   - above 8192 points PW workgroups share a block, so that two still fit a
//     CU and one's LDS phases run under the other's arithmetic.  A thread's
//     first-pass inputs are then sums of QSUM quads with fixed weights, x0 +
//     g x1 + g^2 x2 + g^3 x3 by the quad's byte from a table that the
//     workgroup forms once (g is the same for all its threads, or for every
//     other set).  Every workgroup decodes the whole block, and nothing goes
//     through memory between the passes.  The PW workgroups of a block run
//     side by side on one XCD, whose L2 merges their interleaved channels
//     into lines.  One workgroup of 1024 threads and 16384 points a CU instead
//     left the VALU idle half of the time (16384 points 18.4 ms, 65536 points
//     28.0 ms on the workloads below).
//   - from 2048 to 8192 points a workgroup takes both polarisations of a
//     frequency, which share the rotation: its table, the last pass's twiddles
//     and the channel rotators are formed once, and the second band's samples
//     are in registers when the first is done.
// (Tried and dropped: the first-stage outputs by the quad's byte from a table
// per workgroup, 8192 points: 803 -> 746 VALU instructions a band, 25.2 -> 25.0
// ms, the VALU 84 % busy instead of 90 %: what is left is the barriers that two
// workgroups a CU do not cover.)
// Exchanges are laid out so that both sides hit all banks with immediate
// offsets: the one into the middle pass by exchanging pieces of J2 values
// between neighbouring rows, the one into the last pass by a row pad.
// Against the kernels with rotator tables and padded twiddle products, one
// radix-2 pass more, and from 32768 points a scratch in HBM between two kernels
// (rocprofv3, ms): 8192 points, 16.8 Gsamples 33.4 -> 25.2; 16384 points, 8.2
// Gsamples 24.0 -> 14.5; 65536 points, 7.9 Gsamples 37.5 -> 23.2; 2048 points,
// 1.34 Gsamples 3.23 -> 2.40; 512 points, 8-bit, 0.92 Gsamples 3.53 -> 1.29.
// ---------------------------------------------------------------------------
template <int L, int NBITS>
__global__ __launch_bounds__(FsShape<L>::NT, 4) void k_fstage_lin(FStageArgs A) {
  using Sh = FsShape<L>;
  constexpr int M = Sh::M, PW = Sh::PW;
  constexpr int P = Sh::P, R1 = Sh::R1, J1 = Sh::J1, J2 = Sh::J2, RL = Sh::RL, NTF = Sh::NTF, NB = Sh::NB, NT = Sh::NT;
  constexpr bool MID = Sh::MID;
  constexpr int QW = NBITS == 8 ? L / 4 : L / 16;         // staged quad words of one block
  constexpr int NL = M / RL, LPAD = 32 / RL;               // bins entering the last pass, and its row pad
  // The quads lie in the exchange buffer where a block is within one
  // wavefront (read before that wavefront's first exchange write) and where
  // PW workgroups share a block (a barrier between).
  constexpr bool RAWOWN = PW == 1 && (NTF > 64 || NTF < 32);
  struct Smem {
    float2 tab[NB][Sh::NE];
    float4 quad[NBITS == 2 && PW == 1 ? 256 : 0];
    float2 sums[NBITS == 2 ? 256 * Sh::NSUM : 0];
    unsigned raw_own[RAWOWN ? NB * QW : 0];
    unsigned ok_own[RAWOWN && NBITS == 2 ? NB * QW : 0];
    float2 buf[NB][M + 32 + (NTF < 32 ? 1 : 0)];
  };
  __shared__ __align__(16) Smem sm;

  const int tid = threadIdx.x;
  const int fi = NB == 1 ? 0 : tid / NTF, t = NB == 1 ? tid : tid % NTF;
  unsigned* const raw = RAWOWN ? sm.raw_own + fi * QW : (unsigned*)sm.buf[fi];
  unsigned* const ok = RAWOWN ? sm.ok_own + fi * QW : (unsigned*)sm.buf[fi] + QW;
  // this workgroup's bands and group of blocks within the chunk
  const FsPlace place = fstage_place(blockIdx.x, blockIdx.y, gridDim.x, (unsigned)(A.nchunk + NB - 1) / NB, PW);
  if (place.row >= (unsigned)A.nrows || place.grp * NB >= (unsigned)A.nchunk) return;
  const int pw = PW == 1 ? 0 : place.pw;
  const int cbx = place.grp * NB + fi;
  const bool mine = NB == 1 || cbx < A.nchunk;
  const int cb = mine ? cbx : A.nchunk - 1;
  // one band, or two that share a rotation (the polarisations of a frequency)
  const int2 pair = A.pairs[place.row];
  const int nband = Sh::TWO && pair.y >= 0 ? 2 : 1;
  const DevBand& B0 = A.bands[pair.x];
  const DevBand& B1 = A.bands[nband == 2 ? pair.y : pair.x];
  const DevStationSub& Q = A.ss[B0.station];
  const DevRot& R = A.rots[(long long)B0.rot * A.nblocks_subint + A.chunk0 + cb];
  constexpr int C = L / 2;
  const bool dead = R.status != 0;
  if (NB == 1 && dead) {
    for (int b = 0; b < nband && pw == 0; b++)
      zero_spec(A.spectra, A.prec, (b ? B1 : B0).specoff + (long long)cb * A.bstride, C, A.gstride, tid, NT);
    return;
  }

  // ---- the block's samples of a band: four rows a quarter block apart, their
  // first loads (and the second band's) in flight under the tables' sines
  constexpr int GROUPS = NBITS == 8 ? L / 16 : L / 64;
  const bool fast = R.allvalid != 0 || dead;
  const long long bit0 = (long long)(dead ? 0 : R.t0) * NBITS;
  const long long nwords = Q.ctstride >> 2;
  constexpr int NIT = (GROUPS + NTF - 1) / NTF, AHEAD = NIT > 2 ? 2 : NIT;
  unsigned lo[AHEAD][4], hi[AHEAD][4], lo1[4], hi1[4];
  auto load_rows = [&](const DevBand& B, int g, unsigned (&lo)[4], unsigned (&hi)[4]) {
    const unsigned* src = (const unsigned*)(A.ct + Q.ctbase + (long long)B.band * Q.ctstride);
    const long long w0 = (bit0 >> 5) + g;
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const long long w = w0 + m * GROUPS;
      lo[m] = w < nwords ? src[w] : 0u;
      hi[m] = w + 1 < nwords ? src[w + 1] : 0u;
    }
  };
  auto store_quads = [&](const DevBand& B, int g, const unsigned (&lo)[4], const unsigned (&hi)[4]) {
    unsigned a[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
      a[m] = __builtin_amdgcn_alignbit(hi[m], lo[m], (int)(bit0 & 31));
      if (NBITS == 8) a[m] ^= 0x80808080u;                 // signed levels, 0 = none
    }
    if (!fast) {
      // a blanked sample has no 2-bit code: its validity is staged beside it;
      // 8-bit samples are cleared
      const DevStation& S = A.st[B.station];
      unsigned v[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const long long ts = R.t0 + (long long)(m * GROUPS + g) * (32 / NBITS);
        v[m] = valid_samples<32 / NBITS>(S, Q, A.ftab, ts, R.validend, B.band);
        if (NBITS == 2) {
          v[m] = double_bits16(v[m]);
        } else {
          const unsigned by = ((v[m] & 1u) | ((v[m] & 2u) << 7) | ((v[m] & 4u) << 14) | ((v[m] & 8u) << 21)) * 255u;
          a[m] &= by;
        }
      }
      if (NBITS == 2) {
        quads2(v);
        *(uint4*)&ok[4 * g] = make_uint4(v[0], v[1], v[2], v[3]);
      }
    }
    if (NBITS == 8) quads8(a); else quads2(a);
    *(uint4*)&raw[4 * g] = make_uint4(a[0], a[1], a[2], a[3]);
  };
  auto load_ahead = [&](const DevBand& B, int i0) {
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
      if (t + (i0 + i) * NTF < GROUPS) load_rows(B, t + (i0 + i) * NTF, lo[i], hi[i]);
  };
  // the quads of a band whose first loads are in lo, hi
  auto stage = [&](const DevBand& B) {
#pragma unroll
    for (int i0 = 0; i0 < NIT; i0 += AHEAD) {
      if (i0 > 0) load_ahead(B, i0);
#pragma unroll
      for (int i = 0; i < AHEAD; i++)
        if (t + (i0 + i) * NTF < GROUPS) store_quads(B, t + (i0 + i) * NTF, lo[i], hi[i]);
    }
  };
  static_assert(!Sh::TWO || (NIT == 1 && RAWOWN), "the second band's rows are one round, into the first's place");
  load_ahead(B0, 0);
  if (Sh::TWO && t < GROUPS) load_rows(B1, t, lo1, hi1);
  float4 level;                                            // of quad byte tid % 256, for the tables below
  if (NBITS == 2 && PW > 1) level = A.quad[B0.levels * 256 + (tid & 255)];
  // ---- this block's twiddles and fractional-sample steps
  {
    const double delta = R.delta, theta = R.theta;
    for (int i = NTF - 1 - t; i < Sh::NE; i += NTF) {
      const float4 d = A.cdesc[i];
      double ph = theta * (double)d.y - (delta * (double)d.x + (double)d.z);
      if (PW > 1) ph -= (double)pw * (double)d.w;
      if (i == Sh::LAST + 3 && B0.lsb) ph += 0.5;           // the lower sideband keeps a - w b
      sm.tab[fi][i] = exact_rotator(ph);
    }
  }
  if (NBITS == 2 && PW == 1)
    for (int i = tid; i < 256; i += NT) sm.quad[i] = A.quad[B0.levels * 256 + i];
  stage(B0);
  __syncthreads();
  if (NBITS == 2 && PW > 1) {
    if (tid < 256 * Sh::NSUM) {
      const float2* g = sm.tab[0] + (tid >> 8) * Sh::CP + 9;
      sm.sums[tid] = quad_sum(level, g[0], g[1], g[2]);
    }
    __syncthreads();
  }

  // workgroup barrier, or (a block's threads within one wavefront) only an
  // order for the compiler: LDS accesses of a wavefront complete in order
  auto sync = [] {
    if (NTF > 64) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };
  float2* const buf = sm.buf[fi];
  const float2* const tab = sm.tab[fi];

  // ---- what two bands share: the last pass's twiddles and the rotation of
  // channel PW (t + e M/16) + pw, this thread's phase (FP64, in turns) times
  // E[e]; for one band both are formed where they are used, for registers
  const float2* const cl = tab + Sh::LAST;
  constexpr int NW = RL == 16 ? 4 : 6;
  float2 w[NW], F, FE[8];
  auto last_powers = [&] {
#pragma unroll
    for (int i = 0; i < NW; i++) w[i] = cmulx(A.base[i * NTF + t], cl[RL == 16 ? i : 1 + i / 2]);
  };
  auto channel_phase = [&] {
    const float s = dead ? 0.0f : (NBITS == 8 ? A.scale * (float)(1.0 / 3.3) : A.scale);
    F = exact_rotator(R.phase + R.theta * (double)(PW * t + pw));
    F = make_float2(F.x * s, F.y * s);
  };
  if (Sh::TWO) {
    last_powers();
    channel_phase();
#pragma unroll
    for (int e = 0; e < 8; e++) FE[e] = cmulx(F, cl[4 + e]);
  }

#pragma unroll 1
  for (int band = 0; band < (Sh::TWO ? nband : 1); band++) {
  const DevBand& B = band ? B1 : B0;
  // what a pass derives from the thread's number and its twiddles is formed
  // anew for each band: kept over the loop it would not fit the registers
  int tl = t;
  if (Sh::TWO) asm volatile("" : "+v"(tl));
  __builtin_assume(tl >= 0 && tl < NTF);
  auto fresh = [](float2 w) {
    if (Sh::TWO) asm volatile("" : "+v"(w.x), "+v"(w.y));
    return w;
  };
  // ---- pass 1: decode, radix R1 (this thread's 16 of the R1 outputs)
  {
    const int p = tl / J1, j = tl % J1;
    const float2* c = tab + p * Sh::CP;
    Tw16 w;
    w.w8 = c[0]; w.w4 = c[1]; w.w2 = c[2]; w.w2h = c[3]; w.w1 = c[4]; w.w1a = c[5]; w.w1b = c[6]; w.w1c = c[7];
    // Quads of samples j + r J1, QN at a time, all their LDS reads in flight
    // together: bytes within a group of 16 in the order of quads2.
    constexpr int QN = P == 1 && PW == 1 ? 4 : 8;
    auto quads_at = [&](int r0, float4* x) {                // r0 + r counts J1 samples
      if (NBITS == 8) {
        unsigned q[QN];
#pragma unroll
        for (int r = 0; r < QN; r++) q[r] = raw[j + (r0 + r) * J1];
#pragma unroll
        for (int r = 0; r < QN; r++)
          x[r] = make_float4((float)(signed char)(q[r] & 0xFFu), (float)(signed char)((q[r] >> 8) & 0xFFu),
                             (float)(signed char)((q[r] >> 16) & 0xFFu), (float)(signed char)(q[r] >> 24));
      } else {
        const int at0 = J1 >= 16 ? (j & ~15) + ((j & 3) << 2) + ((j >> 2) & 3) : ((j & 3) << 2) + (j >> 2);
        auto at = [&](int r) { return at0 + (J1 >= 16 ? r * J1 : 16 * (r >> 1) + 2 * (r & 1)); };
        unsigned q[QN];
#pragma unroll
        for (int r = 0; r < QN; r++) q[r] = ((const unsigned char*)raw)[at(r0 + r)];
#pragma unroll
        for (int r = 0; r < QN; r++) x[r] = PW == 1 ? sm.quad[q[r]] : A.quad[B.levels * 256 + q[r]];
        if (!fast) {
#pragma unroll
          for (int r = 0; r < QN; r++) {
            const unsigned m = ((const unsigned char*)ok)[at(r0 + r)];
            x[r].x = m & 1u ? x[r].x : 0.0f;
            x[r].y = m & 4u ? x[r].y : 0.0f;
            x[r].z = m & 16u ? x[r].z : 0.0f;
            x[r].w = m & 64u ? x[r].w : 0.0f;
          }
        }
      }
    };
    float2 v[16];
    if (PW > 1) {
      // QSUM quads 16 J1 samples apart, the later ones times powers of c[8]
      constexpr int QS = PW > 1 ? Sh::QSUM : 1;
      const float2 g1 = c[9], g2 = c[10], g3 = c[11], w1 = c[8];
      if (NBITS == 2 && fast) {
        const float2* sums = sm.sums + (p % (PW > 1 ? Sh::NSUM : 1)) * 256;
        const unsigned char* q0 = (const unsigned char*)raw + (j & ~15) + ((j & 3) << 2) + ((j >> 2) & 3);
#pragma unroll
        for (int h = 0; h < 4; h++) {
          unsigned q[4 * QS];
#pragma unroll
          for (int i = 0; i < 4 * QS; i++) q[i] = q0[(4 * h + i / QS + 16 * (i % QS)) * J1];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            float2 x = sums[q[r * QS + QS - 1]];
#pragma unroll
            for (int m = QS - 2; m >= 0; m--) x = bfly_plus(sums[q[r * QS + m]], x, w1);
            v[4 * h + r] = x;
          }
        }
      } else {
#pragma unroll
        for (int m = QS - 1; m >= 0; m--)
#pragma unroll
          for (int h = 0; h < 2; h++) {
            float4 xq[QN];
            quads_at(8 * h + 16 * m, xq);
#pragma unroll
            for (int r = 0; r < 8; r++) {
              const float2 x = quad_sum(xq[r], g1, g2, g3);
              v[8 * h + r] = m == QS - 1 ? x : bfly_plus(x, v[8 * h + r], w1);
            }
          }
      }
#pragma unroll
      for (int r = 0; r < 8; r++) bfly(v[r], v[r + 8], w.w8);
    } else if (P == 1) {
      // samples r, r + 4, r + 8, r + 12
      float4 xq[QN];
      quads_at(0, xq);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float4 x = xq[r];
        const float s0 = w.w8.y * x.z, s1 = w.w8.y * x.w;
        v[r] = make_float2(__builtin_fmaf(w.w8.x, x.z, x.x), s0);
        v[r + 8] = make_float2(__builtin_fmaf(-w.w8.x, x.z, x.x), -s0);
        v[r + 4] = make_float2(__builtin_fmaf(w.w8.x, x.w, x.y), s1);
        v[r + 12] = make_float2(__builtin_fmaf(-w.w8.x, x.w, x.y), -s1);
      }
    } else if (P == 2) {
      // samples r, r + 8, r + 16, r + 24 of 32
      const float2 g2 = c[8], g3 = c[9];
      float4 xq[QN];
      quads_at(0, xq);
#pragma unroll
      for (int r = 0; r < 8; r++) {
        const float4 x = xq[r];
        const float2 e = make_float2(__builtin_fmaf(g2.x, x.z, x.x), g2.y * x.z);
        const float2 s = make_float2(__builtin_fmaf(g3.x, x.w, __builtin_fmaf(w.w8.x, x.y, e.x)),
                                     __builtin_fmaf(g3.y, x.w, __builtin_fmaf(w.w8.y, x.y, e.y)));
        v[r] = s;
        v[r + 8] = make_float2(__builtin_fmaf(2.0f, e.x, -s.x), __builtin_fmaf(2.0f, e.y, -s.y));
      }
    } else {
      // samples r, r + 16, r + 32, r + 48 of 64
      const float2 g1 = c[8], g2 = c[9], g3 = c[10];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        float4 xq[QN];
        quads_at(8 * h, xq);
#pragma unroll
        for (int r = 0; r < 8; r++) v[8 * h + r] = quad_sum(xq[r], g1, g2, g3);
      }
#pragma unroll
      for (int r = 0; r < 8; r++) bfly(v[r], v[r + 8], w.w8);
    }
    dft16_stage2(v, w);
    dft16_stage3(v, w);
    dft16_stage4<false>(v, w);
    if (PW > 1) __syncthreads();                           // every quad read before the buffer is written
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int k = P * q + p;
      const int slot = MID ? k * J1 + (j ^ (J2 * (k % (32 / J2)))) : j * (NL + LPAD) + k;
      buf[slot] = v[bitrev4(q)];
    }
  }

  sync();
  const bool more = band + 1 < nband;
  if (Sh::TWO && more && t < GROUPS) store_quads(B1, t, lo1, hi1);   // every quad of this band has been read

  // ---- middle pass: radix 16 from R1 to 16 R1 bins
  if (MID) {
    const int j = tl % J2, k = tl / J2;
    Tw16 w;
    const float2* c = tab + Sh::MIDOFF + 8 * k;
    w.w8 = c[0]; w.w4 = c[1]; w.w2 = c[2]; w.w2h = c[3]; w.w1 = c[4]; w.w1a = c[5]; w.w1b = c[6]; w.w1c = c[7];
    constexpr int NX = 32 / J2;
    int off[NX];
#pragma unroll
    for (int i = 0; i < NX; i++) off[i] = k * J1 + j + J2 * (i ^ (k % NX));
    float2 v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = buf[off[r % NX] + J2 * (r - r % NX)];
    dft16_tw<false>(v, w);
    sync();
    float2* op = buf + j * (NL + LPAD) + k;
#pragma unroll
    for (int q = 0; q < 16; q++) op[R1 * q] = v[bitrev4(q)];
  }
  if (!Sh::TWO) {
    last_powers();
    channel_phase();
  }
  if (MID) sync();

  // ---- last pass (radix RL), the sideband's half; fractional-sample rotation
  float2 x[8];                                             // bin t + e M/16
  if (RL == 16) {
    Tw16 tw;
    tw.w8 = w[0]; tw.w4 = w[1]; tw.w2 = fresh(w[2]); tw.w1 = fresh(w[3]);
    tw16_multiples(tw);
    float2 v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = buf[r * (NL + LPAD) + tl];
    dft16_tw<true>(v, tw);
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = v[bitrev4(e)];
  } else {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      float2 v[8];
#pragma unroll
      for (int r = 0; r < 8; r++) v[r] = buf[r * (NL + LPAD) + tl + u * NTF];
      dft8_tw<true>(v, w[u], w[2 + u], fresh(w[4 + u]));
#pragma unroll
      for (int q = 0; q < 4; q++) x[u + 2 * q] = v[bitrev3(q)];
    }
  }
  if (Sh::TWO && more) sync();                             // the buffer has been read
  if (mine) {
    const long long outbase = B.specoff + (long long)cb * A.bstride;
    const long long c0 = cidx(PW * tl + pw, A.gstride), cstep = (PW * NTF / 16) * A.gstride;
    const bool turned = B.polre != 1.0f || B.polim != 0.0f;
    auto store = [&](auto out) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const long long at = NTF % 16 == 0 ? c0 + e * cstep : cidx(tl + e * NTF, A.gstride);
        float2 y = cmulx(x[e], Sh::TWO ? FE[e] : cmulx(F, cl[4 + e]));
        if (turned) y = cmulx(y, make_float2(B.polre, B.polim));
        put_spec(out, at, PW * (tl + e * NTF) + pw, y);
      }
    };
    if (A.prec == FXG_XMAC_FP32) store((float2*)A.spectra + outbase);
    else if (A.prec == FXG_XMAC_FP16) store((__half2*)A.spectra + outbase);
    else if (A.prec == FXG_XMAC_FP8)
      store(Fp8Out{(unsigned short*)A.spectra + outbase, A.cexp + (long long)(band ? pair.y : pair.x) * C});
    else store((__hip_bfloat162*)A.spectra + outbase);
  }
  }
}

// ---------------------------------------------------------------------------
// k_fstage_lin_c<L, NBITS>: complex samples (Mode with usecomplex,
// mode.cpp:1184-1241), linear rotation.  L complex samples a block, each a
// unit of 2 NBITS bits with the real part low, through the passes of
// k_fstage_lin with the same tables; every output is kept, channel c of the
// band being bin m (USB: m = c; DSB: the halves swapped, m = c + L/2 mod L;
// LSB: conjugated in reverse order, m = L - c with DC kept; LSB DSB: m = L/2 -
// c mod L, conjugated; a conjugated bin's phase has its sign in DevRot).
// The first pass reads units half a block apart in pairs: one LDS byte (2-bit)
// and one 16-byte lookup, or one word (8-bit), decode two complex samples.
// Bound by FP32 VALU issue like k_fstage_lin; the pairs lie in the exchange
// buffer, for two workgroups a CU up to 8192 points, which a third barrier
// pays.  1024 points, 2-bit, 8 stations of 8 bands, 4001 blocks (0.26
// Gsamples): 1.10 -> 0.70 ms against k_fstage_c's rotator tables and radix-4
// pass.
// ---------------------------------------------------------------------------
template <int L, int NBITS>
__global__ __launch_bounds__(FsShape<L>::NT, 4) void k_fstage_lin_c(FStageArgs A) {
  using Sh = FsShape<L>;
  static_assert(Sh::PW == 1, "a workgroup holds whole blocks");
  constexpr int P = Sh::P, R1 = Sh::R1, J1 = Sh::J1, J2 = Sh::J2, RL = Sh::RL, NTF = Sh::NTF, NB = Sh::NB, NT = Sh::NT;
  constexpr bool MID = Sh::MID;
  constexpr int UB = 2 * NBITS, UPW = 32 / UB;            // bits of a unit, units of a word
  constexpr int GROUPS = L / 2 / UPW;                     // words of half a block
  constexpr int NIT = (GROUPS + NTF - 1) / NTF;
  constexpr int NL = L / RL, LPAD = 32 / RL;
  constexpr int NE = Sh::NE + 8;                          // E[e] = e^{2 pi i theta e L/16} for e >= 8 at the end
  struct Smem {
    float2 tab[NB][NE];
    float4 quad[NBITS == 2 ? 256 : 1];
    float2 buf[NB][L + 32 + (NTF < 32 ? 1 : 0)];
  };
  __shared__ __align__(16) Smem sm;

  const int tid = threadIdx.x;
  const int fi = NB == 1 ? 0 : tid / NTF, t = NB == 1 ? tid : tid % NTF;
  unsigned* const raw = (unsigned*)sm.buf[fi];
  unsigned* const ok = raw + 2 * GROUPS;
  static_assert(NBITS == 8 ? 2 * GROUPS <= 2 * L : 4 * GROUPS <= 2 * L, "pairs and validity fit the buffer");
  const FsPlace place = fstage_place(blockIdx.x, blockIdx.y, gridDim.x, (unsigned)(A.nchunk + NB - 1) / NB, 1);
  if (place.row >= (unsigned)A.nrows || place.grp * NB >= (unsigned)A.nchunk) return;
  const int cbx = place.grp * NB + fi;
  const bool mine = NB == 1 || cbx < A.nchunk;
  const int cb = mine ? cbx : A.nchunk - 1;
  const int gband = A.pairs[place.row].x;
  const DevBand& B = A.bands[gband];
  const DevStationSub& Q = A.ss[B.station];
  const DevRot& R = A.rots[(long long)B.rot * A.nblocks_subint + A.chunk0 + cb];
  const bool dead = R.status != 0;
  if (NB == 1 && dead) {
    zero_spec(A.spectra, A.prec, B.specoff + (long long)cb * A.bstride, L, A.gstride, tid, NT);
    return;
  }

  // ---- the block's samples: two rows half a block apart, to pairs of units
  const bool fast = R.allvalid != 0 || dead;
  const long long bit0 = (long long)(dead ? 0 : R.t0) * UB;
  const long long nwords = Q.ctstride >> 2;
  const unsigned* const src = (const unsigned*)(A.ct + Q.ctbase + (long long)B.band * Q.ctstride);
  unsigned lo[NIT][2], hi[NIT][2];
#pragma unroll
  for (int i = 0; i < NIT; i++)
#pragma unroll
    for (int m = 0; m < 2; m++) {
      const long long w = (bit0 >> 5) + t + i * NTF + m * GROUPS;
      lo[i][m] = w < nwords ? src[w] : 0u;
      hi[i][m] = w + 1 < nwords ? src[w + 1] : 0u;
    }
  {
    const double delta = R.delta, theta = R.theta;
    for (int i = NTF - 1 - t; i < NE; i += NTF) {
      const float4 d = A.cdesc[i];
      sm.tab[fi][i] = exact_rotator(theta * (double)d.y - (delta * (double)d.x + (double)d.z));
    }
  }
  if (NBITS == 2)
    for (int i = tid; i < 256; i += NT) sm.quad[i] = A.quad[B.levels * 256 + i];
#pragma unroll
  for (int i = 0; i < NIT; i++) {
    const int g = t + i * NTF;
    unsigned a[2], v[2] = {0u, 0u};
#pragma unroll
    for (int m = 0; m < 2; m++) a[m] = __builtin_amdgcn_alignbit(hi[i][m], lo[i][m], (int)(bit0 & 31));
    if (!fast) {
      const DevStation& S = A.st[B.station];
#pragma unroll
      for (int m = 0; m < 2; m++)
        v[m] = valid_samples<UPW>(S, Q, A.ftab, R.t0 + (long long)(m * GROUPS + g) * UPW, R.validend, B.band);
      if (NBITS == 2) {
        // a bit for each float of the pair: real and imaginary parts of both
        auto spread = [](unsigned x) { return ((x & 15u) * 0x00204081u) & 0x01010101u; };
        unsigned m0 = spread(v[0]) * 3u | spread(v[1]) * 12u, m1 = spread(v[0] >> 4) * 3u | spread(v[1] >> 4) * 12u;
        if (S.granularity > 1) {
          // one band of 2-bit complex samples: the unpacker's erasure by float
          // index zeroes sample L/2 (even start) or the imaginary part of
          // sample L/2 - 1 (odd start)
          if ((R.t0 & 1) == 0) { if (g == 0) m0 &= ~12u; }
          else if (g == GROUPS - 1) m1 &= ~(2u << 24);
        }
        ok[2 * g] = m0;
        ok[2 * g + 1] = m1;
      }
    }
    if (NBITS == 8) {
#pragma unroll
      for (int m = 0; m < 2; m++) {
        a[m] ^= 0x80808080u;                               // signed levels, 0 = none
        if (!fast) a[m] &= ((v[m] & 1u) | (v[m] & 2u) << 15) * 0xFFFFu;
      }
      *(uint2*)&raw[2 * g] = make_uint2(__builtin_amdgcn_perm(a[1], a[0], 0x05040100u),
                                        __builtin_amdgcn_perm(a[1], a[0], 0x07060302u));
    } else {
      auto spread = [](unsigned x) {
        x = (x | (x << 8)) & 0x00FF00FFu;
        return (x | (x << 4)) & 0x0F0F0F0Fu;
      };
      *(uint2*)&raw[2 * g] = make_uint2(spread(a[0] & 0xFFFFu) | spread(a[1] & 0xFFFFu) << 4,
                                        spread(a[0] >> 16) | spread(a[1] >> 16) << 4);
    }
  }
  __syncthreads();

  auto sync = [] {
    if (NTF > 64) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };
  float2* const buf = sm.buf[fi];
  const float2* const tab = sm.tab[fi];

  // ---- pass 1: decode, radix R1 (this thread's 16 of the R1 outputs)
  {
    const int p = t / J1, j = t % J1;
    const float2* c = tab + p * Sh::CP;
    Tw16 w;
    w.w8 = c[0]; w.w4 = c[1]; w.w2 = c[2]; w.w2h = c[3]; w.w1 = c[4]; w.w1a = c[5]; w.w1b = c[6]; w.w1c = c[7];
    // units j + r J1 and, half a block on, j + (r + R1/2) J1: eight of them
    // from r0 (four from r0 and four from r0 + 16 where P = 4), all their LDS
    // reads in flight together
    auto pairs_at = [&](int r0, float4* x) {
      unsigned q[8];
      auto at = [&](int i) { return j + (r0 + (P == 4 ? (i & 3) + 4 * (i & 4) : i)) * J1; };
      if (NBITS == 8) {
#pragma unroll
        for (int i = 0; i < 8; i++) q[i] = raw[at(i)];
#pragma unroll
        for (int i = 0; i < 8; i++)
          x[i] = make_float4((float)(signed char)(q[i] & 0xFFu), (float)(signed char)((q[i] >> 8) & 0xFFu),
                             (float)(signed char)((q[i] >> 16) & 0xFFu), (float)(signed char)(q[i] >> 24));
        return;
      }
#pragma unroll
      for (int i = 0; i < 8; i++) q[i] = ((const unsigned char*)raw)[at(i)];
#pragma unroll
      for (int i = 0; i < 8; i++) x[i] = sm.quad[q[i]];
      if (!fast) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const unsigned m = ((const unsigned char*)ok)[at(i)];
          x[i].x = m & 1u ? x[i].x : 0.0f;
          x[i].y = m & 2u ? x[i].y : 0.0f;
          x[i].z = m & 4u ? x[i].z : 0.0f;
          x[i].w = m & 8u ? x[i].w : 0.0f;
        }
      }
    };
    float2 v[16];
    if (P == 1) {
      float4 x[8];
      pairs_at(0, x);
#pragma unroll
      for (int r = 0; r < 8; r++) {
        v[r] = make_float2(x[r].x, x[r].y);
        v[r + 8] = make_float2(x[r].z, x[r].w);
      }
    } else if (P == 2) {
      const float2 g2 = c[8];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        float4 x[8];
        pairs_at(8 * h, x);
#pragma unroll
        for (int r = 0; r < 8; r++)
          v[8 * h + r] = bfly_plus(make_float2(x[r].x, x[r].y), make_float2(x[r].z, x[r].w), g2);
      }
    } else {
      // x0 + g1 x1 + g2 x2 + g3 x3 of samples a quarter of the block apart
      const float2 g1 = c[8], g2 = c[9], g3 = c[10];
#pragma unroll
      for (int h = 0; h < 4; h++) {
        float4 x[8];
        pairs_at(4 * h, x);
#pragma unroll
        for (int r = 0; r < 4; r++)
          v[4 * h + r] = bfly_plus(bfly_plus(bfly_plus(make_float2(x[r].x, x[r].y), make_float2(x[r + 4].x, x[r + 4].y), g1),
                                             make_float2(x[r].z, x[r].w), g2),
                                   make_float2(x[r + 4].z, x[r + 4].w), g3);
        // summed before the next lookups, for registers
#pragma unroll
        for (int r = 0; r < 4; r++) asm volatile("" : "+v"(v[4 * h + r].x), "+v"(v[4 * h + r].y) :: "memory");
      }
    }
    dft16_tw<false>(v, w);
    sync();                                                // every pair read before the buffer is written
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int k = P * q + p;
      const int slot = MID ? k * J1 + (j ^ (J2 * (k % (32 / J2)))) : j * (NL + LPAD) + k;
      buf[slot] = v[bitrev4(q)];
    }
  }
  sync();

  // ---- middle pass: radix 16 from R1 to 16 R1 bins
  if (MID) {
    const int j = t % J2, k = t / J2;
    Tw16 w;
    const float2* c = tab + Sh::MIDOFF + 8 * k;
    w.w8 = c[0]; w.w4 = c[1]; w.w2 = c[2]; w.w2h = c[3]; w.w1 = c[4]; w.w1a = c[5]; w.w1b = c[6]; w.w1c = c[7];
    constexpr int NX = 32 / J2;
    int off[NX];
#pragma unroll
    for (int i = 0; i < NX; i++) off[i] = k * J1 + j + J2 * (i ^ (k % NX));
    float2 v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = buf[off[r % NX] + J2 * (r - r % NX)];
    dft16_tw<false>(v, w);
    sync();
    float2* op = buf + j * (NL + LPAD) + k;
#pragma unroll
    for (int q = 0; q < 16; q++) op[R1 * q] = v[bitrev4(q)];
    sync();
  }

  // ---- last pass (radix RL), bins t + e L/16
  const float2* const cl = tab + Sh::LAST;
  float2 x[16];
  if (RL == 16) {
    Tw16 tw;
    tw.w8 = cmulx(A.base[t], cl[0]); tw.w4 = cmulx(A.base[NTF + t], cl[1]);
    tw.w2 = cmulx(A.base[2 * NTF + t], cl[2]); tw.w1 = cmulx(A.base[3 * NTF + t], cl[3]);
    tw16_multiples(tw);
    float2 v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = buf[r * (NL + LPAD) + t];
    dft16_tw<false>(v, tw);
#pragma unroll
    for (int e = 0; e < 16; e++) x[e] = v[bitrev4(e)];
  } else {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      float2 v[8];
#pragma unroll
      for (int r = 0; r < 8; r++) v[r] = buf[r * (NL + LPAD) + t + u * NTF];
      dft8_tw<false>(v, cmulx(A.base[u * NTF + t], cl[1]), cmulx(A.base[(2 + u) * NTF + t], cl[2]),
                     cmulx(A.base[(4 + u) * NTF + t], cl[3]));
#pragma unroll
      for (int q = 0; q < 8; q++) x[u + 2 * q] = v[bitrev3(q)];
    }
  }
  if (!mine) return;

  // ---- to the channels: bin t + e L/16 is channel c0 + f L/16
  const bool lsb = B.lsb;
  const int c0 = !lsb ? t : t == 0 ? 0 : NTF - t;
  const float s = dead ? 0.0f : (NBITS == 8 ? A.scale * (float)(1.0 / 3.3) : A.scale);
  float2 dc = make_float2(0.0f, 0.0f);
  float2 F = exact_rotator(R.phase + R.theta * (double)c0);
  F = make_float2(F.x * s, F.y * s);
  if (B.polre != 1.0f || B.polim != 0.0f) F = cmulx(F, make_float2(B.polre, B.polim));
  if (lsb && !B.dsb && t == 0) {
    // DC is not conjugated: its phase is theta0 - ph, where F's is theta0 + ph,
    // theta0 = -theta L
    float2 G = exact_rotator(-2.0 * R.theta * (double)L - R.phase);
    G = make_float2(G.x * s, G.y * s);
    if (B.polre != 1.0f || B.polim != 0.0f) G = cmulx(G, make_float2(B.polre, B.polim));
    dc = cmulx(x[0], G);
  }
  const int f0 = (lsb ? (t == 0 ? 16 : 15) : 0) + (B.dsb ? 8 : 0), fs = lsb ? -1 : 1;
  const long long outbase = B.specoff + (long long)cb * A.bstride;
  auto store = [&](auto out) {
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int f = (f0 + fs * e) & 15, c = c0 + f * NTF;
      float2 y = cmulx(lsb ? make_float2(x[e].x, -x[e].y) : x[e], cmulx(F, tab[f < 8 ? Sh::LAST + 4 + f : Sh::NE - 8 + f]));
      if (e == 0 && lsb && !B.dsb && t == 0) y = dc;
      put_spec(out, cidx(c, A.gstride), c, y);
    }
  };
  if (A.prec == FXG_XMAC_FP32) store((float2*)A.spectra + outbase);
  else if (A.prec == FXG_XMAC_FP16) store((__half2*)A.spectra + outbase);
  else if (A.prec == FXG_XMAC_FP8) store(Fp8Out{(unsigned short*)A.spectra + outbase, A.cexp + (long long)gband * L});
  else store((__hip_bfloat162*)A.spectra + outbase);
}

// ---------------------------------------------------------------------------
// host side: the tables of one length
// ---------------------------------------------------------------------------
template <int L>
static void fill_tables(std::vector<float4>* cdesc, std::vector<float2>* base) {
  using Sh = FsShape<L>;
  constexpr int M = Sh::M, PW = Sh::PW, P = Sh::P;
  cdesc->assign(Sh::NE + 8, make_float4(0.f, 0.f, 0.f, 0.f));
  // entry = e^{2 pi i (theta y - delta x - z - pw w)}
  auto set = [&](int i, double x, double z, double w, double y = 0.0) {
    (*cdesc)[i] = make_float4((float)x, (float)y, (float)(z - std::floor(z)), (float)w);
  };
  // the eight twiddles of a radix-16 pass to N bins at bin k: powers of
  // e^{-2 pi i (k + d)/N}, d = (pw + delta L)/PW
  auto tw16 = [&](int i, int N, double k) {
    const int m[8] = {8, 4, 2, 2, 1, 1, 1, 1};
    const double add[8] = {0, 0, 0, 1.0 / 8, 0, 1.0 / 16, 2.0 / 16, 3.0 / 16};
    for (int e = 0; e < 8; e++) set(i + e, (double)(M / N) * m[e], k * m[e] / N + add[e], (double)m[e] / (PW * N));
  };
  for (int p = 0; p < P; p++) {
    const int i = p * Sh::CP;
    tw16(i, 16 * P, p);
    if (PW > 1) {
      // samples 16 J1 apart, then a quarter of the block apart
      set(i + 8, L / (P * PW), (double)p / P, 1.0 / (P * PW));
      for (int e = 1; e < 4; e++) set(i + 8 + e, (double)(L / 4) * e, 0.25 * PW * p * e, 0.25 * e);
    } else if (P > 1) {
      // samples a quarter of the block apart (m = 1 is w^8 where P = 2)
      for (int m = P == 2 ? 2 : 1; m < 4; m++) set(i + (P == 2 ? 6 + m : 7 + m), (double)(L / 4) * m, 0.25 * p * m, 0.0);
    }
  }
  const int ml[4] = {8, 4, 2, 1};
  for (int i = 0; i < 4; i++) set(Sh::LAST + i, ml[i], 0.0, (double)ml[i] / L);
  for (int e = 0; e < 8; e++) set(Sh::LAST + 4 + e, 0.0, 0.0, 0.0, (double)(L / 16) * e);
  for (int e = 8; e < 16; e++) set(Sh::NE - 8 + e, 0.0, 0.0, 0.0, (double)(L / 16) * e);   // complex samples
  if (Sh::MID)
    for (int k = 0; k < Sh::R1; k++) tw16(Sh::MIDOFF + 8 * k, 16 * Sh::R1, k);
  // last pass at d = 0: powers 8, 4, 2, 1 (radix 16) or 4, 2, 1 of its two
  // butterflies (radix 8), one entry per thread
  base->clear();
  const int nb = Sh::RL == 16 ? 4 : 3, nu = Sh::RL == 16 ? 1 : 2;
  for (int i = 0; i < nb; i++)
    for (int k = 0; k < nu * Sh::NTF; k++) {
      const double ang = -kTwoPi * (double)k * (1 << (nb - 1 - i)) / M;
      base->push_back(make_float2((float)std::cos(ang), (float)std::sin(ang)));
    }
}

// Two bands to a workgroup (8192 points 25.9 -> 25.2 ms, 2048 points 2.80 ->
// 2.40) where that leaves several times what the chip holds at once, two to
// seven workgroups a CU; below it one each, for the latency of a small call
constexpr long long kPairWorkgroups = 4096;

#define FX_LENGTHS(X) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192) X(16384) \
  X(32768) X(65536)

bool fstage_lin_tables(int L, std::vector<float4>* cdesc, std::vector<float2>* base) {
  switch (L) {
#define X(Lv) case Lv: fill_tables<Lv>(cdesc, base); return true;
    FX_LENGTHS(X)
#undef X
  }
  return false;
}

void fstage_quad_levels(const float* lut, float4* out) {
  for (int b = 0; b < 256; b++)
    out[b] = make_float4(lut[b & 3], lut[(b >> 2) & 3], lut[(b >> 4) & 3], lut[(b >> 6) & 3]);
}

hipError_t launch_fstage_lin(int L, int nbits, const FStageArgs& a, const BandLists& l, int nblocks,
                             hipStream_t stream) {
  if (nbits != 2 && nbits != 8) return hipErrorInvalidValue;
  FStageArgs b = a;
  b.nchunk = nblocks;
  switch (L) {
#define X(Lv)                                                                                                       \
    case Lv: {                                                                                                      \
      const int groups = (nblocks + FsShape<Lv>::NB - 1) / FsShape<Lv>::NB;                                         \
      const bool two = FsShape<Lv>::TWO && (groups + 7LL) / 8 * 8 * l.npairs >= kPairWorkgroups;                    \
      b.pairs = two ? l.pairs : l.singles;                                                                          \
      b.nrows = two ? l.npairs : l.nsingles;                                                                        \
      const FsGrid g = fstage_grid(groups, b.nrows, FsShape<Lv>::PW);                                               \
      const dim3 grid(g.x, g.y);                                                                                    \
      if (nbits == 2) hipLaunchKernelGGL((k_fstage_lin<Lv, 2>), grid, dim3(FsShape<Lv>::NT), 0, stream, b);         \
      else hipLaunchKernelGGL((k_fstage_lin<Lv, 8>), grid, dim3(FsShape<Lv>::NT), 0, stream, b);                    \
      break;                                                                                                        \
    }
    FX_LENGTHS(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_fstage_lin_c(int L, int nbits, const FStageArgs& a, const BandLists& l, int nblocks,
                               hipStream_t stream) {
  if (nbits != 2 && nbits != 8) return hipErrorInvalidValue;
  FStageArgs b = a;
  b.nchunk = nblocks;
  b.pairs = l.singles;
  b.nrows = l.nsingles;
  switch (L) {
#define X(Lv)                                                                                                       \
    case Lv: {                                                                                                      \
      const FsGrid g = fstage_grid((nblocks + FsShape<Lv>::NB - 1) / FsShape<Lv>::NB, l.nsingles, 1);               \
      const dim3 grid(g.x, g.y);                                                                                    \
      if (nbits == 2) hipLaunchKernelGGL((k_fstage_lin_c<Lv, 2>), grid, dim3(FsShape<Lv>::NT), 0, stream, b);       \
      else hipLaunchKernelGGL((k_fstage_lin_c<Lv, 8>), grid, dim3(FsShape<Lv>::NT), 0, stream, b);                  \
      break;                                                                                                        \
    }
    X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace fxg
