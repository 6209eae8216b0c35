// fx_bits.h — bit-level helpers shared by device code and host-side tests.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define FXG_HD __host__ __device__ __forceinline__
#else
#define FXG_HD inline
#endif

namespace fxg {

// Transpose a 16 x 16 matrix of 2-bit fields held in 16 words:
// on entry field k of w[t] (bits 2k..2k+1) is element (t, k); on exit field t
// of w[k] is that element.  Four block-swap stages (8, 4, 2, 1 fields), each
// exchanging the off-diagonal blocks of every 2x2 block of the stage.
FXG_HD void transpose16x2(uint32_t* w) {
#define FXG_SWAP(a, b, sh, m)                    \
  {                                              \
    uint32_t t_ = (((a) >> (sh)) ^ (b)) & (m);  \
    (b) ^= t_;                                   \
    (a) ^= t_ << (sh);                           \
  }
  for (int t = 0; t < 8; t++) FXG_SWAP(w[t], w[t + 8], 16, 0x0000FFFFu);
  for (int t = 0; t < 16; t++)
    if ((t & 4) == 0) FXG_SWAP(w[t], w[t + 4], 8, 0x00FF00FFu);
  for (int t = 0; t < 16; t++)
    if ((t & 2) == 0) FXG_SWAP(w[t], w[t + 2], 4, 0x0F0F0F0Fu);
  for (int t = 0; t < 16; t += 2) FXG_SWAP(w[t], w[t + 1], 2, 0x33333333u);
#undef FXG_SWAP
}

// A group of 32/U sample-times of 2^N channels of U bits (sample-time major,
// channel minor, LSB first) held in 2^N words, to one word per channel: on
// exit w[i] holds channel turned_channel<U, N>(i)'s 32/U samples in time order.
// Written over the bits of a field's index, in-word bits below word bits, the
// input is (time, channel) and the output (channel, time); each step below
// exchanges two index bits, one delta swap per word or pair of words.
constexpr int fields_log2(int U) { return U == 2 ? 4 : U == 4 ? 3 : U == 8 ? 2 : 1; }
// the fields whose index has bit J clear
constexpr uint32_t fields_clear(int U, int J) {
  uint32_t m = 0;
  for (int p = 0; p < 32 / U; p++)
    if (!((p >> J) & 1)) m |= ((U == 32 ? 0u : (1u << U)) - 1u) << (p * U);
  return m;
}
template <int U, int N> FXG_HD constexpr int turned_channel(int i) {
  constexpr int F = fields_log2(U);
  return N > F ? ((i & ((1 << (N > F ? N - F : 0)) - 1)) << F) | (i >> (N > F ? N - F : 0)) : i;
}
template <int U, int N> FXG_HD void turn_units(uint32_t* w) {
  constexpr int F = fields_log2(U), D = N < F ? N : F, LOW = N - D;
  // word bits LOW.. (time, or the words' own order) with in-word bits 0.. (channel)
#pragma unroll
  for (int i = 0; i < D; i++) {
    const int sh = U << i;
    const uint32_t m = fields_clear(U, i);
#pragma unroll
    for (int a = 0; a < (1 << N); a++) {
      if ((a >> (LOW + i)) & 1) continue;
      const int b = a | (1 << (LOW + i));
      const uint32_t t = ((w[a] >> sh) ^ w[b]) & m;
      w[b] ^= t;
      w[a] ^= t << sh;
    }
  }
  // fewer channels than fields: in-word bit p now holds time bit
  // F - N + p (p < N) or p - N, sorted into place
  if (N > 0 && N < F) {
    int cur[F];
    for (int p = 0; p < F; p++) cur[p] = p < N ? F - N + p : p - N;
#pragma unroll
    for (int p = 0; p < F; p++) {
#pragma unroll
      for (int q = p + 1; q < F; q++) {
        if (cur[q] != p) continue;
        const int d = (U << q) - (U << p);
        const uint32_t m = fields_clear(U, q) & ~fields_clear(U, p);
#pragma unroll
        for (int a = 0; a < (1 << N); a++) {
          const uint32_t t = ((w[a] >> d) ^ w[a]) & m;
          w[a] ^= t ^ (t << d);
        }
        cur[q] = cur[p];
        cur[p] = p;
        break;
      }
    }
  }
}

}  // namespace fxg
