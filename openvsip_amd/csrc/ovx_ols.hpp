// ovx_ols.hpp -- overlap-save launch interface (correlation / convolution).
#pragma once
#include <hip/hip_runtime.h>

namespace ovx {

struct OlsArgs {
  const float2 *in;  // input signal, length N
  long N;            // input length
  long M;            // kernel length
  const float2 *H;   // FFT_L of the padded kernel, or null:
  const float2 *h;   // the correlation's reference, transformed in the kernel
  const float2 *tw;  // twiddles of the length-L plan
  float scale;       // 1/L
  int conj_input;    // correlation: conj(in)
  int unbiased;      // correlation: per-position divisors
  int support;       // 0 full, 1 same, 2 min
  long decimation;   // convolution: D (1 for correlation)
  long out_off;      // out[n] = c[n*D + out_off]
  long c_first;      // first c index of segment 0 (= out_off)
  long c_step;       // c indices per segment (S = L - (M-1))
  long P;            // output length
  float2 *out;
  // ceil(2^32 / decimation): i / decimation is the high half of i * dmagic
  // while i * decimation < 2^32, which a segment's indices (below 2^15 + the
  // decimation) keep for decimations up to kOlsMaxMagic
  unsigned dmagic;
};
constexpr long kOlsMaxMagic = 32768;
inline unsigned ols_magic(long decimation)
{
  if (decimation < 2 || decimation > kOlsMaxMagic) return 0;
  return (unsigned)(((1ull << 32) + (unsigned long)decimation - 1) / (unsigned long)decimation);
}

// `segments` segments of length L with P values per thread.
hipError_t launch_ols(int L, int P, const OlsArgs &a, long segments, hipStream_t s);
hipError_t launch_ols_spectrum(int L, int P, const float2 *h, long M, int reverse, float2 *H, const float2 *tw,
                               hipStream_t s);

} // namespace ovx
