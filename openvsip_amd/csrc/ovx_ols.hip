// ovx_ols.hip -- FFT-based 1-D correlation and convolution by overlap-save
// on the LDS-resident engine.
//
// Both operations reduce to one linear convolution c = h * g:
//   correlation (src/ovxx/signal/corr.hpp:91-215)
//       out[n] = sum_k ref[k] conj(in[n + k - shift])
//              = c[n + M-1-shift],  h[j] = ref[M-1-j],  g = conj(in)
//       shift = M-1 (full), M/2 (same), 0 (min);
//   convolution (src/ovxx/signal/conv.hpp:232-330)
//       out[n] = sum_k kernel[k] in[n D + off - k] = c[n D + off],
//       h = kernel, g = in, off = 0 (full), M/2 (same), M-1 (min).
// Segment s of length L covers c[i0, i0 + S), S = L - (M-1): the kernel
// gathers g[i0 - (M-1) + u] (zero outside [0, N)), runs forward FFT,
// multiplies by H = FFT_L(h) / L, inverse FFT, and scatters the valid outputs
// u >= M-1, applying the unbiased divisors (correlation) or the decimation
// (convolution).  One workgroup per segment, or per wave of short segments.
//
// A call is bound by the latency of one segment's chain of stages (a 65536 x
// 1024 correlation has 65 segments for 256 CUs), so short segments run with 8
// values per thread (2048 points: 4.9 us with 8, 5.8 with 16) and one segment
// per workgroup (four of 512 points in one: 4.2 against 3.4 us).  A
// correlation's reference comes with the call; its spectrum is computed by
// every segment for itself while the segment's input is on its way, which
// adds 1.6 us to a 2048-point segment where a launch of its own took 3.4 us
// and more.  With thousands of segments the extra transform is work, not
// latency (3900 of 1024 points: 16.2 to 19.8 us), and H is computed once
// (ols_fuse_ref).  65536 x 1024: 18.1 us in three launches before, 7.6 us now;
// 10^6 x 129 taps, every fourth output: 12.4 and 6.5 us.
#include "ovx_ols_dev.hpp"

namespace ovx {

// Segments of less than 64 threads share a wave: 256 threads a workgroup took
// 3.7 instead of 3.2 us for 20000 x 17, 3.8 instead of 3.6 for 126694 x 17.
template <int L, int P>
struct OlsCfg {
  static constexpr int T = L / P;
  static constexpr int B = T < 64 ? 64 / T : 1;
  static constexpr int NT = T * B;
};

template <int L, int P, bool REF>
__global__ __launch_bounds__((OlsCfg<L, P>::NT)) void k_ols(OlsArgs a)
{
  using C = OlsCfg<L, P>;
  __shared__ float2 lds[C::B * Engine<L, P>::LROW];
  const int copy = C::B == 1 ? 0 : (int)threadIdx.x / C::T;
  const int t = C::B == 1 ? (int)threadIdx.x : (int)threadIdx.x % C::T;
  ols_body<L, P, REF>(a, (long)blockIdx.x * C::B, copy, t, lds + copy * Engine<L, P>::LROW);
}

// H = FFT_L of the reversed (correlation) or plain (convolution) kernel,
// zero-padded to L.
template <int L, int P>
__global__ __launch_bounds__(L / P) void k_ols_spectrum(const float2 *__restrict__ h, long M, int reverse,
                                                        float2 *__restrict__ H, const float2 *__restrict__ tw)
{
  using E = Engine<L, P, line_in_wave(L / P)>;
  __shared__ float2 lds[E::LROW];
  const int t = threadIdx.x;
  float2 v[P];
  ols_load_kernel<L, P>(h, M, reverse != 0, t, v);
  E::template fft<-1>(v, lds, t, make_rsrc(tw, (uint32_t)(E::plan.twtotal + 1) * 8u));
#pragma unroll
  for (int q = 0; q < P; ++q) H[t + E::T * q] = v[q];
}

// X(L, P): the compiled segments.  8 values per thread for the plans' short
// segments; 16 for the longer ones and for every length of the server's
// references, whose batch tiles run the same body.
#define OVX_OLS_CONFIGS(X) \
  X(64, 4) X(128, 8) X(512, 8) X(1024, 8) X(2048, 8) X(1024, 16) X(2048, 16) X(4096, 16) X(8192, 16) X(16384, 16)

hipError_t launch_ols(int L, int P, const OlsArgs &a, long segments, hipStream_t s)
{
  if (segments <= 0) return hipSuccess;
#define X(L_, P_)                                                                                  \
  if (L == L_ && P == P_) {                                                                        \
    using C = OlsCfg<L_, P_>;                                                                      \
    const dim3 grid((unsigned)((segments + C::B - 1) / C::B)), block(C::NT);                       \
    if (a.H) hipLaunchKernelGGL((k_ols<L_, P_, false>), grid, block, 0, s, a);                     \
    else hipLaunchKernelGGL((k_ols<L_, P_, true>), grid, block, 0, s, a);                          \
    return hipGetLastError();                                                                      \
  }
  OVX_OLS_CONFIGS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_ols_spectrum(int L, int P, const float2 *h, long M, int reverse, float2 *H, const float2 *tw,
                               hipStream_t s)
{
#define X(L_, P_)                                                                                                \
  if (L == L_ && P == P_) {                                                                                      \
    hipLaunchKernelGGL((k_ols_spectrum<L_, P_>), dim3(1), dim3(L_ / P_), 0, s, h, M, reverse, H, tw);            \
    return hipGetLastError();                                                                                    \
  }
  OVX_OLS_CONFIGS(X)
#undef X
  return hipErrorInvalidValue;
}

} // namespace ovx
