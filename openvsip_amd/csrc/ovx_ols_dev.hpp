// ovx_ols_dev.hpp -- device body of overlap-save segments (see ovx_ols.hip),
// shared by the standalone kernels and the persistent kernel.
#pragma once
#include "ovx_internal.hpp"
#include "ovx_ols.hpp"

namespace ovx {

// unbiased divisor of output n (corr.hpp:115-124, 163-178, 204-206)
__device__ __forceinline__ float corr_divisor(int support, long n, long M, long N)
{
  if (support == 0) {
    if (n < M - 1) return (float)(n + 1);
    if (n >= N) return (float)(N + M - 1 - n);
    return (float)M;
  } else if (support == 1) {
    if (n < M / 2) return (float)(n + (M + 1) / 2);
    if (n >= N - M / 2) return (float)(N - 1 + (M + 1) / 2 - n);
    return (float)M;
  }
  return (float)M;
}

// Buffer offset of a value a lane does not have: past every descriptor made
// here (kOlsRecords bytes), so a load of it gives zero and a store of it is
// dropped.  The out-of-range ends of a segment cost a compare and a select
// this way; as branches around each access they made the compiler wait for
// every load before the next one (a 4096-point segment took 12 us, most of it
// 16 memory latencies in turn).
constexpr uint32_t kOlsNone = 0x80000000u;
constexpr uint32_t kOlsRecords = 0x7ffffff8u;

// Kernel values h[u] (reversed: h[M - 1 - u]) of slot form, zero from M on.
template <int L, int P>
__device__ __forceinline__ void ols_load_kernel(const float2 *h, long M, bool reverse, int t, float2 (&v)[P])
{
  constexpr int T = L / P;
  const rsrc_t r = make_rsrc(h, kOlsRecords);
  const int m = (int)M;
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int u = t + T * q;
    v[q] = bload(r, u < m ? (uint32_t)(reverse ? m - 1 - u : u) * 8u : kOlsNone, 0);
  }
}

// Segment seg0 + copy by thread t of L/P threads, LDS region `lds` (E::LROW);
// seg0 is the same for the whole workgroup.  REF: the kernel's spectrum is
// computed here from a.h (a correlation's reference, reversed), else read
// from a.H.  Copies past the last segment store nothing.
template <int L, int P, bool REF = false, typename LP>
__device__ __forceinline__ void ols_body(const OlsArgs &a, long seg0, int copy, int t, LP lds)
{
  using E = Engine<L, P, line_in_wave(L / P)>;
  constexpr int T = E::T;
  const int m1 = (int)(a.M - 1);
  const int at = copy * (int)a.c_step; // this copy's distance from segment seg0
  const rsrc_t rtw = make_rsrc(a.tw, (uint32_t)(E::plan.twtotal + 1) * 8u);

  // input g[i0 - (M-1) + u], zero outside [0, N)
  const long g0 = a.c_first + seg0 * a.c_step - m1;
  const rsrc_t rin = make_rsrc(a.in + g0, kOlsRecords);
  const int lo = g0 < 0 ? (int)-g0 : 0;
  const int hi = (int)min(max(a.N - g0, (long)lo), 1l << 27);
  float2 v[P];
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int rel = at + t + T * q;
    v[q] = bload(rin, (uint32_t)(rel - lo) < (uint32_t)(hi - lo) ? (uint32_t)rel * 8u : kOlsNone, 0);
  }
  float2 h[P];
  if constexpr (REF) {
    ols_load_kernel<L, P>(a.h, a.M, true, t, h);
    E::template fft<-1>(h, lds, t, rtw);
  } else {
    const rsrc_t rh = make_rsrc(a.H, (uint32_t)L * 8u);
#pragma unroll
    for (int q = 0; q < P; ++q) h[q] = bload(rh, (uint32_t)t * 8u, (uint32_t)(T * q) * 8u);
  }
  if (a.conj_input) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q].y = -v[q].y;
  }
  E::template fft<-1>(v, lds, t, rtw);
#pragma unroll
  for (int q = 0; q < P; ++q) v[q] = cmul(v[q], cscale(h[q], a.scale));
  E::template fft<+1>(v, lds, t, rtw);

  // outputs u >= M-1: c index first + at + u - (M-1), n = index / D where D
  // divides it
  const long first = seg0 * a.c_step;
  if (a.decimation == 1) {
    const rsrc_t rout = make_rsrc(a.out + first, kOlsRecords);
    const int left = (int)min(a.P - first, 1l << 27);
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int u = t + T * q, n = at + u - m1;
      float2 r = v[q];
      if (a.unbiased) {
        const float d = corr_divisor(a.support, first + n, a.M, a.N);
        r.x /= d;
        r.y /= d;
      }
      bstore(rout, r, u >= m1 && n < left ? (uint32_t)n * 8u : kOlsNone, 0);
    }
  } else if (a.decimation <= kOlsMaxMagic) {
    const uint32_t d = (uint32_t)a.decimation;
    const long n0 = first / a.decimation;
    const uint32_t r0 = (uint32_t)(first - n0 * a.decimation);
    const rsrc_t rout = make_rsrc(a.out + n0, kOlsRecords);
    const uint32_t left = (uint32_t)max(min(a.P - n0, 1l << 27), 0l);
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int u = t + T * q;
      const uint32_t i = (uint32_t)(at + u - m1) + r0;
      const uint32_t n = __umulhi(i, a.dmagic);
      bstore(rout, v[q], u >= m1 && i == n * d && n < left ? n * 8u : kOlsNone, 0);
    }
  } else { // at most one output of a segment
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int u = t + T * q;
      const long i = first + at + u - m1;
      if (u >= m1 && i % a.decimation == 0 && i / a.decimation < a.P) a.out[i / a.decimation] = v[q];
    }
  }
}

} // namespace ovx
