// ovx_row_dev.hpp -- device body of the register-resident Stockham fused
// fastconv (any compiled N <= 16384), shared by the standalone kernel and the
// persistent batch kernel.
#pragma once
#include "ovx_internal.hpp"
#include "ovx_pair_dev.hpp"

namespace ovx {

// Whether the stage twiddles stay in registers from the forward to the inverse
// transform (30 values at most here) instead of being loaded for each: 4096
// points, 64 / 1000 rows 7.5 / 20.4 to 7.2 / 19.5 us, 2048 6.5 / 10.3 to 5.6 /
// 9.9.  With 8 values a thread the early loads cost the few-line forms 0.5 us,
// and longer lines have no registers left (16384: 25 to 36 us).
constexpr bool row_holds_twiddles(int N, int P) { return P == 16 && N >= 1024 && N <= 4096; }

// Rows row0 + lrow of the job, thread t of the row's T = N/P threads, LDS row
// region `lds` (Engine LROW elements).  Every thread of the workgroup calls
// it; rows at or beyond `rows` compute on zeros and store nothing.  ix / iy
// access the thread's input and output line and iw its spectrum (interleaved IoC
// or split IoS), element e of the thread at ld(e) / st(v, e).  The spectrum of a
// row at or beyond `rows` is some row's below.
template <int N, int P, typename IX, typename IW, typename IY, typename LP>
__device__ __forceinline__ void row_fastconv_io(const IX &ix, const IW &iw, const IY &iy, long rows,
                                                const float2 *__restrict__ tw, float scale, long row0, int lrow, int t,
                                                LP lds)
{
  using E = Engine<N, P, line_in_wave(N / P)>;
  constexpr int T = E::T;
  const long row = row0 + lrow;
  const bool valid = row < rows;
  const rsrc_t rtw = make_rsrc(tw, (uint32_t)(E::plan.twtotal + 1) * 8u);

  float2 v[P];
  if (valid) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = ix.ld((uint32_t)(T * q));
  } else {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = make_float2(0.f, 0.f);
  }
  constexpr bool HOLD = row_holds_twiddles(N, P);
  float2 st[E::HELD];
  if constexpr (HOLD) {
    E::load_held(t, rtw, st);
    E::template fft_held<-1>(v, lds, t, st);
  } else {
    E::template fft<-1>(v, lds, t, rtw);
  }
  // multiply by the replica spectrum; slot q holds frequency t + T q
#pragma unroll
  for (int q = 0; q < P; ++q) v[q] = cmul(v[q], iw.ld((uint32_t)(T * q)));
  if (scale != 1.0f) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cscale(v[q], scale);
  }
  if constexpr (HOLD) E::template fft_held<+1>(v, lds, t, st);
  else E::template fft<+1>(v, lds, t, rtw);
  if (valid) {
#pragma unroll
    for (int q = 0; q < P; ++q) iy.st(v[q], (uint32_t)(T * q));
  }
}

template <int N, int P, bool NTL = false, typename LP>
__device__ __forceinline__ void row_fastconv_body(const float2 *__restrict__ x, long ldx,
                                                  const float2 *__restrict__ w, long ldw,
                                                  float2 *__restrict__ y, long ldy, long rows,
                                                  const float2 *__restrict__ tw, float scale, long row0, int lrow,
                                                  int t, LP lds)
{
  const int wrow = row0 + lrow < rows ? lrow : 0;
  row_fastconv_io<N, P>(IoCx<NTL>{make_rsrc(x + row0 * ldx, 0xffffffffu), (uint32_t)(lrow * ldx + t) * 8u},
                        IoC{make_rsrc(w + row0 * ldw, 0xffffffffu), (uint32_t)(wrow * ldw + t) * 8u},
                        IoC{make_rsrc(y + row0 * ldy, 0xffffffffu), (uint32_t)(lrow * ldy + t) * 8u}, rows, tw, scale,
                        row0, lrow, t, lds);
}

// Forward (DIR = -1) or inverse (+1) transform of rows row0 + lrow, times
// scale (skipped when 1); same geometry contract as row_fastconv_io.
template <int N, int P, int DIR, typename IX, typename IY, typename LP>
__device__ __forceinline__ void row_fft_io(const IX &ix, const IY &iy, long rows, const float2 *__restrict__ tw,
                                           float scale, long row0, int lrow, int t, LP lds)
{
  using E = Engine<N, P, line_in_wave(N / P)>;
  constexpr int T = E::T;
  const long row = row0 + lrow;
  const bool valid = row < rows;
  const rsrc_t rtw = make_rsrc(tw, (uint32_t)(E::plan.twtotal + 1) * 8u);
  float2 v[P];
  if (valid) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = ix.ld((uint32_t)(T * q));
  } else {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = make_float2(0.f, 0.f);
  }
  E::template fft<DIR>(v, lds, t, rtw);
  if (scale != 1.0f) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cscale(v[q], scale);
  }
  if (valid) {
#pragma unroll
    for (int q = 0; q < P; ++q) iy.st(v[q], (uint32_t)(T * q));
  }
}

template <int N, int P, int DIR, bool NTL = false, typename LP>
__device__ __forceinline__ void row_fft_body(const float2 *__restrict__ in, long ld_in, float2 *__restrict__ out,
                                             long ld_out, long rows, const float2 *__restrict__ tw, float scale,
                                             long row0, int lrow, int t, LP lds)
{
  row_fft_io<N, P, DIR>(IoCx<NTL>{make_rsrc(in + row0 * ld_in, 0xffffffffu), (uint32_t)(lrow * ld_in + t) * 8u},
                        IoC{make_rsrc(out + row0 * ld_out, 0xffffffffu), (uint32_t)(lrow * ld_out + t) * 8u}, rows,
                        tw, scale, row0, lrow, t, lds);
}

// ---------------------------------------------------------------- real transforms
// A real line of n = 2N values is read as N complex pairs z; with Z = FFT_N(z)
// and W = e^{-2 pi i/n} its spectrum is, for k = 0 .. N/2,
//   X[k] = E + W^k O,  X[N-k] = conj(E - W^k O),
//   E = (Z[k] + conj Z[N-k]) / 2,  O = -i (Z[k] - conj Z[N-k]) / 2
// (Z[N] standing for Z[0]).  r2c_pair (ovx_pair_dev.hpp) gives both from Z[k] and
// Z[N-k], c2r_pair the way back: Z[k] = A + i C, Z[N-k] = conj(A - i C) with
// A = X[k] + conj X[N-k], C = W^-k (X[k] - conj X[N-k]).

// The pairs (k, N-k) of one thread: k = t + T q for q < NQ, so that the thread
// holds Z[k] itself (slot form) and finds Z[N-k] in another thread's upper
// slots, through one LDS exchange of half the line.  The mirrored positions
// N - k of a thread are at base(t) + T (NQ - 1 - q).  The middle k = N/2 of an
// even N (its own mirror) is slot P/2 of thread 0.
template <int N, int P>
struct RealPairs {
  static constexpr int T = N / P;
  static constexpr int NQ = (P + 1) / 2;
  static constexpr bool MID = P % 2 == 0;
  static_assert(P % 2 == 0 || T == 1, "an odd number of values per thread only for one-thread lines");
  __device__ static constexpr int mirror_base(int t) { return N - t - T * (NQ - 1); }
  __device__ static constexpr int mirror_off(int q) { return T * (NQ - 1 - q); }
};

// Forward: real lines ix (as N complex pairs per line) to half spectra of
// N + 1 values, times scale: iy stores element t + e of the spectrum at
// st(v, e), iym element mirror_base(t) + e.  wt[k] = W^k, k <= N/2.  Geometry
// contract as row_fastconv_io.
template <int N, int P, typename IX, typename IY, typename LP>
__device__ __forceinline__ void row_r2c_io(const IX &ix, const IY &iy, const IY &iym, long rows,
                                           const float2 *__restrict__ tw, const float2 *__restrict__ wt, float scale,
                                           long row0, int lrow, int t, LP lds)
{
  using E = Engine<N, P, line_in_wave(N / P)>;
  using L = typename E::Layout;
  using R = RealPairs<N, P>;
  constexpr int T = E::T;
  const bool valid = row0 + lrow < rows;
  const rsrc_t rtw = make_rsrc(tw, (uint32_t)(E::plan.twtotal + 1) * 8u);
  const rsrc_t rwt = make_rsrc(wt, (uint32_t)(N / 2 + 1) * 8u);
  float2 v[P];
#pragma unroll
  for (int q = 0; q < P; ++q) v[q] = valid ? ix.ld((uint32_t)(T * q)) : make_float2(0.f, 0.f);
  E::template fft<-1>(v, lds, t, rtw);
  float2 w[R::NQ];
#pragma unroll
  for (int q = 0; q < R::NQ; ++q) w[q] = bload(rwt, (uint32_t)t * 8u, (uint32_t)(T * q) * 8u);
#pragma unroll
  for (int q = P / 2; q < P; ++q) lds_st(lds, L::idx(t + T * q), v[q]);
  exchange_sync<line_in_wave(N / P)>();
  float2 z[R::NQ];
#pragma unroll
  for (int q = 0; q < R::NQ; ++q) {
    const int m = R::mirror_base(t) + R::mirror_off(q); // N - k, N itself for k = 0
    z[q] = lds_ld(lds, L::idx(q == 0 && t == 0 ? N - 1 : m));
  }
  if (t == 0) z[0] = v[0];
  if (!valid) return;
#pragma unroll
  for (int q = 0; q < R::NQ; ++q) {
    float2 xk, xm;
    r2c_pair(v[q], z[q], w[q], scale, xk, xm);
    iy.st(xk, (uint32_t)(T * q));
    iym.st(xm, (uint32_t)R::mirror_off(q));
  }
  if (R::MID && t == 0) {
    float2 xk, xm;
    r2c_pair(v[P / 2], v[P / 2], bload(rwt, 0u, (uint32_t)(N / 2) * 8u), scale, xk, xm);
    iy.st(xk, (uint32_t)(N / 2));
  }
}

// Inverse (unnormalised, times scale): half spectra of N + 1 values (ix at
// t + e, ixm at mirror_base(t) + e; the imaginary parts of X[0] and X[N] are
// ignored) to real lines, stored by iy as N complex pairs per line.
template <int N, int P, typename IX, typename IY, typename LP>
__device__ __forceinline__ void row_c2r_io(const IX &ix, const IX &ixm, const IY &iy, long rows,
                                           const float2 *__restrict__ tw, const float2 *__restrict__ wt, float scale,
                                           long row0, int lrow, int t, LP lds)
{
  constexpr bool WAVE = line_in_wave(N / P);
  using E = Engine<N, P, WAVE>;
  using L = typename E::Layout;
  using R = RealPairs<N, P>;
  constexpr int T = E::T;
  const bool valid = row0 + lrow < rows;
  const rsrc_t rtw = make_rsrc(tw, (uint32_t)(E::plan.twtotal + 1) * 8u);
  const rsrc_t rwt = make_rsrc(wt, (uint32_t)(N / 2 + 1) * 8u);
  float2 v[P], xm[R::NQ], w[R::NQ], mid = make_float2(0.f, 0.f);
  if (valid) {
#pragma unroll
    for (int q = 0; q < R::NQ; ++q) {
      v[q] = ix.ld((uint32_t)(T * q));
      xm[q] = ixm.ld((uint32_t)R::mirror_off(q));
    }
    if (R::MID && t == 0) mid = ix.ld((uint32_t)(N / 2));
  } else {
#pragma unroll
    for (int q = 0; q < R::NQ; ++q) v[q] = xm[q] = make_float2(0.f, 0.f);
  }
#pragma unroll
  for (int q = 0; q < R::NQ; ++q) w[q] = bload(rwt, (uint32_t)t * 8u, (uint32_t)(T * q) * 8u);
  if (t == 0) v[0].y = xm[0].y = 0.f; // DC and Nyquist carry no imaginary part in a real signal
#pragma unroll
  for (int q = 0; q < R::NQ; ++q) {
    float2 zk, zm;
    c2r_pair(v[q], xm[q], w[q], zk, zm);
    v[q] = zk;
    const int m = R::mirror_base(t) + R::mirror_off(q);
    if (q > 0) lds_st(lds, L::idx(m), zm);
    else if (t > 0) lds_st(lds, L::idx(m), zm); // Z[N] of k = 0 is Z[0] itself
  }
  if (R::MID && t == 0) {
    float2 zk, zm;
    c2r_pair(mid, mid, bload(rwt, 0u, (uint32_t)(N / 2) * 8u), zk, zm);
    lds_st(lds, L::idx(N / 2), zk);
  }
  exchange_sync<WAVE>();
#pragma unroll
  for (int q = R::NQ; q < P; ++q) v[q] = lds_ld(lds, L::idx(t + T * q));
  exchange_sync<WAVE>();
  E::template fft<+1>(v, lds, t, rtw);
  if (scale != 1.0f) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cscale(v[q], scale);
  }
  if (valid) {
#pragma unroll
    for (int q = 0; q < P; ++q) iy.st(v[q], (uint32_t)(T * q));
  }
}

} // namespace ovx
