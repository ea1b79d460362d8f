// ovx_real.hip -- real <-> complex Fftm by a half-length complex transform.
//
// A real line x of even length n is read as the complex line
// z[m] = x[2m] + i x[2m+1] of length h = n/2.  With Z = FFT_h(z),
//   E[k] = (Z[k] + conj Z[h-k]) / 2,   O[k] = -i (Z[k] - conj Z[h-k]) / 2
// are the transforms of the even and odd samples, and
//   X[k] = E[k] + W^k O[k],   X[h-k] = conj(E[k] - W^k O[k]),   W = e^{-2 pi i/n},
// for k = 0 .. h/2 (a pair is one thread's, so the pass runs in place).
// The inverse (unnormalised, the imaginary parts of X[0] and X[h] ignored)
// builds Z[k] = A + i C, Z[h-k] = conj(A - i C) with
// A = X[k] + conj X[h-k], C = W^-k (X[k] - conj X[h-k]), then
// z = IFFT_h(Z) holds x[2m] + i x[2m+1].
#include "ovx_fs_dev.hpp"
#include "ovx_pair_dev.hpp"
#include "ovx_real.hpp"

namespace ovx {

// Workgroups take rows as the four-step passes do (fs_place), so that rows that
// are in an L2 are worked there; each thread has one pair or, once there are
// plenty, four with their loads in flight together.  Forward / inverse transform,
// rows over all XCDs and one pair a thread / as here, us: 20 x 65536 real values
// 14.2 / 13.5 and 13.2 / 13.0, 18 x 131072 20.5 / 19.1 and 17.5 / 17.2; four pairs
// with few rows, 1 x 65536 9.1, one 8.2.
constexpr int kPairThreads = 256;

// Spectrum line access: interleaved or split.
struct CLine {
  float2 *p;
  __device__ __forceinline__ float2 ld(long k) const { return p[k]; }
  __device__ __forceinline__ void st(long k, float2 v) const { p[k] = v; }
};
struct SLine {
  float *re, *im;
  __device__ __forceinline__ float2 ld(long k) const { return make_float2(re[k], im[k]); }
  __device__ __forceinline__ void st(long k, float2 v) const
  {
    re[k] = v.x;
    im[k] = v.y;
  }
};

template <int kPairs, typename Out>
__device__ __forceinline__ void r2c_row(const float2 *z, const Out out, long group, long h,
                                        const float2 *__restrict__ wt, float scale)
{
  const long k0 = group * (kPairs * kPairThreads) + threadIdx.x;
  float2 zk[kPairs], zm[kPairs], w[kPairs];
#pragma unroll
  for (int i = 0; i < kPairs; ++i) {
    const long k = k0 + i * kPairThreads;
    if (k <= h / 2) {
      zk[i] = z[k];
      zm[i] = z[k == 0 ? 0 : h - k];
      w[i] = wt[k];
    }
  }
#pragma unroll
  for (int i = 0; i < kPairs; ++i) {
    const long k = k0 + i * kPairThreads;
    if (k <= h / 2) {
      float2 xk, xm;
      r2c_pair(zk[i], zm[i], w[i], scale, xk, xm);
      out.st(k, xk);
      if (k != h - k) out.st(h - k, xm);
    }
  }
}
template <int kPairs, typename In>
__device__ __forceinline__ void c2r_row(const In in, float2 *__restrict__ z, long group, long h,
                                        const float2 *__restrict__ wt)
{
  const long k0 = group * (kPairs * kPairThreads) + threadIdx.x;
  float2 xk[kPairs], xm[kPairs], w[kPairs];
#pragma unroll
  for (int i = 0; i < kPairs; ++i) {
    const long k = k0 + i * kPairThreads;
    if (k <= h / 2) {
      xk[i] = in.ld(k);
      xm[i] = in.ld(h - k);
      w[i] = wt[k];
    }
  }
#pragma unroll
  for (int i = 0; i < kPairs; ++i) {
    const long k = k0 + i * kPairThreads;
    if (k <= h / 2) {
      if (k == 0) xk[i].y = xm[i].y = 0.f; // DC and Nyquist carry no imaginary part in a real signal
      float2 zk, zm;
      c2r_pair(xk[i], xm[i], w[i], zk, zm);
      z[k] = zk;
      if (k != 0 && k != h - k) z[h - k] = zm;
    }
  }
}

// In place: each pair is read and written by one thread.
template <int kPairs>
__global__ __launch_bounds__(kPairThreads) void k_r2c_post(float2 *y, long ldy, unsigned groups, unsigned lines, long h,
                                                           const float2 *__restrict__ wt, float scale)
{
  long row, group;
  fs_place(blockIdx.x, groups, lines, row, group);
  r2c_row<kPairs>(y + row * ldy, CLine{ y + row * ldy }, group, h, wt, scale);
}

template <int kPairs>
__global__ __launch_bounds__(kPairThreads) void k_c2r_pre(const float2 *__restrict__ x, long ldx,
                                                          float2 *__restrict__ z, long ldz, unsigned groups,
                                                          unsigned lines, long h, const float2 *__restrict__ wt)
{
  long row, group;
  fs_place(blockIdx.x, groups, lines, row, group);
  c2r_row<kPairs>(CLine{ const_cast<float2 *>(x) + row * ldx }, z + row * ldz, group, h, wt);
}

// Split-storage forms: the post-pass reads Z from an interleaved workspace
// and writes X as separate real / imaginary arrays; the pre-pass reads X
// from them.  Same arithmetic as the interleaved passes.
template <int kPairs>
__global__ __launch_bounds__(kPairThreads) void k_r2c_post_split(const float2 *__restrict__ z, long ldz,
                                                                 float *__restrict__ yr, float *__restrict__ yi,
                                                                 long ldy, unsigned groups, unsigned lines, long h,
                                                                 const float2 *__restrict__ wt, float scale)
{
  long row, group;
  fs_place(blockIdx.x, groups, lines, row, group);
  r2c_row<kPairs>(z + row * ldz, SLine{ yr + row * ldy, yi + row * ldy }, group, h, wt, scale);
}

template <int kPairs>
__global__ __launch_bounds__(kPairThreads) void k_c2r_pre_split(const float *__restrict__ xr,
                                                                const float *__restrict__ xi, long ldx,
                                                                float2 *__restrict__ z, long ldz, unsigned groups,
                                                                unsigned lines, long h, const float2 *__restrict__ wt)
{
  long row, group;
  fs_place(blockIdx.x, groups, lines, row, group);
  c2r_row<kPairs>(SLine{ const_cast<float *>(xr) + row * ldx, const_cast<float *>(xi) + row * ldx }, z + row * ldz, group, h,
          wt);
}

// Pairs per thread and workgroups of a row.
static int pairs_of(long h, long lines) { return (h / 2 / kPairThreads) * lines >= 2048 ? 4 : 1; }
static unsigned pair_groups(long h, int pairs)
{
  return (unsigned)((h / 2 + 1 + pairs * kPairThreads - 1) / (pairs * kPairThreads));
}
#define OVX_PAIRS(kernel, ...)                                                                                        \
  do {                                                                                                                \
    if (lines <= 0 || h <= 0) return hipSuccess;                                                                      \
    const int pairs = pairs_of(h, lines);                                                                             \
    const unsigned g = pair_groups(h, pairs);                                                                         \
    const dim3 grid(g * (unsigned)lines), block(kPairThreads);                                                        \
    if (pairs == 4) hipLaunchKernelGGL(kernel<4>, grid, block, 0, s, __VA_ARGS__);                                    \
    else hipLaunchKernelGGL(kernel<1>, grid, block, 0, s, __VA_ARGS__);                                               \
    return hipGetLastError();                                                                                         \
  } while (0)

hipError_t launch_r2c_post_split(const float2 *z, long ldz, float *yr, float *yi, long ldy, long lines, long h,
                                 const float2 *wt, float scale, hipStream_t s)
{
  OVX_PAIRS(k_r2c_post_split, z, ldz, yr, yi, ldy, g, (unsigned)lines, h, wt, scale);
}

hipError_t launch_c2r_pre_split(const float *xr, const float *xi, long ldx, float2 *z, long ldz, long lines, long h,
                                const float2 *wt, hipStream_t s)
{
  OVX_PAIRS(k_c2r_pre_split, xr, xi, ldx, z, ldz, g, (unsigned)lines, h, wt);
}

hipError_t launch_r2c_post(float2 *y, long ldy, long lines, long h, const float2 *wt, float scale, hipStream_t s)
{
  OVX_PAIRS(k_r2c_post, y, ldy, g, (unsigned)lines, h, wt, scale);
}

hipError_t launch_c2r_pre(const float2 *x, long ldx, float2 *z, long ldz, long lines, long h, const float2 *wt,
                          hipStream_t s)
{
  OVX_PAIRS(k_c2r_pre, x, ldx, z, ldz, g, (unsigned)lines, h, wt);
}

} // namespace ovx
