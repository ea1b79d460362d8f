// ovx_rowreal.hip -- real <-> complex row transforms of n = 2N <= 32768 points
// in one pass: the half-length complex transform of a line and the pass that
// turns it into (or builds it from) the half spectrum, with the line in
// registers between the two.
//
// Bound by HBM: each line is read once and written once (n * 4 bytes of reals,
// (N + 1) * 8 of spectrum).  The two values Z[k] and Z[N-k] of a pair lie in
// different threads, so half a line goes through LDS once more.  As two
// launches (transform, then a pass over its result) the spectrum was written,
// read and written again.  Time per call, two launches / one (forward, then
// inverse): 256 x 8192 13.2 / 6.0 and 11.7 / 6.5 us (16.8 MB: 2.8 TB/s),
// 1000 x 8192 33.3 / 16.7 and 24.9 / 16.7 us (3.9 TB/s), 64 x 4096 7.5 / 5.3
// and 6.9 / 5.3 us, 256 x 32768 38.6 / 19.7 and 30.4 / 18.8 us.
//
// Complex sides may be interleaved or split (two float arrays); the arithmetic
// is the same, so both give the same floats.
#include "ovx_internal.hpp"
#include "ovx_row_dev.hpp"
#include "ovx_rowcfg.hpp"

namespace ovx {

// The lane's accessor of the complex side at element e of line lrow.
template <bool SPLIT>
__device__ __forceinline__ auto real_cside(const RealArgs &a, long row0, int lrow, int e)
{
  if constexpr (SPLIT)
    return IoS{make_rsrc(a.cr + row0 * a.ldc, 0xffffffffu), make_rsrc(a.ci + row0 * a.ldc, 0xffffffffu),
               (uint32_t)(lrow * a.ldc + e) * 4u};
  else
    return IoC{make_rsrc(a.c + row0 * a.ldc, 0xffffffffu), (uint32_t)(lrow * a.ldc + e) * 8u};
}

template <int N, int P, bool SPLIT>
__global__ __launch_bounds__((RowCfg<N, P>::NT)) void k_row_r2c(RealArgs a)
{
  const RowPlace<N, P> r;
  row_r2c_io<N, P>(IoC{make_rsrc(a.z + r.row0 * a.ldz, 0xffffffffu), (uint32_t)(r.lrow * a.ldz + r.t) * 8u},
                   real_cside<SPLIT>(a, r.row0, r.lrow, r.t),
                   real_cside<SPLIT>(a, r.row0, r.lrow, RealPairs<N, P>::mirror_base(r.t)), a.lines, a.tw, a.wt,
                   a.scale, r.row0, r.lrow, r.t, r.lds);
}

template <int N, int P, bool SPLIT>
__global__ __launch_bounds__((RowCfg<N, P>::NT)) void k_row_c2r(RealArgs a)
{
  const RowPlace<N, P> r;
  row_c2r_io<N, P>(real_cside<SPLIT>(a, r.row0, r.lrow, r.t),
                   real_cside<SPLIT>(a, r.row0, r.lrow, RealPairs<N, P>::mirror_base(r.t)),
                   IoC{make_rsrc(a.z + r.row0 * a.ldz, 0xffffffffu), (uint32_t)(r.lrow * a.ldz + r.t) * 8u}, a.lines,
                   a.tw, a.wt, a.scale, r.row0, r.lrow, r.t, r.lds);
}

template <int N, int P>
static hipError_t do_real(int dir, const RealArgs &a, hipStream_t s)
{
  const RowLaunch<N, P> l(a.lines);
  if (dir < 0) {
    if (a.cr) hipLaunchKernelGGL((k_row_r2c<N, P, true>), l.grid, l.block, l.lds, s, a);
    else hipLaunchKernelGGL((k_row_r2c<N, P, false>), l.grid, l.block, l.lds, s, a);
  } else {
    if (a.cr) hipLaunchKernelGGL((k_row_c2r<N, P, true>), l.grid, l.block, l.lds, s, a);
    else hipLaunchKernelGGL((k_row_c2r<N, P, false>), l.grid, l.block, l.lds, s, a);
  }
  return hipGetLastError();
}

hipError_t launch_row_real(const RowConfig &cfg, int dir, const RealArgs &a, hipStream_t s)
{
  if (a.lines <= 0) return hipSuccess;
#define X(N, P) \
  if (cfg.n == N && cfg.p == P) return do_real<N, P>(dir, a, s);
  OVX_ROW_CONFIGS(X)
#undef X
  return hipErrorInvalidValue;
}

} // namespace ovx
