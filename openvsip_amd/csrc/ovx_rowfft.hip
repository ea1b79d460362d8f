// ovx_rowfft.hip -- LDS-resident row transforms for N <= 16384 on gfx950:
// forward / inverse Fftm by row and the fused fast convolution
// (forward FFT, multiply by the replica spectrum, inverse FFT, scale) in one
// pass over HBM: each line is read once and written once.
//
// Reference behaviour being replaced:
//   Fftm row loop        src/ovxx/fftw/fftw.cpp:965-977 (one execute per row)
//   scale pass           src/ovxx/signal/fft/workspace.hpp:474-478
//   vmmul<0> row loop    src/vsip/impl/vmmul.hpp:79-85
#include "ovx_internal.hpp"
#include "ovx_row_dev.hpp"
#include "ovx_rowcfg.hpp"

namespace ovx {

template <int N, int P, int DIR, bool NTL>
__global__ __launch_bounds__((RowCfg<N, P>::NT)) void k_row_fft(const float2 *__restrict__ in, long ld_in,
                                                               float2 *__restrict__ out, long ld_out, long rows,
                                                               const float2 *__restrict__ tw, float scale)
{
  const RowPlace<N, P> r;
  row_fft_body<N, P, DIR, NTL>(in, ld_in, out, ld_out, rows, tw, scale, r.row0, r.lrow, r.t, r.lds);
}

template <int N, int P>
__global__ __launch_bounds__((RowCfg<N, P>::NT)) void k_row_fastconv(const float2 *__restrict__ x, long ldx,
                                                                    const float2 *__restrict__ w, long ldw,
                                                                    float2 *__restrict__ y, long ldy, long rows,
                                                                    const float2 *__restrict__ tw, float scale)
{
  const RowPlace<N, P> r;
  row_fastconv_body<N, P>(x, ldx, w, ldw, y, ldy, rows, tw, scale, r.row0, r.lrow, r.t, r.lds);
}

// Split-storage forms: real and imaginary parts of the lines, and of a
// fastconv's spectra, in two float arrays with the same strides.
template <int N, int P, int DIR>
__global__ __launch_bounds__((RowCfg<N, P>::NT)) void k_row_fft_split(const float *__restrict__ in_re,
                                                                     const float *__restrict__ in_im, long ld_in,
                                                                     float *__restrict__ out_re,
                                                                     float *__restrict__ out_im, long ld_out,
                                                                     long rows, const float2 *__restrict__ tw,
                                                                     float scale)
{
  const RowPlace<N, P> r;
  row_fft_io<N, P, DIR>(
      IoS{make_rsrc(in_re + r.row0 * ld_in, 0xffffffffu), make_rsrc(in_im + r.row0 * ld_in, 0xffffffffu),
          (uint32_t)(r.lrow * ld_in + r.t) * 4u},
      IoS{make_rsrc(out_re + r.row0 * ld_out, 0xffffffffu), make_rsrc(out_im + r.row0 * ld_out, 0xffffffffu),
          (uint32_t)(r.lrow * ld_out + r.t) * 4u},
      rows, tw, scale, r.row0, r.lrow, r.t, r.lds);
}

template <int N, int P>
__global__ __launch_bounds__((RowCfg<N, P>::NT)) void k_row_fastconv_split(
    const float *__restrict__ xr, const float *__restrict__ xi, long ldx, const float *__restrict__ wr,
    const float *__restrict__ wi, long ldw, float *__restrict__ yr, float *__restrict__ yi, long ldy, long rows,
    const float2 *__restrict__ tw, float scale)
{
  const RowPlace<N, P> r;
  const int wrow = r.row0 + r.lrow < rows ? r.lrow : 0;
  row_fastconv_io<N, P>(
      IoS{make_rsrc(xr + r.row0 * ldx, 0xffffffffu), make_rsrc(xi + r.row0 * ldx, 0xffffffffu),
          (uint32_t)(r.lrow * ldx + r.t) * 4u},
      IoS{make_rsrc(wr + r.row0 * ldw, 0xffffffffu), make_rsrc(wi + r.row0 * ldw, 0xffffffffu),
          (uint32_t)(wrow * ldw + r.t) * 4u},
      IoS{make_rsrc(yr + r.row0 * ldy, 0xffffffffu), make_rsrc(yi + r.row0 * ldy, 0xffffffffu),
          (uint32_t)(r.lrow * ldy + r.t) * 4u},
      rows, tw, scale, r.row0, r.lrow, r.t, r.lds);
}

// ---------------------------------------------------------------- twiddles
struct TwStageDesc {
  int nst;
  int radix[16];
  int ns[16];
  int off[16];
};

__global__ void k_twiddles(TwStageDesc d, float2 *tw, int total)
{
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  // find the stage holding entry i
  int s = 0;
  for (int k = 0; k < d.nst; ++k)
    if (d.ns[k] > 1 && i >= d.off[k]) s = k;
  const int Ns = d.ns[s];
  const int rel = i - d.off[s];
  const int r = rel / Ns + 1;
  const int k = rel % Ns;
  const long L = (long)Ns * d.radix[s];
  const long m = ((long)r * k) % L;
  double sn, cs;
  sincospi(-2.0 * (double)m / (double)L, &sn, &cs);
  tw[i] = make_float2((float)cs, (float)sn);
}

__global__ void k_unit_roots(long n, long count, float2 *out)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  long m = i % n;
  double sn, cs;
  sincospi(-2.0 * (double)m / (double)n, &sn, &cs);
  out[i] = make_float2((float)cs, (float)sn);
}

hipError_t launch_twiddles(const RadixPlan &plan, float2 *tw, hipStream_t s)
{
  if (plan.twtotal == 0) return hipSuccess;
  TwStageDesc d{};
  d.nst = plan.nst;
  for (int k = 0; k < plan.nst; ++k) { d.radix[k] = plan.radix[k]; d.ns[k] = plan.ns[k]; d.off[k] = plan.twoff[k]; }
  int blocks = (plan.twtotal + 255) / 256;
  hipLaunchKernelGGL(k_twiddles, dim3(blocks), dim3(256), 0, s, d, tw, plan.twtotal);
  return hipGetLastError();
}

__global__ void k_scale_copy(const float2 *__restrict__ in, float2 *__restrict__ out, long n, float scale)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = cscale(in[i], scale);
}

hipError_t launch_scale_copy(const float2 *in, float2 *out, long n, float scale, hipStream_t s)
{
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_scale_copy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, in, out, n, scale);
  return hipGetLastError();
}

hipError_t launch_unit_roots(long n, long count, float2 *out, hipStream_t s)
{
  if (count <= 0) return hipSuccess;
  long blocks = (count + 255) / 256;
  hipLaunchKernelGGL(k_unit_roots, dim3((unsigned)blocks), dim3(256), 0, s, n, count, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------- registry
template <int N, int P>
static void fill_cfg(RowConfig *c, int variant)
{
  using C = RowCfg<N, P>;
  c->n = N;
  c->p = P;
  c->rows_per_block = C::B;
  c->threads = C::NT;
  c->plan = Engine<N, P>::plan;
  c->variant = variant;
}

// Whether a transform loads its lines past the caches.  In place the result
// follows the line into its cache lines, and while all of them are in the 32 MB
// of L2, or too many for the Infinity Cache, the load is better not kept.
// Ordinary / non-temporal loads, in place, us: 4000 x 512 8.6 / 7.9, 2000 x 1024
// 8.9 / 7.5, 1000 x 2048 9.8 / 8.3, 1000 x 3072 12.6 / 10.8, 600 x 6144 15.5 /
// 14.2; between, 4000 x 1024 13.2 / 14.5, 1000 x 4096 14.2 / 15.6, 1000 x 6144 22.6 /
// 23.2; 4000 x 4096 57.1 / 53.8, 1000 x 16384 68.9 / 66.0; from 8192 points on, a
// line a CU, ordinary ones stay ahead, 300 x 8192 13.8 / 14.4, and for lines of a
// thread or a few, whose loads of a wave lie apart, 256 x 18 3.2 / 3.5, 4000 x 12
// 2.5 / 2.8.  Out of place: 2000 x 2048 12.3 / 15.6, 1000 x 4096 12.1 / 16.1.
static bool row_streams_in(const float2 *in, const float2 *out, long rows, int n)
{
  const long bytes = rows * n * (long)sizeof(float2);
  return in == out && n >= 256 && ((n < 8192 && bytes <= (30l << 20)) || bytes >= (120l << 20));
}

template <int N, int P, int DIR>
static hipError_t do_fft_dir(const float2 *in, long ld_in, float2 *out, long ld_out, long rows, const float2 *tw,
                             float scale, hipStream_t s)
{
  const RowLaunch<N, P> l(rows);
  if (row_streams_in(in, out, rows, N))
    hipLaunchKernelGGL((k_row_fft<N, P, DIR, true>), l.grid, l.block, l.lds, s, in, ld_in, out, ld_out, rows, tw, scale);
  else
    hipLaunchKernelGGL((k_row_fft<N, P, DIR, false>), l.grid, l.block, l.lds, s, in, ld_in, out, ld_out, rows, tw, scale);
  return hipGetLastError();
}

template <int N, int P>
static hipError_t do_fft(int dir, const float2 *in, long ld_in, float2 *out, long ld_out, long rows,
                         const float2 *tw, float scale, hipStream_t s)
{
  return dir < 0 ? do_fft_dir<N, P, -1>(in, ld_in, out, ld_out, rows, tw, scale, s)
                 : do_fft_dir<N, P, +1>(in, ld_in, out, ld_out, rows, tw, scale, s);
}

template <int N, int P>
static hipError_t do_fastconv(const float2 *x, long ldx, const float2 *w, long ldw, float2 *y, long ldy,
                              long rows, const float2 *tw, float scale, hipStream_t s)
{
  const RowLaunch<N, P> l(rows);
  hipLaunchKernelGGL((k_row_fastconv<N, P>), l.grid, l.block, l.lds, s, x, ldx, w, ldw, y, ldy, rows, tw, scale);
  return hipGetLastError();
}

template <int N, int P>
static hipError_t do_fft_split(int dir, const float *ir, const float *ii, long ld_in, float *orr, float *oi,
                               long ld_out, long rows, const float2 *tw, float scale, hipStream_t s)
{
  const RowLaunch<N, P> l(rows);
  if (dir < 0)
    hipLaunchKernelGGL((k_row_fft_split<N, P, -1>), l.grid, l.block, l.lds, s, ir, ii, ld_in, orr, oi, ld_out, rows,
                       tw, scale);
  else
    hipLaunchKernelGGL((k_row_fft_split<N, P, +1>), l.grid, l.block, l.lds, s, ir, ii, ld_in, orr, oi, ld_out, rows,
                       tw, scale);
  return hipGetLastError();
}

template <int N, int P>
static hipError_t do_fastconv_split(const float *xr, const float *xi, long ldx, const float *wr, const float *wi,
                                    long ldw, float *yr, float *yi, long ldy, long rows, const float2 *tw, float scale,
                                    hipStream_t s)
{
  const RowLaunch<N, P> l(rows);
  hipLaunchKernelGGL((k_row_fastconv_split<N, P>), l.grid, l.block, l.lds, s, xr, xi, ldx, wr, wi, ldw, yr, yi, ldy,
                     rows, tw, scale);
  return hipGetLastError();
}

struct Entry {
  int n, p;
  void (*fill)(RowConfig *, int);
  hipError_t (*fft)(int, const float2 *, long, float2 *, long, long, const float2 *, float, hipStream_t);
  hipError_t (*fconv)(const float2 *, long, const float2 *, long, float2 *, long, long, const float2 *, float,
                      hipStream_t);
  hipError_t (*fft_split)(int, const float *, const float *, long, float *, float *, long, long, const float2 *,
                          float, hipStream_t);
  hipError_t (*fconv_split)(const float *, const float *, long, const float *, const float *, long, float *, float *, long, long,
                            const float2 *, float, hipStream_t);
};

#define OVX_ENTRY(N, P)                                                                              \
  { N, P, &fill_cfg<N, P>, &do_fft<N, P>, &do_fastconv<N, P>, &do_fft_split<N, P>, &do_fastconv_split<N, P> },
static const Entry kEntries[] = { OVX_ROW_CONFIGS(OVX_ENTRY) };
static const int kNumEntries = (int)(sizeof(kEntries) / sizeof(kEntries[0]));

static const Entry *find_entry(int n, int variant)
{
  int seen = 0;
  for (int i = 0; i < kNumEntries; ++i)
    if (kEntries[i].n == n) {
      if (seen == variant) return &kEntries[i];
      ++seen;
    }
  return nullptr;
}

int row_variants(int n)
{
  int c = 0;
  for (int i = 0; i < kNumEntries; ++i)
    if (kEntries[i].n == n) ++c;
  return c;
}

bool row_config(int n, int variant, RowConfig *out)
{
  const Entry *e = find_entry(n, variant);
  if (!e) return false;
  e->fill(out, variant);
  return true;
}

int row_config_with(int n, int p)
{
  for (int v = 0;; ++v) {
    const Entry *e = find_entry(n, v);
    if (!e) return -1;
    if (e->p == p) return v;
  }
}

// The first configuration of a length, or the one with fewer values per thread
// for up to 8 lines a CU if its lines keep to a wave, to one a CU with 128
// threads and 4 with 256; above 256 threads (6144, 12288) it is the slower one
// from one line on.  Fastconv, first / fewer values, us: 384 points, 256 lines 5.7 /
// 4.4, 2000 6.5 / 6.0; 576, 256 6.5 / 4.3, 2000 7.9 / 7.5; 640, 256 7.2 / 5.5, 2000
// 8.9 / 8.8; 1024, 256 4.8 / 4.4, 400 5.2 / 5.3, 1000 6.2 / 6.4; 1536, 256 6.8 / 6.8
// (64 7.3 / 6.7), 400 7.4 / 8.2; 2048, 256 6.8 / 5.3, 600 9.6 / 8.4, 1000 11.2 / 11.0
// (a spectrum per line 13.7 / 11.1), 2000 17.3 / 18.3; 6144, 400 15.9 / 18.3.
// Plain transforms of 256 threads a line cross over sooner: 2048, 700 6.5 / 6.3,
// 800 7.1 / 7.75 (in place 8.2 / 8.9), 900 7.7 / 7.9, 1000 8.0 / 8.0.
int row_pick(int n, long rows, bool plain)
{
  const Entry *first = find_entry(n, 0);
  if (!first) return 0;
  for (int v = 1; const Entry *e = find_entry(n, v); ++v) {
    const int threads = n / e->p;
    const long per_cu = threads <= 64 ? 8 : threads <= 128 ? 1 : threads <= 256 ? (plain ? 3 : 4) : 0;
    if (e->p < first->p && rows <= per_cu * kRowCus) return v;
  }
  return 0;
}

hipError_t launch_row_fft(const RowConfig &cfg, int dir, const float2 *in, long ld_in, float2 *out, long ld_out,
                          long rows, const float2 *tw, float scale, hipStream_t s)
{
  const Entry *e = find_entry(cfg.n, cfg.variant);
  if (!e) return hipErrorInvalidValue;
  if (rows <= 0) return hipSuccess;
  return e->fft(dir, in, ld_in, out, ld_out, rows, tw, scale, s);
}

hipError_t launch_row_fastconv(const RowConfig &cfg, const float2 *x, long ldx, const float2 *w, long ldw,
                               float2 *y, long ldy, long rows, const float2 *tw, float scale, hipStream_t s)
{
  const Entry *e = find_entry(cfg.n, cfg.variant);
  if (!e) return hipErrorInvalidValue;
  if (rows <= 0) return hipSuccess;
  return e->fconv(x, ldx, w, ldw, y, ldy, rows, tw, scale, s);
}

hipError_t launch_row_fft_split(const RowConfig &cfg, int dir, const float *in_re, const float *in_im, long ld_in,
                                float *out_re, float *out_im, long ld_out, long rows, const float2 *tw, float scale,
                                hipStream_t s)
{
  const Entry *e = find_entry(cfg.n, cfg.variant);
  if (!e) return hipErrorInvalidValue;
  if (rows <= 0) return hipSuccess;
  return e->fft_split(dir, in_re, in_im, ld_in, out_re, out_im, ld_out, rows, tw, scale, s);
}

hipError_t launch_row_fastconv_split(const RowConfig &cfg, const float *xr, const float *xi, long ldx,
                                     const float *wr, const float *wi, long ldw, float *yr, float *yi, long ldy, long rows,
                                     const float2 *tw, float scale, hipStream_t s)
{
  const Entry *e = find_entry(cfg.n, cfg.variant);
  if (!e) return hipErrorInvalidValue;
  if (rows <= 0) return hipSuccess;
  return e->fconv_split(xr, xi, ldx, wr, wi, ldw, yr, yi, ldy, rows, tw, scale, s);
}

} // namespace ovx
