// ovx_corr.cpp -- FFT-based Correlation and Convolution plans (C-ABI part).
//
// Semantics follow the reference's direct implementations:
//   Correlation::correlate   src/ovxx/signal/corr.hpp:663-719
//   corr_full/same/min       src/ovxx/signal/corr.hpp:91-215
//   output sizes             support/test/ref/corr.hpp:24-36,
//                            src/ovxx/signal/conv.hpp:103-121
//   kernel symmetry          src/ovxx/signal/conv.hpp:144-175
//   conv_full/same/min       src/ovxx/signal/conv.hpp:232-330
// The arithmetic is overlap-save on the gfx950 FFT engine (ovx_ols.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <new>
#include <vector>

#include "ovx_hier.hpp"
#include "ovx_ols.hpp"
#include "ovx_plan.hpp"

namespace ovx {

struct CorrState {
  int is_conv = 0;
  int support = 0;
  long M = 0, N = 0, P = 0, D = 1;
  long out_off = 0;
  int L = 0;
  LineFFT fftL;
  int Lp = 0; // values per thread of a segment
  DevBuf H, ref_stage, in_stage, out_stage;
};

// Segments of length L over the plan's outputs.
static long segment_count(const CorrState &c, int L)
{
  const long span = (c.P - 1) * c.D + 1, step = L - (c.M - 1);
  return (span + step - 1) / step;
}

// Segments up to which a segment is a matter of latency: four per CU.
constexpr long kOlsFew = 1024;

// Segment length: the shortest power of two from 512 of which the kernel
// overlap takes no more than half (the chain of stages is what a call waits
// for: 65536 x 1024 takes 7.6 us in segments of 2048 and 11.6 in segments of
// 4096), and while there are more segments than the chip runs at once, twice
// that until the overlap is under 30 % (2 * 10^6 x 513: 17.5 us in segments
// of 1024, 13.9 in 2048, 14.0 in 4096).  Few samples keep the length of which
// the overlap takes no more than a quarter: the rounding error of an output goes
// with the root of the samples in a segment over its length, and next to a long
// segment's padding a short one's would be up to 1.4 times larger (1630 x 574,
// unbiased, 1.9e-6 in segments of 2048, 1.5e-6 in 4096).  Kernels of up to 33
// values keep segments of which the overlap takes a quarter for the same
// reason, fewer levels of rounding: error against 64 bits and time of 126694 x
// 17, segments of 64 / 512, 1.45e-7 / 1.70e-7 and 3.6 / 4.6 us, of 126694 x 33,
// 128 / 512, 1.58e-7 / 1.73e-7 and 4.6 / 4.7 us (2 * 10^6 x 17 13.4 / 12.6, x 33
// 13.6 / 13.3).
static int choose_L(const CorrState &c)
{
  if (c.M <= 17) return 64;
  if (c.M <= 33) return 128;
  long L = 512, longer = 512;
  while (L < 2 * (c.M - 1) && L < kMaxRowN) L *= 2;
  while (longer < 4 * (c.M - 1) && longer < kMaxRowN) longer *= 2;
  while (L < longer && c.N * L < longer * (L - (c.M - 1))) L *= 2;
  while (L < kMaxRowN && segment_count(c, (int)L) > kOlsFew && 10 * (c.M - 1) > 3 * L) L *= 2;
  return (int)L;
}

// The reference's spectrum in every segment or once in a launch of its own.
// Short segments: 5 * 10^5 x 17 6.6 us with the launch, 5.3 without, 1.2 * 10^6 x
// 17 10.0 and 9.4, 2 * 10^6 x 17 13.5 either way.
static bool ols_fuse_ref(const CorrState &c)
{
  return !c.is_conv && (c.L < 512 || segment_count(c, c.L) <= kOlsFew);
}

// Whether two runs of values share memory.
static bool runs_meet(const float2 *a, long na, const float2 *b, long nb) { return a < b + nb && b < a + na; }

// A single segment reads all of its samples before its first store, so a result
// over the signal is right; several segments run at once and store over each
// other's samples.  A signal of which one segment of the greatest length could
// hold all that the outputs need is copied out of the result's way then (with a
// decimation the signal itself may be longer).
static bool ols_copies_meeting(const CorrState &c)
{
  return segment_count(c, c.L) > 1 && (c.N <= kMaxRowN || (c.P - 1) * c.D + 1 + c.M - 1 <= kMaxRowN);
}

// Puts the samples in `in` out of the way of a result over them.
static int ols_copy_input(CorrState &c, const float2 *&in, hipStream_t s)
{
  hipError_t e = hipMemcpyAsync(c.in_stage.p, in, (size_t)c.N * 8, hipMemcpyDeviceToDevice, s);
  in = (const float2 *)c.in_stage.p;
  return e == hipSuccess ? OVX_OK : hip_fail(e, "signal copy");
}

static int ols_init(CorrState &c)
{
  if (c.M - 1 >= kMaxRowN) return fail(OVX_ERR_UNSUPPORTED, "kernel length %ld too long for overlap-save", c.M);
  c.L = choose_L(c);
  c.Lp = c.L == 64 ? 4 : c.L <= 2048 ? 8 : 16;
  // the overlap-save kernels are built on the register-Stockham engine: take
  // the configuration of that length and values per thread and its twiddles
  int st = c.fftL.init(c.L, LineFFT::row_variant(c.L, row_config_with(c.L, c.Lp)));
  if (st) return st;
  if (c.fftL.kind != LineFFT::LDS || c.fftL.rc.p != c.Lp || !c.fftL.tw.p)
    return fail(OVX_ERR_UNSUPPORTED, "no register-Stockham configuration for segment length %d", c.L);
  if ((st = c.H.alloc((size_t)c.L * 8))) return st;
  return ols_copies_meeting(c) ? c.in_stage.alloc((size_t)c.N * 8) : OVX_OK;
}

// H = FFT_L(h padded); h is a device pointer of M values
static int ols_spectrum(CorrState &c, const float2 *h, int reverse, hipStream_t s)
{
  hipError_t e = launch_ols_spectrum(c.L, c.Lp, h, c.M, reverse, (float2 *)c.H.p, (const float2 *)c.fftL.tw.p, s);
  return e == hipSuccess ? OVX_OK : hip_fail(e, "kernel spectrum");
}

// ref: the correlation's reference when its spectrum is not in c.H
static int ols_run(CorrState &c, const float2 *ref, const float2 *in, float2 *out, int conj_input, int unbiased,
                   hipStream_t s)
{
  if (c.fftL.kind != LineFFT::LDS || !c.fftL.tw.p || !(ref || c.H.p))
    return fail(OVX_ERR_STATE, "overlap-save plan has no twiddle table");
  OlsArgs a{};
  a.in = in;
  a.N = c.N;
  a.M = c.M;
  a.H = ref ? nullptr : (const float2 *)c.H.p;
  a.h = ref;
  a.tw = (const float2 *)c.fftL.tw.p;
  a.scale = 1.0f / (float)c.L;
  a.conj_input = conj_input;
  a.unbiased = unbiased;
  a.support = c.support;
  a.decimation = c.P > 1 ? c.D : 1; // a single output is c[out_off] whatever the decimation
  a.dmagic = ols_magic(a.decimation);
  a.out_off = c.out_off;
  a.c_first = c.out_off;
  a.c_step = c.L - (c.M - 1);
  a.P = c.P;
  a.out = out;
  hipError_t e = launch_ols(c.L, c.Lp, a, segment_count(c, c.L), s);
  if (e != hipSuccess) return hip_fail(e, "overlap-save launch");
  return OVX_OK;
}

} // namespace ovx

using namespace ovx;

ovx_plan_s::~ovx_plan_s()
{
  delete corr;
}

const char *ovx_plan_s::name() const
{
  switch (kind) {
  case PLAN_FFTM: return line.kind == LineFFT::LDS ? "fftm:lds-resident" : line.kind == LineFFT::FOURSTEP ? "fftm:four-step" : line.kind == LineFFT::HIER ? "fftm:hierarchical-lds" : "fftm:none";
  case PLAN_FFT:
    return line.kind == LineFFT::LDS        ? "fft:lds-resident"
           : line.kind == LineFFT::FOURSTEP ? "fft:four-step"
           : line.kind == LineFFT::HIER     ? "fft:hierarchical-lds"
                                            : "fft:none";
  case PLAN_FASTCONV:
    if (bf16x3) return "fastconv:bf16x3-mfma";
    return line.kind == LineFFT::LDS        ? "fastconv:fused-lds-resident"
           : line.kind == LineFFT::FOURSTEP ? "fastconv:four-step-3pass"
           : line.kind == LineFFT::HIER     ? "fastconv:fused-hierarchical-lds"
                                            : "fastconv:none";
  case PLAN_FFTM_REAL:
    return dir == OVX_FFT_FWD ? "fftm-real:r2c-half-length" : "fftm-real:c2r-half-length";
  case PLAN_CORR: return "corr:overlap-save";
  case PLAN_CONV: return "conv:overlap-save";
  default: return "unknown";
  }
}

size_t ovx_plan_s::device_bytes() const
{
  size_t b = line.device_bytes() + stage_in.bytes + stage_out.bytes + stage_w.bytes + u256.bytes + wtab.bytes +
             split_ws.bytes;
  if (corr)
    b += corr->fftL.device_bytes() + corr->H.bytes + corr->ref_stage.bytes +
         corr->in_stage.bytes + corr->out_stage.bytes;
  return b;
}

// ---------------------------------------------------------------- correlation
extern "C" long ovx_corr_output_size(int support, long m, long n)
{
  if (support == OVX_SUPPORT_FULL) return n + m - 1;
  if (support == OVX_SUPPORT_SAME) return n;
  return n - m + 1;
}

extern "C" int ovx_corr_plan_create(ovx_plan *plan, int support, long m, long n, unsigned flags)
{
  if (!plan) return fail(OVX_ERR_INVALID, "null plan pointer");
  *plan = nullptr;
  if (support < OVX_SUPPORT_FULL || support > OVX_SUPPORT_MIN) return fail(OVX_ERR_INVALID, "bad support");
  // corr_full requires ref_size <= in_size (corr.hpp:103)
  if (m < 1 || n < 1 || m > n) return fail(OVX_ERR_INVALID, "bad sizes m=%ld n=%ld (need 1 <= m <= n)", m, n);
  std::unique_ptr<ovx_plan_s> p(new (std::nothrow) ovx_plan_s());
  if (!p) return fail(OVX_ERR_NOMEM, "host allocation");
  p->kind = PLAN_CORR;
  p->flags = flags;
  p->corr = new (std::nothrow) CorrState();
  if (!p->corr) return fail(OVX_ERR_NOMEM, "host allocation");
  CorrState &c = *p->corr;
  c.support = support;
  c.M = m;
  c.N = n;
  c.P = ovx_corr_output_size(support, m, n);
  c.D = 1;
  long shift = support == OVX_SUPPORT_FULL ? m - 1 : support == OVX_SUPPORT_SAME ? m / 2 : 0;
  c.out_off = m - 1 - shift;
  int st = ols_init(c);
  if (st) return st;
  *plan = p.release();
  return OVX_OK;
}

extern "C" int ovx_corr_exec(ovx_plan p, int bias, const void *ref, const void *in, void *out, void *stream)
{
  if (!p || p->kind != PLAN_CORR) return fail(OVX_ERR_INVALID, "not a correlation plan");
  if (!ref || !in || !out) return fail(OVX_ERR_INVALID, "null data pointer");
  if (bias != OVX_BIASED && bias != OVX_UNBIASED) return fail(OVX_ERR_INVALID, "bad bias");
  CorrState &c = *p->corr;
  hipStream_t s = (hipStream_t)stream;
  const float2 *dref = (const float2 *)ref, *din = (const float2 *)in;
  float2 *dout = (float2 *)out;
  int st;
  bool host = p->flags & OVX_FLAG_HOST_POINTERS;
  if (host) {
    if ((st = c.ref_stage.alloc((size_t)c.M * 8)) || (st = c.in_stage.alloc((size_t)c.N * 8)) ||
        (st = c.out_stage.alloc((size_t)c.P * 8)))
      return st;
    hipError_t e = hipMemcpyAsync(c.ref_stage.p, ref, (size_t)c.M * 8, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(c.in_stage.p, in, (size_t)c.N * 8, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return hip_fail(e, "H2D copy");
    dref = (const float2 *)c.ref_stage.p;
    din = (const float2 *)c.in_stage.p;
    dout = (float2 *)c.out_stage.p;
  }
  // a reference that the result is written over is read whole by a launch of
  // its own first
  const bool fuse = ols_fuse_ref(c) && !runs_meet(dref, c.M, dout, c.P);
  const bool copy = !host && runs_meet(din, c.N, dout, c.P) && ols_copies_meeting(c);
  const bool scratch = !host && (copy || !fuse);
  if (scratch && (st = order_plan(p, s))) return st;
  if (copy && (st = ols_copy_input(c, din, s))) return st;
  if (!fuse && (st = ols_spectrum(c, dref, 1, s))) return st;
  if ((st = ols_run(c, fuse ? dref : nullptr, din, dout, 1, bias == OVX_UNBIASED, s))) return st;
  if (scratch) return mark_plan(p, s, OVX_OK);
  if (host) {
    hipError_t e = hipMemcpyAsync(out, c.out_stage.p, (size_t)c.P * 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_fail(e, "D2H copy");
  }
  return OVX_OK;
}

// ---------------------------------------------------------------- convolution
extern "C" long ovx_conv_output_size(int support, long m, long n, long d)
{
  if (d < 1) return -1;
  if (support == OVX_SUPPORT_FULL) return ((n + m - 2) / d) + 1;
  if (support == OVX_SUPPORT_SAME) return ((n - 1) / d) + 1;
  // VSIP_IMPL_CONV_CORRECT_MIN_SUPPORT_SIZE == 1 (conv.hpp:36, 115-117)
  return ((n - m + 1) / d) + ((n - m + 1) % d == 0 ? 0 : 1);
}

extern "C" int ovx_conv_plan_create(ovx_plan *plan, int symmetry, int support, const void *coeff, long mc, long n,
                                    long decimation, unsigned flags)
{
  if (!plan) return fail(OVX_ERR_INVALID, "null plan pointer");
  *plan = nullptr;
  if (!coeff) return fail(OVX_ERR_INVALID, "null coefficients");
  if (support < OVX_SUPPORT_FULL || support > OVX_SUPPORT_MIN) return fail(OVX_ERR_INVALID, "bad support");
  if (symmetry < OVX_NONSYM || symmetry > OVX_SYM_EVEN_LEN_EVEN) return fail(OVX_ERR_INVALID, "bad symmetry");
  if (mc < 1 || n < 1 || decimation < 1) return fail(OVX_ERR_INVALID, "bad sizes");
  // kernel from coefficients and symmetry (conv.hpp:144-175); coefficients
  // are host data here, as the reference copies them at construction.
  const float2 *cf = (const float2 *)coeff;
  std::vector<float2> k;
  if (symmetry == OVX_SYM_EVEN_LEN_ODD) {
    k.assign(cf, cf + mc);
    for (long i = 0; i < mc - 1; ++i) k.push_back(cf[mc - 2 - i]);
  } else if (symmetry == OVX_SYM_EVEN_LEN_EVEN) {
    k.assign(cf, cf + mc);
    for (long i = 0; i < mc; ++i) k.push_back(cf[mc - 1 - i]);
  } else {
    k.assign(cf, cf + mc);
  }
  long m = (long)k.size();
  if (support == OVX_SUPPORT_MIN && m > n) return fail(OVX_ERR_INVALID, "kernel longer than input for min support");
  std::unique_ptr<ovx_plan_s> p(new (std::nothrow) ovx_plan_s());
  if (!p) return fail(OVX_ERR_NOMEM, "host allocation");
  p->kind = PLAN_CONV;
  p->flags = flags;
  p->corr = new (std::nothrow) CorrState();
  if (!p->corr) return fail(OVX_ERR_NOMEM, "host allocation");
  CorrState &c = *p->corr;
  c.is_conv = 1;
  c.support = support;
  c.M = m;
  c.N = n;
  c.D = decimation;
  c.P = ovx_conv_output_size(support, m, n, decimation);
  c.out_off = support == OVX_SUPPORT_FULL ? 0 : support == OVX_SUPPORT_SAME ? m / 2 : m - 1;
  int st = ols_init(c);
  if (st) return st;
  if ((st = c.ref_stage.alloc((size_t)m * 8))) return st;
  hipError_t e = hipMemcpy(c.ref_stage.p, k.data(), (size_t)m * 8, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_fail(e, "coefficient upload");
  if ((st = ols_spectrum(c, (const float2 *)c.ref_stage.p, 0, nullptr))) return st;
  e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) return hip_fail(e, "kernel spectrum");
  *plan = p.release();
  return OVX_OK;
}

extern "C" int ovx_conv_exec(ovx_plan p, const void *in, void *out, void *stream)
{
  if (!p || p->kind != PLAN_CONV) return fail(OVX_ERR_INVALID, "not a convolution plan");
  if (!in || !out) return fail(OVX_ERR_INVALID, "null data pointer");
  CorrState &c = *p->corr;
  hipStream_t s = (hipStream_t)stream;
  const float2 *din = (const float2 *)in;
  float2 *dout = (float2 *)out;
  int st;
  bool host = p->flags & OVX_FLAG_HOST_POINTERS;
  if (host) {
    if ((st = c.in_stage.alloc((size_t)c.N * 8)) || (st = c.out_stage.alloc((size_t)c.P * 8))) return st;
    hipError_t e = hipMemcpyAsync(c.in_stage.p, in, (size_t)c.N * 8, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return hip_fail(e, "H2D copy");
    din = (const float2 *)c.in_stage.p;
    dout = (float2 *)c.out_stage.p;
  }
  const bool copy = !host && runs_meet(din, c.N, dout, c.P) && ols_copies_meeting(c);
  if (copy && ((st = order_plan(p, s)) || (st = ols_copy_input(c, din, s)))) return st;
  if ((st = ols_run(c, nullptr, din, dout, 0, 0, s))) return st;
  if (copy) return mark_plan(p, s, OVX_OK);
  if (host) {
    hipError_t e = hipMemcpyAsync(out, c.out_stage.p, (size_t)c.P * 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_fail(e, "D2H copy");
  }
  return OVX_OK;
}
