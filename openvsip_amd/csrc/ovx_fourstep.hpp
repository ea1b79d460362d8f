// ovx_fourstep.hpp -- launch interface of the two-pass four-step kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace ovx {

struct FsArgs {
  const float2 *in;
  long ld_in;
  float2 *out;
  long ld_out;
  long n1, n2, nbig;       // N = n1 * n2
  const float2 *tw1, *tw2; // line twiddles of the n1 and n2 plans
  const float2 *tw2c;      // of the n2 plan of a fastconv's middle pass
  const float2 *tlo, *thi; // W_N^m = thi[m >> sbits] * tlo[m & (2^sbits - 1)]
  int sbits;
  const float2 *tfull;     // W_N^{k1 n2} at [k1 * n2count + n2], or null (two-level)
  const float2 *wp;        // fastconv: permuted, scaled spectrum [k1][k2]
  long ldwp;               // 0: one spectrum for every row
  float scale;
  // split storage for a call's first read / last write (separate real and
  // imaginary arrays at the strides ld_in / ld_out); null: in / out are used
  const float *in_re = nullptr, *in_im = nullptr;
  float *out_re = nullptr, *out_im = nullptr;
  // interleaved column pass: non-temporal loads (forward) or loads and stores
  // (inverse), see fs_streams_in / fs_streams_out
  bool stream = false;
};

// Whether the first / last pass of a fastconv over `bytes` of rows goes past
// the caches: X, which is read once, should not push Y out of the 256 MB
// Infinity Cache, nor the result the rows of Y still to be read.  All ordinary
// / first / last / both, us: 64 MB (32 x 262144) 75 / 72 / 77 / 77, 96 MB 106 /
// 106 / 104 / 104, 128 MB 139 / 139 / 133 / 131, 256 MB 285 / 266 / 273 / 257;
// 256 x 65536 127 / 124 / 120 / 120; at 32 MB 41 / 43 / 48 / 49.
inline bool fs_streams_in(size_t bytes) { return bytes >= ((size_t)64 << 20); }
inline bool fs_streams_out(size_t bytes) { return bytes >= ((size_t)96 << 20); }

// Column pass of `rows` rows in direction dir; row pass of a transform; middle
// pass of a fastconv.
hipError_t launch_fs_col(int dir, const FsArgs &a, long rows, hipStream_t s);
hipError_t launch_fs_row(int dir, const FsArgs &a, long rows, hipStream_t s);
hipError_t launch_fs_conv(const FsArgs &a, long rows, hipStream_t s);
// rows per workgroup of a middle pass of that many workgroups of one row
int fs_conv_rows(long workgroups);
// twiddle entries of a middle pass over lines of length l, and the table
int fs_conv_twiddle_count(long l);
hipError_t launch_fs_conv_twiddles(long l, float2 *tw, hipStream_t s);
hipError_t launch_fs_permute(const float2 *w, long ldw, float2 *wp, long n1, long n2, long rows, float scale,
                             hipStream_t s);
bool fs_length_supported(long l);
// Longest transform whose full twiddle table (n entries) the plans keep.
constexpr long kFsFullTwiddleMax = 1l << 18;
hipError_t launch_fs_full_twiddles(long n1, long n2, float2 *out, hipStream_t s);

} // namespace ovx
