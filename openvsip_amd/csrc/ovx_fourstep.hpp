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
  // wp is instead the spectrum in natural order, W[k1 + N1 k2], to be scaled by
  // wscale (fs_takes_natural)
  bool natural = false;
  float wscale = 1.0f;
  float scale;
  // split storage for a call's first read / last write (separate real and
  // imaginary arrays at the strides ld_in / ld_out); null: in / out are used
  const float *in_re = nullptr, *in_im = nullptr;
  float *out_re = nullptr, *out_im = nullptr;
  // interleaved column pass: non-temporal loads (forward) or loads and stores
  // (inverse), see fs_streams_in / fs_streams_out
  bool stream = false;
  // row pass: the result is read again in this call; it takes the input's place
  // and is stored the ordinary way (fs_keeps_in_place)
  bool reread = false;
  bool in_place = false;
  // row and middle passes: each row on the XCD of its column pass
  // (fs_stays_in_l2)
  bool placed = false;
};

// Whether a call's rows stay in the eight XCDs' L2s (4 MB each) from pass to
// pass: the column pass works each row on one XCD, the next pass then does the
// same.  Otherwise its groups go to the XCDs in turn, which suits rows that are
// not in L2 better.  In turn / on the row's XCD, us: fastconv 256 x 256 lines,
// 9 rows 16.8 / 14.7, 24 25.9 / 21.7, 40 33.0 / 27.8, 64 38.6 / 36.7, 96 54.0 /
// 54.2; 256 x 512, 24 rows 35.9 / 31.2.  Fftm 256 x 256, 24 rows 16.5 / 13.3, 256 x
// 512, 24 rows 22.3 / 21.7.  Of rows of 2 MB an L2 holds one beside what is being
// loaded, so eight of them, the middle pass, which works in place, two more: Fftm
// 512 x 512, 8 rows 20.9 / 20.1, in place 22.7 / 20.9, 9 rows 24.0 / 25.0; fastconv 8
// rows 37.4 / 31.5, in place 42.5 / 30.1, 9 rows 41.2 / 38.5, 10 40.4 / 39.7, 12 40.8 /
// 44.2.
inline bool fs_stays_in_l2(long n, long rows, bool middle = false)
{
  const long row = n * 8, all = rows * row;
  if (row <= (1l << 20)) return all <= 8 * (4l << 20);
  return row <= (2l << 20) && rows >= 8 && all <= (middle ? 10 : 8) * (2l << 20);
}

// Whether every row begins on a 128-byte line.  Runs of other rows straddle
// lines: each part loaded or stored past the caches is a memory access of its
// own, where ordinary ones meet in L2.  Rows of n + 33 values, past the caches /
// ordinary, us: fastconv 64 x 262144 225 / 160, 50 x 262144 179 / 135, 200 x
// 65536 167 / 115 (n + 8 values 132 / 115); transforms (last pass) 20 x 262144 55 /
// 45, 8 x 262144 28.2 / 22.0, 24 x 131072 32.2 / 24.9, 30 x 65536 21.2 / 17.6.
inline bool fs_whole_lines(const float2 *p, long ld, long rows)
{
  return (size_t)p % 128 == 0 && (rows == 1 || ld % 16 == 0);
}

// Whether the first / last pass of a fastconv over `bytes` of rows goes past
// the caches: X, which is read once, should not push Y out of the 256 MB
// Infinity Cache, nor the result the rows of Y still to be read.  All ordinary
// / first / last / both, us: 64 MB (32 x 262144) 75 / 72 / 77 / 77, 96 MB 106 /
// 106 / 104 / 104, 128 MB 139 / 139 / 133 / 131, 256 MB 285 / 266 / 273 / 257;
// 256 x 65536 127 / 124 / 120 / 120; at 32 MB 41 / 43 / 48 / 49.
inline bool fs_streams_in(size_t bytes) { return bytes >= ((size_t)64 << 20); }
inline bool fs_streams_out(size_t bytes) { return bytes >= ((size_t)96 << 20); }

// Whether the result of a transform in place of a caller's data is stored the
// ordinary way: the column pass has left the lines it replaces in the caches
// (where the call itself has just written them, before a real inverse transform,
// it is the slower way: 24 x 524288 real values 59.4 / 64.5, 48 x 262144 54.4 /
// 58.8).  Non-temporal /
// ordinary stores, in place, us: 128 x 32768 29.7 / 26.7, 64 x 65536 30.5 / 27.5, 32
// x 131072 31.8 / 30.1, 20 x 262144 39.0 / 37.3, 12 x 524288 47.9 / 47.2, 6 x
// 1048576 56.2 / 52.4, 4 x 2097152 75.8 / 71.4; fewer or more rows, 64 x 32768
// 16.8 / 17.8, 32 x 65536 17.4 / 18.1, 256 x 65536 88 / 93.
inline bool fs_keeps_in_place(const void *in, const void *out, size_t bytes)
{
  return in == out && bytes >= ((size_t)20 << 20) && bytes <= ((size_t)64 << 20);
}

// Whether the middle pass reads spectra in natural order itself, or
// launch_fs_permute lays them out first.  The C neighbouring lines of a
// workgroup (16 to 4 up to 512 points) make runs of 128 to 32 bytes, which
// neighbouring groups complete in L2; 32-byte runs only pay while the call fits
// there.  Laid out / natural, us: 256-point lines, one spectrum, 1 row of 65536
// 12.8 / 10.9, a spectrum per row, 64 rows 54.4 / 42.4, 256 rows 190 / 169;
// 512-point lines, one spectrum, 1 row of 262144 18.9 / 16.6, a spectrum per row,
// 24 rows of 131072 42.9 / 37.5, 100 rows 151 / 162, 16 rows of 262144 57.5 / 62.2.
inline bool fs_takes_natural(long n2, long n, long rows)
{
  return n2 <= 256 || (n2 == 512 && rows * n * 8 < 8 * (4l << 20));
}

// Column pass of `rows` rows in direction dir; row pass of a transform; middle
// pass of a fastconv.
hipError_t launch_fs_col(int dir, const FsArgs &a, long rows, hipStream_t s);
hipError_t launch_fs_row(int dir, const FsArgs &a, long rows, hipStream_t s);
hipError_t launch_fs_conv(const FsArgs &a, long rows, hipStream_t s);
// rows per workgroup of a middle pass of that many workgroups of one row
int fs_conv_rows(long workgroups, bool placed);
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
