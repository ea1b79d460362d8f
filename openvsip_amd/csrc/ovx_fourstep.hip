// ovx_fourstep.hip -- transforms and fast convolution for lines longer than
// one workgroup's LDS (N > 16384) on gfx950.
//
// A line of N = N1*N2 is viewed as an N1 x N2 row-major matrix,
// n = N2*n1 + n2.  Forward:
//   column pass:  B[k1][n2] = sum_n1 A[n1][n2] W_N1^{n1 k1}
//   row pass:     X[k1 + N1 k2] = sum_n2 W_N^{n2 k1} B[k1][n2] W_N2^{n2 k2}
// The inverse is the same with conjugate factors; the way back of a fastconv
// runs the passes in the other order:
//   row pass:     U[k1][n2] = W_N^{-n2 k1} * sum_k2 X[k1 + N1 k2] W_N2^{-n2 k2}
//   column pass:  x[N2 n1 + n2] = sum_k1 U[k1][n2] W_N1^{-n1 k1}
// Fftm uses column pass + row pass with an LDS-staged transposed store
// (output in natural order).  Fast convolution needs no transpose at all:
// column pass (forward), one row pass doing forward row FFT, multiply by the
// spectrum permuted to [k1][k2] order, inverse row FFT and the inverse
// twiddle, then the inverse column pass -- three passes over HBM.
//
// The column pass moves C adjacent columns per block with the column index
// fastest across lanes, so every global access is a C*8-byte contiguous run.
// W_N^m is rebuilt from two small FP64-generated tables:
// W_N^m = Thi[m >> S] * Tlo[m & (2^S - 1)].
#include "ovx_fs_dev.hpp"

namespace ovx {

template <int L, int P, int C, int DIR, bool SIN, bool SOUT, bool STREAM>
__global__ __launch_bounds__(C *(L / P)) void k_fs_col(FsArgs a, unsigned groups, unsigned rows)
{
  __shared__ float2 lds_all[C * FsLds<L>::LROW];
  long row, group;
  fs_place(blockIdx.x, groups, rows, row, group);
  if (C == 8 && row >= (rows & ~7u)) group = fs_neighbours(group);
  fs_col_body<L, P, C, DIR, SIN, SOUT, STREAM, STREAM && (DIR > 0)>(a, row, group, threadIdx.x, lds_all);
}

template <int L, int P, int C, int DIR, bool SOUT, bool REREAD>
__global__ __launch_bounds__(C *(L / P)) void k_fs_row(FsArgs a, unsigned groups, unsigned rows)
{
  __shared__ float2 lds_all[C * FsLds<L>::LROW];
  long row = blockIdx.x / groups, group = blockIdx.x % groups;
  if (a.placed) fs_place(blockIdx.x, groups, rows, row, group);
  if (C == 8 && !(a.placed && row < (rows & ~7u))) group = fs_neighbours(group);
  fs_row_body<L, P, C, DIR, SOUT, REREAD>(a, row, group, threadIdx.x, lds_all);
}

// 256 threads: fewer lines per workgroup leave it sooner (C = 16 / 4 at 512:
// 56 / 53 us)
template <int L>
struct FsConvCfg {
  static constexpr int C = 256 / FsConv<L>::T;
};
// Sets of `per` rows that the rows of one XCD (an eighth of `whole`) make.
__host__ __device__ static inline int fs_conv_sets(int whole, int per) { return (whole / 8 + per - 1) / per; }

template <int L, bool NATURAL>
__global__ __launch_bounds__(256, 4) void k_fs_conv(FsArgs a, int groups, int rows, int per)
{
  __shared__ float2 lds_all[FsConvCfg<L>::C * FsConv<L>::LROW];
  const int w = (int)blockIdx.x;
  int row0 = w / groups * per, nrows = min(per, rows - row0), step = 1, group = w % groups;
  if (a.placed) { // fs_place()'s rows of one XCD: `per` of the rows x, x + 8, ...
    const int whole = rows & ~7, split = fs_conv_sets(whole, per) * 8 * groups;
    if (w < split) {
      row0 = w / 8 / groups * 8 * per + w % 8;
      nrows = min(per, (whole - row0 + 7) / 8);
      step = 8;
      group = w / 8 % groups;
    } else {
      row0 = whole + (w - split) / groups;
      nrows = 1;
      group = (w - split) % groups;
    }
  }
  fs_conv_body<L, FsConvCfg<L>::C, NATURAL>(a, row0, nrows, step, group, threadIdx.x, lds_all);
}

// Wp[k1][k2] = scale * W[k1 + N1 k2] for `rows` coefficient rows (ldw = 0:
// a single vector): a transposition, 32 x 32 values a workgroup through LDS, so
// that both sides move runs of 256 bytes.  Element by element, reads 8 bytes of
// each line, the whole fastconv with a spectrum per row took 264 us for 64 rows of
// 262144, now 200; one spectrum of 4194304 88 and 79.
__global__ __launch_bounds__(256) void k_fs_permute(const float2 *__restrict__ w, long ldw, float2 *__restrict__ wp,
                                                    unsigned n1, unsigned n2, float scale)
{
  __shared__ float2 tile[32][33];
  const unsigned across = n1 / 32, tx = threadIdx.x % 32, ty = threadIdx.x / 32;
  const unsigned k1 = blockIdx.x % across * 32, k2 = blockIdx.x / across * 32;
  const float2 *src = w + blockIdx.y * ldw + k1 + tx;
#pragma unroll
  for (unsigned i = 0; i < 32; i += 8) tile[ty + i][tx] = src[(long)(k2 + ty + i) * n1];
  __syncthreads();
  float2 *dst = wp + blockIdx.y * ((long)n1 * n2) + k2 + tx;
#pragma unroll
  for (unsigned i = 0; i < 32; i += 8) dst[(long)(k1 + ty + i) * n2] = cscale(tile[tx][ty + i], scale);
}

// ---------------------------------------------------------------- dispatch

// Passes that read or write split storage move 4-byte values, so their
// groups take 32 lines where the thread count allows (128-byte runs per
// array instead of 64).
template <int L>
struct FsSplitCfg {
  static constexpr int P = FsCfg<L>::P;
  static constexpr int C = (L / P) * 32 <= 1024 ? 32 : FsCfg<L>::C;
  static constexpr int NT = C * (L / P);
};

template <int L, int DIR, int C, bool SIN, bool SOUT, bool STREAM>
static hipError_t col_launch_c(const FsArgs &a, long rows, hipStream_t s)
{
  constexpr int P = FsCfg<L>::P;
  const unsigned groups = (unsigned)(a.n2 / C);
  hipLaunchKernelGGL((k_fs_col<L, P, C, DIR, SIN, SOUT, STREAM>), dim3(groups * (unsigned)rows), dim3(C * (L / P)), 0,
                     s, a, groups, (unsigned)rows);
  return hipGetLastError();
}

// Columns per workgroup of the column pass: 16, or 8 where 16 make few
// workgroups or few threads, so that each is done sooner.  16 / 8 columns, us: 256
// x 256, 1 row 3.85 / 3.25, 8 rows 4.25 / 3.68, 256 x 512, 4 rows 4.36 / 3.74, 8
// rows 4.78 / 4.64, 512 x 512, 2 rows 6.65 / 5.20, 4 rows 7.11 / 7.36, 1024 x
// 1024, 1 row 11.6 / 9.5, 4 rows 15.9 / 18.8.  Split storage, read by a call's
// first pass or written by its last, has 32 (FsSplitCfg); 64-byte runs of
// 2048-point columns are not streamed (4 rows 229 us ordinary, 240 streamed).
template <int L, int DIR>
static hipError_t col_launch(const FsArgs &a, long rows, hipStream_t s)
{
  constexpr int C = FsCfg<L>::C;
  if (a.in_re) return col_launch_c<L, DIR, FsSplitCfg<L>::C, true, false, false>(a, rows, s);
  if (a.out_re) return col_launch_c<L, DIR, FsSplitCfg<L>::C, false, true, false>(a, rows, s);
  if constexpr (C == 16) {
    const long groups = a.n2 / C * rows;
    if (groups <= 64 || groups * FsCfg<L>::NT <= 32768) return col_launch_c<L, DIR, 8, false, false, false>(a, rows, s);
    if (a.stream) return col_launch_c<L, DIR, C, false, false, true>(a, rows, s);
  }
  return col_launch_c<L, DIR, C, false, false, false>(a, rows, s);
}

template <int L, int DIR, int C, bool SPLIT, bool REREAD = false>
static hipError_t row_launch_c(FsArgs a, long rows, hipStream_t s)
{
  constexpr int P = FsCfg<L>::P, CL = C < FsSplitCfg<L>::C ? C : FsSplitCfg<L>::C;
  const unsigned groups = (unsigned)(a.n1 / CL);
  a.placed = fs_stays_in_l2(a.nbig, rows);
  hipLaunchKernelGGL((k_fs_row<L, P, CL, DIR, SPLIT, REREAD>), dim3(groups * (unsigned)rows), dim3(CL * (L / P)), 0, s, a,
                     groups, (unsigned)rows);
  return hipGetLastError();
}

// Lines per workgroup of the row pass.  8 up to 64 MB of rows: twice the
// workgroups where they are few, each sooner at its store, and the 64-byte runs
// of neighbouring groups meet in L2; 16 beyond.  16 / 8 lines, us, both
// passes: 256 x 512 lines, 24 rows 23.4 / 22.3, 256 x 256, 1 row 8.4 / 7.6, 512
// x 512, 1 row 14.0 / 12.1, 128 x 256, 100 rows 22.6 / 21.0, 1000 rows 199 / 221;
// 1024 x 1024, 8 rows 66.3 / 60.7.  Split storage, whose runs are half as long:
// 32 lines, 8 where those would leave half the CUs without one (32 / 8, 256 x
// 256, 1 row 10.9 / 8.5, 9 rows 11.8 / 10.3, 24 rows 14.5 / 15.2).
// A result that is read again (REREAD) is better in whole lines: 16 from 320
// workgroups on; real forward, 8 / 16, 63 x 65536 25.4 / 25.0, 256 81.4 / 78.3, 18 x
// 131072 (288 workgroups) 19.2 / 20.2.  Rows off the 128-byte lines
// (fs_whole_lines) are stored the same way, 16 from 144 workgroups on; rows of n +
// 33 values, 8 / 16, 5 x 262144 21.3 / 19.8, 6 20.9 / 22.0, 13 x 131072 19.3 / 18.0, 2 x
// 262144 13.1 / 14.6.
template <int L, int DIR>
static hipError_t row_launch(const FsArgs &a, long rows, hipStream_t s)
{
  if (a.out_re)
    return rows * a.n1 < 128 * 32 ? row_launch_c<L, DIR, 8, true>(a, rows, s)
                                  : row_launch_c<L, DIR, 32, true>(a, rows, s);
  const long bytes = rows * a.nbig * 8;
  const bool whole = fs_whole_lines(a.out, a.ld_out, rows);
  if (a.in_place && whole) return row_launch_c<L, DIR, 8, false, true>(a, rows, s);
  if (a.reread || !whole)
    return rows * a.n1 < (whole ? 320 : 144) * 16 ? row_launch_c<L, DIR, 8, false, true>(a, rows, s)
                                  : row_launch_c<L, DIR, FsCfg<L>::C, false, true>(a, rows, s);
  return bytes <= (64l << 20) ? row_launch_c<L, DIR, 8, false>(a, rows, s)
                                         : row_launch_c<L, DIR, FsCfg<L>::C, false>(a, rows, s);
}

// Rows per workgroup of the middle pass: as many as leave 8 workgroups a CU
// (four rows), or 3 (two; 2 where the rows are in L2): 512 x 512 lines, 64 rows,
// 1 / 2 / 4 / 8 rows 56 / 46 / 44 / 51 us; the whole fastconv, 1 / 2 rows: 512
// x 512, 12 rows 41.3 / 39.3, 9 rows 41.1 / 41.4, 1024 x 1024, 2 rows 41.0 /
// 42.8; in L2, 256 x 512, 24 rows 33.0 / 31.2, 256 x 256, 40 rows 28.8 / 27.8, 32
// rows 24.8 / 24.7, 16 rows 16.5 / 17.2.
int fs_conv_rows(long workgroups, bool placed)
{
  return workgroups >= 4 * 2048 ? 4 : workgroups >= 2 * (placed ? 512 : 768) ? 2 : 1;
}

template <int L>
static hipError_t conv_launch(FsArgs a, long rows, hipStream_t s)
{
  const int groups = (int)(a.n1 / FsConvCfg<L>::C), whole = (int)rows & ~7;
  a.placed = fs_stays_in_l2(a.nbig, rows, true);
  const int per = fs_conv_rows(groups * rows, a.placed);
  const long sets = a.placed ? 8l * fs_conv_sets(whole, per) + (rows - whole) : (rows + per - 1) / per;
  const dim3 grid((unsigned)(groups * sets));
  if (a.natural) {
    if constexpr (L <= 512)
      hipLaunchKernelGGL((k_fs_conv<L, true>), grid, dim3(256), 0, s, a, groups, (int)rows, per);
    else
      return hipErrorInvalidValue;
  } else
    hipLaunchKernelGGL((k_fs_conv<L, false>), grid, dim3(256), 0, s, a, groups, (int)rows, per);
  return hipGetLastError();
}

#define OVX_FS_LENGTHS(X) X(128) X(256) X(512) X(1024) X(2048)

hipError_t launch_fs_col(int dir, const FsArgs &a, long rows, hipStream_t s)
{
  switch (a.n1) {
#define X(L) \
  case L: return dir < 0 ? col_launch<L, -1>(a, rows, s) : col_launch<L, +1>(a, rows, s);
    OVX_FS_LENGTHS(X)
#undef X
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_fs_row(int dir, const FsArgs &a, long rows, hipStream_t s)
{
  switch (a.n2) {
#define X(L) \
  case L: return dir < 0 ? row_launch<L, -1>(a, rows, s) : row_launch<L, +1>(a, rows, s);
    OVX_FS_LENGTHS(X)
#undef X
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_fs_conv(const FsArgs &a, long rows, hipStream_t s)
{
  switch (a.n2) {
#define X(L) \
  case L: return conv_launch<L>(a, rows, s);
    OVX_FS_LENGTHS(X)
#undef X
  default: return hipErrorInvalidValue;
  }
}

int fs_conv_twiddle_count(long l) { return make_plan((int)l, FsConv<128>::P).twtotal; }
hipError_t launch_fs_conv_twiddles(long l, float2 *tw, hipStream_t s)
{
  return launch_twiddles(make_plan((int)l, FsConv<128>::P), tw, s);
}

// tfull[k1 * n2 + c] = W_N^{k1 c}, N = n1 n2, from FP64 values rounded once.
__global__ void k_fs_full_twiddles(long n1, long n2, float2 *__restrict__ out)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = n1 * n2;
  if (i >= n) return;
  const long m = (i / n2) * (i % n2); // < n1 n2
  double sn, cs;
  sincospi(-2.0 * (double)m / (double)n, &sn, &cs);
  out[i] = make_float2((float)cs, (float)sn);
}

hipError_t launch_fs_full_twiddles(long n1, long n2, float2 *out, hipStream_t s)
{
  long n = n1 * n2;
  hipLaunchKernelGGL(k_fs_full_twiddles, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n1, n2, out);
  return hipGetLastError();
}

hipError_t launch_fs_permute(const float2 *w, long ldw, float2 *wp, long n1, long n2, long rows, float scale,
                             hipStream_t s)
{
  const dim3 grid((unsigned)(n1 / 32 * (n2 / 32)), (unsigned)rows);
  hipLaunchKernelGGL(k_fs_permute, grid, dim3(256), 0, s, w, ldw, wp, (unsigned)n1, (unsigned)n2, scale);
  return hipGetLastError();
}

bool fs_length_supported(long l)
{
  switch (l) {
#define X(L) case L:
    OVX_FS_LENGTHS(X)
#undef X
    return true;
  default: return false;
  }
}

} // namespace ovx
