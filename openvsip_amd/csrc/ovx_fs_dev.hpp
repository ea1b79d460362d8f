// ovx_fs_dev.hpp -- device bodies of the two-pass four-step kernels (see
// ovx_fourstep.hip for the algorithm), shared by the standalone kernels and
// the persistent batch kernel.
#pragma once
#include "ovx_fourstep.hpp"
#include "ovx_internal.hpp"

namespace ovx {

// LDS stride per line: odd number of float2 so that lanes that differ in the
// line index land on different banks.
template <int L>
struct FsLds {
  static constexpr int LROW = LdsLayout<L, 16>::elems | 1;
};

__device__ __forceinline__ float2 big_twiddle(const float2 *__restrict__ tlo, const float2 *__restrict__ thi,
                                              int sbits, uint32_t m)
{
  float2 lo = tlo[m & ((1u << sbits) - 1u)];
  float2 hi = thi[m >> sbits];
  return cmul(hi, lo);
}

// Row and column group of workgroup w: the groups of a row on one XCD
// (workgroups go to the eight XCDs in turn), so that its accesses cover whole
// matrix rows, not every eighth 128-byte run of each, which at a row of
// 256 columns left an XCD two of its L2's sixteen channels.  256 x 256 lines,
// 256 rows: 58 to 52 us; 512 x 512: 62 to 58.
__device__ __forceinline__ void fs_place(unsigned w, unsigned groups, unsigned rows, long &row, long &group)
{
  const unsigned whole = rows & ~7u;
  if (w < whole * groups) {
    row = (w / 8 / groups) * 8 + w % 8;
    group = (w / 8) % groups;
  } else {
    const unsigned r = w - whole * groups;
    row = whole + r / groups;
    group = r % groups;
  }
}

// Order of a row's groups of 8 (a multiple of 16 of them) dealt to the XCDs in
// turn: the two that share 128-byte lines get the same one, or each line is put
// together from two L2s.  Inverse transform in place, in turn / paired, us: 6 x
// 65536 9.6 / 8.3, 6 x 131072 14.5 / 12.1, 4 x 262144 18.9 / 15.8.
__device__ __forceinline__ long fs_neighbours(long g) { return (g & ~15l) | (g & 7) << 1 | (g >> 3 & 1); }

// The passes' global reads and writes: one row's buffer, element offsets of at
// most N values.  Interleaved lines (a.in, a.out) or, when SPLIT, separate real
// and imaginary arrays (a.in_re / a.in_im, a.out_re / a.out_im).  NT:
// non-temporal (fs_streams_in(), fs_streams_out()).
template <bool SPLIT, bool NT>
__device__ __forceinline__ auto fs_in(const FsArgs &a, long row, uint32_t lane)
{
  if constexpr (SPLIT)
    return IoSx<NT, false>{ make_rsrc(a.in_re + row * a.ld_in, 0xffffffffu),
                            make_rsrc(a.in_im + row * a.ld_in, 0xffffffffu), lane * 4u };
  else
    return IoCx<NT, false>{ make_rsrc(a.in + row * a.ld_in, 0xffffffffu), lane * 8u };
}
template <bool SPLIT, bool NT>
__device__ __forceinline__ auto fs_out(const FsArgs &a, long row, uint32_t lane)
{
  if constexpr (SPLIT)
    return IoSx<false, NT>{ make_rsrc(a.out_re + row * a.ld_out, 0xffffffffu),
                            make_rsrc(a.out_im + row * a.ld_out, 0xffffffffu), lane * 4u };
  else
    return IoCx<false, NT>{ make_rsrc(a.out + row * a.ld_out, 0xffffffffu), lane * 8u };
}

// ---------------------------------------------------------------- column pass
// Column FFT in direction DIR, times a.scale unless 1.  The twiddle
// W_N^{n2 k1} between the two passes is applied by the row pass, where a line's
// table entries are contiguous and serve both sides of a fastconv: read here,
// at the columns' stride, they cost 15 us of a 67 us pass over 134 MB.
// One group of C columns of one row: `group` selects columns
// [group*C, group*C + C), `tid` is the thread within the group's C*(L/P)
// threads, `lds_all` the group's C*LROW LDS elements.
template <int L, int P, int C, int DIR, bool SIN = false, bool SOUT = false, bool NTL = false, bool NTS = false,
          typename LP>
__device__ __forceinline__ void fs_col_body(const FsArgs &a, long row, long group, int tid, LP lds_all)
{
  using E = Engine<L, P>;
  constexpr int T = E::T;
  constexpr int LROW = FsLds<L>::LROW;
  const int c = tid % C;
  const int t = tid / C;
  const uint32_t N2 = (uint32_t)a.n2;
  const uint32_t lane = (uint32_t)t * N2 + (uint32_t)(group * C + c);
  const auto in = fs_in<SIN, NTL>(a, row, lane);
  const auto out = fs_out<SOUT, NTS>(a, row, lane);
  const rsrc_t rtw = make_rsrc(a.tw1, (uint32_t)(E::plan.twtotal + 1) * 8u);
  LP lds = lds_all + c * LROW;

  float2 v[P];
#pragma unroll
  for (int q = 0; q < P; ++q) v[q] = in.ld((uint32_t)(T * q) * N2);
  E::template fft<DIR>(v, lds, t, rtw);
  if (a.scale != 1.0f) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cscale(v[q], a.scale);
  }
#pragma unroll
  for (int q = 0; q < P; ++q) out.st(v[q], (uint32_t)(T * q) * N2);
}

// ---------------------------------------------------------------- row pass
// The twiddles W_N^{k1 n2} of line k1 at the thread's positions n2 = t + T q.
template <int L, int P>
__device__ __forceinline__ void fs_line_twiddles(const FsArgs &a, long k1, int t, float2 (&w)[P])
{
  constexpr int T = L / P;
  if (a.tfull) {
    const float2 *tf = a.tfull + k1 * L;
#pragma unroll
    for (int q = 0; q < P; ++q) w[q] = tf[t + T * q];
  } else {
#pragma unroll
    for (int q = 0; q < P; ++q)
      w[q] = big_twiddle(a.tlo, a.thi, a.sbits, (uint32_t)(t + T * q) * (uint32_t)k1); // < N1 N2
  }
}

// Row pass of a transform in direction DIR: * W_N^{-+ k1 n2}, row FFT,
// transposed store X[k1 + N1 k2], * scale.  One group of C lines k1 in
// [group*C, group*C + C) of one row.
// The result is written once, non-temporally where a run is 64 bytes or more:
// 512 x 512 lines, 24 rows, both passes 42 to 36 us, 64 rows 95 to 88; 256 x
// 256, 256 rows, 84 to 80; runs of 32 bytes (split, 2048 lines) 57 to 75.  REREAD:
// a kernel of the same call reads it again (a real transform's recombination), so
// it is stored the ordinary way: 63 x 65536 real values forward 30.4 us
// non-temporally, 25.3 so, 256 113 and 87.
// Rows off the 128-byte lines are stored so too (fs_whole_lines).
template <int L, int P, int C, int DIR, bool SOUT = false, bool REREAD = false, typename LP>
__device__ __forceinline__ void fs_row_body(const FsArgs &a, long row, long group, int tid, LP lds_all)
{
  // a line's L/P threads are consecutive; when they fit one wavefront its
  // exchanges need no workgroup barrier
  using E = Engine<L, P, line_in_wave(L / P)>;
  constexpr int T = E::T;
  constexpr int LROW = FsLds<L>::LROW;
  const int c = tid / T; // consecutive threads walk along a line
  const int t = tid % T;
  const long k1 = group * C + c;
  const uint32_t N1 = (uint32_t)a.n1;
  const rsrc_t rtw = make_rsrc(a.tw2, (uint32_t)(E::plan.twtotal + 1) * 8u);
  LP lds = lds_all + c * LROW;
  const auto in = fs_in<false, false>(a, row, (uint32_t)k1 * L + t);

  float2 v[P], w[P];
#pragma unroll
  for (int q = 0; q < P; ++q) v[q] = in.ld((uint32_t)(T * q));
  fs_line_twiddles<L, P>(a, k1, t, w);
#pragma unroll
  for (int q = 0; q < P; ++q) v[q] = twmul<DIR>(v[q], w[q]);
  E::template fft<DIR>(v, lds, t, rtw);
  if (a.scale != 1.0f) {
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cscale(v[q], a.scale);
  }
  // transpose through LDS: element k2 of line c -> out[k1_0 + c + N1 k2]
#pragma unroll
  for (int q = 0; q < P; ++q) lds_st(lds, t + T * q, v[q]);
  __syncthreads();
  const int c2 = tid % C;
  const int t2 = tid / C;
  LP lsrc = lds_all + c2 * LROW;
  const auto out = fs_out<SOUT, !REREAD && (C * (SOUT ? 4 : 8) >= 64)>(a, row, (uint32_t)t2 * N1 + (uint32_t)(group * C + c2));
#pragma unroll
  for (int q = 0; q < P; ++q) out.st(lds_ld(lsrc, t2 + T * q), (uint32_t)(T * q) * N1);
}

// Middle pass of a fastconv (in place allowed): * W_N^{k1 n2}, forward row
// FFT, * Wp[k1][k2], inverse row FFT, * W_N^{-k1 n2}; C lines of the nrows rows
// row0, row0 + step, ...  A line's stage twiddles, its W_N entries (the same on both
// sides) and, with one spectrum for all rows, its spectrum stay in registers
// over the rows: what bounded this pass was neither HBM nor latency but the
// loads through L1, 110 of which for 16 values of a line were tables and stage
// twiddles against 16 of data.  8 values per thread leave the registers for
// them (100 of 128 VGPRs; with 16 the 512-point lines spill).  512 x 512
// lines, 64 rows: 63 us with every table read where it is used, 53 with the
// stage twiddles held, 56 with 8 values and W_N held as well (and none of it
// left to the column pass), 46 over 2 rows and 44 over 4; the same loads and
// stores alone take 40.
template <int L>
struct FsConv {
  static constexpr int P = 8;
  static constexpr int T = L / P;
  static constexpr int LROW = LdsLayout<L, P>::elems | 1;
};
// NATURAL: the spectrum is W[k1 + N1 k2], read in runs of the C lines and
// turned over in LDS (fs_takes_natural()).
template <int L, int C, bool NATURAL = false, typename LP>
__device__ __forceinline__ void fs_conv_body(const FsArgs &a, long row0, int nrows, int step, long group, int tid, LP lds_all)
{
  constexpr int P = FsConv<L>::P, T = FsConv<L>::T;
  using E = Engine<L, P, line_in_wave(T)>;
  const int c = tid / T;
  const int t = tid % T;
  const long k1 = group * C + c;
  const rsrc_t rtw = make_rsrc(a.tw2c, (uint32_t)(E::plan.twtotal + 1) * 8u);
  LP lds = lds_all + c * FsConv<L>::LROW;
  const uint32_t lane = (uint32_t)k1 * L + t;
  // this thread's entry of the spectrum: its own in [k1][k2] order, or entry tid,
  // tid + C T, ... of the lines' C values of each k2
  const float2 *wp = a.wp + row0 * a.ldwp;
  if constexpr (NATURAL) wp += group * C + tid % C + (long)(tid / C) * a.n1;
  else wp += k1 * L + t;

  float2 w[P], ws[P], st[E::HELD];
  auto spectrum = [&] {
#pragma unroll
    for (int q = 0; q < P; ++q) {
      if constexpr (NATURAL) ws[q] = cscale(wp[(long)(T * q) * a.n1], a.wscale);
      else ws[q] = wp[T * q];
    }
  };
  // natural order: from entries by number to the thread's own
  auto turn = [&] {
    if constexpr (NATURAL) {
      __syncthreads(); // the exchanges before are done with the lines
#pragma unroll
      for (int q = 0; q < P; ++q) lds_st(lds_all, tid % C * FsConv<L>::LROW + tid / C + T * q, ws[q]);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < P; ++q) ws[q] = lds_ld(lds, t + T * q);
      asm volatile("" ::: "memory"); // read before the line is written again
    }
  };
  fs_line_twiddles<L, P>(a, k1, t, w);
  spectrum();
  E::load_held(t, rtw, st);
#pragma unroll 1
  for (int r = 0; r < nrows; ++r) {
    const auto in = fs_in<false, false>(a, row0 + r * step, lane);
    const auto out = fs_out<false, false>(a, row0 + r * step, lane);
    float2 v[P];
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = in.ld((uint32_t)(T * q));
    if (a.ldwp || r == 0) turn();
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cmul(v[q], w[q]);
    E::template fft_held<-1>(v, lds, t, st);
#pragma unroll
    for (int q = 0; q < P; ++q) v[q] = cmul(v[q], ws[q]);
    if (a.ldwp && r + 1 < nrows) { // one spectrum per row: the next one
      wp += a.ldwp * step;
      spectrum();
    }
    E::template fft_held<+1>(v, lds, t, st);
#pragma unroll
    for (int q = 0; q < P; ++q) out.st(cmulc(v[q], w[q]), (uint32_t)(T * q));
  }
}

// Threads and LDS of one group (C lines of length L, P values per thread).
template <int L>
struct FsCfg {
  static constexpr int P = 16;
  static constexpr int C = (L / P) * 16 <= 1024 ? 16 : 1024 / (L / P);
  static constexpr int NT = C * (L / P);
  static constexpr int LDS = C * FsLds<L>::LROW;
};

} // namespace ovx
