// ovx_rowcfg.hpp -- the compiled register-Stockham row configurations.
#pragma once
#include <algorithm>

#include "ovx_engine.hpp"

namespace ovx {

constexpr long kRowCus = 256; // CUs, for rules that go by lines per CU

// Compiled configurations: (N, P).  Rows per block B makes blocks of at
// least 256 threads for short lines.
template <int N, int P>
struct RowCfg {
  static constexpr int T = N / P;
  static constexpr int B = T >= 256 ? 1 : 256 / T;
  static constexpr int NT = T * B;
};

// The launch of `rows` lines.  Lines share a workgroup (RowCfg::B at most) once
// there are more than four workgroups per CU, so that few lines spread over the
// chip; below that as many as fill a wave, whose threads a workgroup has anyway.
// One line a workgroup up to one per CU and packed from there / so, fastconv, us:
// 600 x 2560 16.5 / 13.8, 1300 x 1280 12.4 / 11.2, 3000 x 576 11.9 / 10.5, 1000 x
// 576 5.9 / 5.3; 256 lines of 2 points 2.8 / 2.2, 16 2.5 / 2.4, 72 3.4 / 3.1, 160
// 5.5 / 5.0.  One-thread lines wait for each other's LDS banks in a wave: up to 16
// points they fill half of one (4000 x 12 2.57 us, a whole one 2.72), beyond they
// spread as far as they go (256 x 24 3.0, a whole wave 3.4; 256 x 40 4.0 and 5.4).
template <int N, int P>
struct RowLaunch {
  dim3 grid, block;
  unsigned lds;
  explicit RowLaunch(long rows)
  {
    using C = RowCfg<N, P>;
    constexpr bool ALONE = C::T == 1 && N > 16;
    constexpr long spread = ALONE ? kRowCus : 4 * kRowCus, least = ALONE || C::T > 64 ? 1 : C::T == 1 ? 32 : 64 / C::T;
    const long packed = std::max<long>((rows + spread - 1) / spread, least);
    const long b = std::max<long>(std::min({ (long)C::B, packed, rows }), 1);
    grid = dim3((unsigned)((rows + b - 1) / b));
    block = dim3((unsigned)(b * C::T));
    lds = C::B == 1 ? 0 : (unsigned)(b * Engine<N, P>::LROW * sizeof(float2));
  }
};

// Which lines a block handles: blockDim.x / T lines of T threads each, lines
// contiguous in memory at stride ld.  Out-of-range lines (the tail block)
// compute on zeros and store nothing, but still take part in every barrier.
// Several lines' LDS is sized at launch (one row region per line); a line that
// has the workgroup to itself has its region as a static array, whose address
// the compiler folds into the accesses (sized at launch, fastconv 256 x 16384
// took 25.4 instead of 24.5 us).
extern __shared__ float2 row_lds[];

template <int N, int P>
struct RowPlace {
  using E = Engine<N, P, line_in_wave(N / P)>;
  static constexpr bool ONE = RowCfg<N, P>::B == 1;
  int lrow, t;
  long row0;
  float2 *lds;
  __device__ __forceinline__ RowPlace()
  {
    lrow = ONE ? 0 : (int)threadIdx.x / E::T;
    t = ONE ? (int)threadIdx.x : (int)threadIdx.x % E::T;
    row0 = ONE ? (long)blockIdx.x : (long)blockIdx.x * (long)(blockDim.x / E::T);
    if constexpr (ONE) {
      __shared__ float2 line[E::LROW];
      lds = line;
    } else {
      lds = row_lds + lrow * E::LROW;
    }
  }
};

// X(N, P): every compiled configuration, a length's in the order of its variant
// numbers.  P is chosen per length by measurement (one launch, fastconv of 1,
// 256 and 4000 lines of data that no cache holds, us):
//   fewer values per thread put more threads on a line, which is what a few
//   lines need (2304: P 36 9.7 / 10.8, P 12 5.6 / 6.7; 384: P 24 6.7 / 7.6,
//   P 6 4.2 / 4.9; 2048: P 16 5.9 / 6.9, P 8 4.6 / 5.7), more values per thread
//   save stages, which is what many lines need (1536 at 4000: P 12 30.1, P 24
//   25.1; 1024 at 4000: P 8 21.5, P 16 17.2).
// Where one P is best or within a few per cent everywhere it is the only one;
// else row_pick() chooses by the number of lines.  16 values per thread at
// powers of two from 64 and 12 at 3072, 6144 and 12288 are also what the
// four-step, overlap-save and batch kernels run; 8 at 128 points is there for
// the overlap-save segments alone.
#define OVX_ROW_CONFIGS(X)                                                      \
  X(2, 2) X(4, 4) X(8, 8) X(16, 4) X(32, 4) X(64, 4) X(64, 16) X(128, 4)        \
  X(128, 16) X(128, 8) X(256, 4) X(256, 16) X(512, 8) X(512, 16) X(1024, 16) X(1024, 8)   \
  X(2048, 16) X(2048, 8) X(4096, 16) X(8192, 16) X(16384, 16)                   \
  X(3, 3) X(6, 6) X(12, 12) X(24, 24) X(48, 6) X(96, 6) X(192, 6) X(384, 12)    \
  X(384, 6) X(768, 12) X(1536, 24) X(1536, 12) X(3072, 12) X(6144, 24)          \
  X(6144, 12) X(12288, 24) X(12288, 12)                                         \
  X(5, 5) X(10, 10) X(20, 20) X(40, 40) X(80, 10) X(160, 10) X(320, 20)         \
  X(640, 20) X(640, 10) X(1280, 20) X(2560, 20) X(5120, 20) X(10240, 40)        \
  X(9, 9) X(18, 18) X(36, 36) X(72, 6) X(144, 12) X(288, 12) X(576, 24)         \
  X(576, 12) X(1152, 12) X(2304, 12) X(4608, 12) X(9216, 24)

} // namespace ovx
