// ovx_rowcfg.hpp -- the compiled register-Stockham row configurations.
#pragma once

namespace ovx {

// Compiled configurations: (N, P).  Rows per block B makes blocks of at
// least 256 threads for short lines.
template <int N, int P>
struct RowCfg {
  static constexpr int T = N / P;
  static constexpr int B = T >= 256 ? 1 : 256 / T;
  static constexpr int NT = T * B;
};

// X(N, P): every compiled configuration; the first listed for an N is
// variant 0 (the default).
#define OVX_ROW_CONFIGS(X)                                                      \
  X(2, 2) X(4, 4) X(8, 8) X(16, 16) X(32, 16) X(64, 16) X(128, 16) X(256, 16)   \
  X(512, 16) X(1024, 16) X(2048, 16) X(4096, 16) X(8192, 16) X(16384, 16)       \
  X(3, 3) X(6, 6) X(12, 12) X(24, 24) X(48, 24) X(96, 24) X(192, 24)            \
  X(384, 24) X(768, 24) X(1536, 24) X(3072, 24) X(6144, 24) X(12288, 24)       \
  X(3072, 12) X(6144, 12) X(12288, 12)                                          \
  X(5, 5) X(10, 10) X(20, 20) X(40, 40) X(80, 40) X(160, 40) X(320, 40)         \
  X(640, 40) X(1280, 40) X(2560, 40) X(5120, 40) X(10240, 40)                 \
  X(9, 9) X(18, 18) X(36, 36) X(72, 36) X(144, 36) X(288, 36) X(576, 36)       \
  X(1152, 36) X(2304, 36) X(4608, 36) X(9216, 36)

} // namespace ovx
