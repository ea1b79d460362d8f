// ovx_overlap.hpp -- whether the lines of two matrices share memory (host).
#pragma once
#include <algorithm>

namespace ovx {

// Whether `lines` lines of n values at a stride of ld and `lines2` at ld2 share
// memory.  Lines that lie between each other's, as the halves of one wide
// matrix do, do not.
template <typename T>
inline bool lines_meet(const T *a, long lines, long ld, const T *b, long lines2, long ld2, long n)
{
  if (a >= b + (lines2 - 1) * ld2 + n || b >= a + (lines - 1) * ld + n) return false;
  const long size = (long)sizeof(T), len = n * size, step2 = ld2 * size;
  const long d = (long)((const char *)a - (const char *)b);
  // line i of a against the first line of b that ends beyond its begin
  auto meets = [&](long i) {
    const long at = d + i * ld * size;
    const long j = at < len || lines2 == 1 ? 0 : (at - len) / step2 + 1;
    return j < lines2 && j * step2 < at + len && at < j * step2 + len;
  };
  // with one stride for both, only the first line of either can be the first to meet
  if (ld == ld2 && lines > 1 && lines2 > 1) {
    if (meets(0)) return true;
    if (d >= 0) return false;
    const long first = (-d - len) / step2; // the lines of a around b's first
    for (long i = std::max(first, 0l); i < std::min(first + 3, lines); ++i)
      if (meets(i)) return true;
    return false;
  }
  for (long i = 0; i < lines; ++i)
    if (meets(i)) return true;
  return false;
}

} // namespace ovx
