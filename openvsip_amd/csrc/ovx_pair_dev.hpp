// ovx_pair_dev.hpp -- a pair (k, N - k) of a half-length complex transform and of
// the real line's half spectrum, for the one-pass and the two-pass real
// transforms (see ovx_row_dev.hpp and ovx_real.hip).
#pragma once
#include "ovx_device.hpp"

namespace ovx {

__device__ __forceinline__ void r2c_pair(float2 zk, float2 zm, float2 w, float scale, float2 &xk, float2 &xm)
{
  const float2 e = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
  const float2 o = make_float2(0.5f * (zk.y + zm.y), -0.5f * (zk.x - zm.x));
  const float2 wo = cmul(w, o);
  const float2 d = csub(e, wo);
  xk = cscale(cadd(e, wo), scale);
  xm = cscale(make_float2(d.x, -d.y), scale);
}
__device__ __forceinline__ void c2r_pair(float2 xk, float2 xm, float2 w, float2 &zk, float2 &zm)
{
  const float2 a = make_float2(xk.x + xm.x, xk.y - xm.y);
  const float2 c = cmulc(make_float2(xk.x - xm.x, xk.y + xm.y), w);
  zk = make_float2(a.x - c.y, a.y + c.x);
  zm = make_float2(a.x + c.y, c.x - a.y);
}

} // namespace ovx
