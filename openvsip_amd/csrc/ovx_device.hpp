// ovx_device.hpp -- device-side building blocks for the gfx950 FFT kernels.
//
// Complex values are float2 (re, im), the interleaved complex<float> layout
// OpenVSIP uses by default (src/ovxx/storage/block.hpp:27-42).  DIR is the
// transform exponent sign: -1 forward, +1 inverse
// (src/ovxx/signal/fft/util.hpp:43-51).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

namespace ovx {

// ---------------------------------------------------------------- complex
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
  return make_float2(__builtin_fmaf(a.x, b.x, -a.y * b.y), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b)
{
  return make_float2(__builtin_fmaf(a.x, b.x, a.y * b.y), __builtin_fmaf(a.y, b.x, -a.x * b.y));
}
// multiply by the table twiddle w (stored for the forward sign); the inverse
// direction uses its conjugate.
template <int DIR>
__device__ __forceinline__ float2 twmul(float2 a, float2 w)
{
  if constexpr (DIR < 0) return cmul(a, w);
  else return cmulc(a, w);
}
// a * (DIR * i): forward multiplies by -i, inverse by +i.
template <int DIR>
__device__ __forceinline__ float2 rot(float2 a)
{
  if constexpr (DIR < 0) return make_float2(a.y, -a.x);
  else return make_float2(-a.y, a.x);
}

// ---------------------------------------------------------------- small DFTs
// In-place DFT of R values in natural order: y_k = sum_n x_n W_R^{nk},
// W_R = exp(DIR*2*pi*i/R).
template <int R, int DIR> struct Dft;

template <int DIR> struct Dft<1, DIR> {
  __device__ __forceinline__ static void run(float2 *) {}
};

template <int DIR> struct Dft<2, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  }
};

template <int DIR> struct Dft<3, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    const float c = -0.5f, s = 0.86602540378443864676f; // cos, sin(2pi/3)
    float2 a = v[0], t = cadd(v[1], v[2]), d = csub(v[1], v[2]);
    float2 m = make_float2(__builtin_fmaf(c, t.x, a.x), __builtin_fmaf(c, t.y, a.y));
    float2 r = rot<DIR>(cscale(d, s));
    v[0] = cadd(a, t);
    v[1] = cadd(m, r);
    v[2] = csub(m, r);
  }
};

template <int DIR> struct Dft<4, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    float2 s0 = cadd(v[0], v[2]), d0 = csub(v[0], v[2]);
    float2 s1 = cadd(v[1], v[3]), d1 = rot<DIR>(csub(v[1], v[3]));
    v[0] = cadd(s0, s1);
    v[1] = cadd(d0, d1);
    v[2] = csub(s0, s1);
    v[3] = csub(d0, d1);
  }
};

template <int DIR> struct Dft<5, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
    const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
    float2 x0 = v[0];
    float2 t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
    float2 t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
    float2 a1 = make_float2(x0.x + c1 * t1.x + c2 * t2.x, x0.y + c1 * t1.y + c2 * t2.y);
    float2 a2 = make_float2(x0.x + c2 * t1.x + c1 * t2.x, x0.y + c2 * t1.y + c1 * t2.y);
    float2 b1 = rot<DIR>(make_float2(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y));
    float2 b2 = rot<DIR>(make_float2(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y));
    v[0] = cadd(x0, cadd(t1, t2));
    v[1] = cadd(a1, b1);
    v[4] = csub(a1, b1);
    v[2] = cadd(a2, b2);
    v[3] = csub(a2, b2);
  }
};

// multiply by W8^1 = sqrt(1/2)(1 + DIR i)
template <int DIR> __device__ __forceinline__ float2 mul_w8_1(float2 a)
{
  const float h = 0.70710678118654752440f;
  if constexpr (DIR < 0) return make_float2((a.x + a.y) * h, (a.y - a.x) * h);
  else return make_float2((a.x - a.y) * h, (a.y + a.x) * h);
}
// multiply by W8^3 = sqrt(1/2)(-1 + DIR i)
template <int DIR> __device__ __forceinline__ float2 mul_w8_3(float2 a)
{
  const float h = 0.70710678118654752440f;
  if constexpr (DIR < 0) return make_float2((a.y - a.x) * h, -(a.x + a.y) * h);
  else return make_float2(-(a.x + a.y) * h, (a.x - a.y) * h);
}

template <int DIR> struct Dft<8, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    float2 u[4], w[4];
    u[0] = cadd(v[0], v[4]); w[0] = csub(v[0], v[4]);
    u[1] = cadd(v[1], v[5]); w[1] = mul_w8_1<DIR>(csub(v[1], v[5]));
    u[2] = cadd(v[2], v[6]); w[2] = rot<DIR>(csub(v[2], v[6]));
    u[3] = cadd(v[3], v[7]); w[3] = mul_w8_3<DIR>(csub(v[3], v[7]));
    Dft<4, DIR>::run(u);
    Dft<4, DIR>::run(w);
#pragma unroll
    for (int k = 0; k < 4; ++k) { v[2 * k] = u[k]; v[2 * k + 1] = w[k]; }
  }
};

// 16 = 4 x 4: y[k1 + 4 k2] = DFT4_n( W16^{n k1} * DFT4_{n2}(x[n + 4 n2])[k1] )[k2]
template <int DIR> struct Dft<16, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    const float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f;
    const float d = (float)DIR;
    float2 z[4][4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      float2 a[4] = { v[n], v[n + 4], v[n + 8], v[n + 12] };
      Dft<4, DIR>::run(a);
#pragma unroll
      for (int k = 0; k < 4; ++k) z[n][k] = a[k];
    }
    // twiddles W16^{n k1}, n,k1 in 1..3
    z[1][1] = cmul(z[1][1], make_float2(c1, d * s1));
    z[1][2] = mul_w8_1<DIR>(z[1][2]);
    z[1][3] = cmul(z[1][3], make_float2(s1, d * c1));
    z[2][1] = mul_w8_1<DIR>(z[2][1]);
    z[2][2] = rot<DIR>(z[2][2]);
    z[2][3] = mul_w8_3<DIR>(z[2][3]);
    z[3][1] = cmul(z[3][1], make_float2(s1, d * c1));
    z[3][2] = mul_w8_3<DIR>(z[3][2]);
    z[3][3] = cmul(z[3][3], make_float2(-c1, -d * s1));
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      float2 b[4] = { z[0][k1], z[1][k1], z[2][k1], z[3][k1] };
      Dft<4, DIR>::run(b);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = b[k2];
    }
  }
};

// 9 = 3 x 3: y[k1 + 3 k2] = DFT3_n( W9^{n k1} * DFT3_{n2}(x[n + 3 n2])[k1] )[k2]
template <int DIR> struct Dft<9, DIR> {
  __device__ __forceinline__ static void run(float2 *v)
  {
    const float d = (float)DIR;
    const float2 w1 = make_float2(0.76604444311897803520f, d * 0.64278760968653932632f);  // W9
    const float2 w2 = make_float2(0.17364817766693034885f, d * 0.98480775301220805937f);  // W9^2
    const float2 w4 = make_float2(-0.93969262078590838405f, d * 0.34202014332566873304f); // W9^4
    float2 z[3][3];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      float2 a[3] = { v[n], v[n + 3], v[n + 6] };
      Dft<3, DIR>::run(a);
#pragma unroll
      for (int k = 0; k < 3; ++k) z[n][k] = a[k];
    }
    z[1][1] = cmul(z[1][1], w1);
    z[1][2] = cmul(z[1][2], w2);
    z[2][1] = cmul(z[2][1], w2);
    z[2][2] = cmul(z[2][2], w4);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      float2 b[3] = { z[0][k1], z[1][k1], z[2][k1] };
      Dft<3, DIR>::run(b);
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = b[k2];
    }
  }
};

// R = A * B with A, B coprime (Good's prime-factor mapping, no twiddles):
// input n = (B n1 + A n2) mod R, output k with k = k1 mod A, k = k2 mod B.
// All indices are compile-time, so the maps cost nothing.
template <int A, int B, int DIR> struct DftCoprime {
  static constexpr int out(int k1, int k2)
  {
    for (int k = 0; k < A * B; ++k)
      if (k % A == k1 && k % B == k2) return k;
    return 0;
  }
  template <int K1, int... K2>
  __device__ __forceinline__ static void put(float2 *v, const float2 *b, std::integer_sequence<int, K2...>)
  {
    ((v[std::integral_constant<int, out(K1, K2)>::value] = b[K2]), ...);
  }
  template <int... K1>
  __device__ __forceinline__ static void second(float2 *v, const float2 (&z)[B][A], std::integer_sequence<int, K1...>)
  {
    (
        [&] {
          float2 b[B];
#pragma unroll
          for (int n2 = 0; n2 < B; ++n2) b[n2] = z[n2][K1];
          Dft<B, DIR>::run(b);
          put<K1>(v, b, std::make_integer_sequence<int, B>());
        }(),
        ...);
  }
  __device__ __forceinline__ static void run(float2 *v)
  {
    float2 z[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) z[n2][n1] = v[(B * n1 + A * n2) % (A * B)];
      Dft<A, DIR>::run(z[n2]);
    }
    second(v, z, std::make_integer_sequence<int, A>());
  }
};
template <int DIR> struct Dft<6, DIR> : DftCoprime<2, 3, DIR> {};
template <int DIR> struct Dft<10, DIR> : DftCoprime<2, 5, DIR> {};
template <int DIR> struct Dft<12, DIR> : DftCoprime<4, 3, DIR> {};
template <int DIR> struct Dft<18, DIR> : DftCoprime<2, 9, DIR> {};
template <int DIR> struct Dft<20, DIR> : DftCoprime<4, 5, DIR> {};
template <int DIR> struct Dft<24, DIR> : DftCoprime<8, 3, DIR> {};
template <int DIR> struct Dft<36, DIR> : DftCoprime<4, 9, DIR> {};
template <int DIR> struct Dft<40, DIR> : DftCoprime<8, 5, DIR> {};

// ---------------------------------------------------------------- buffer IO
// Raw buffer loads/stores: one 128-bit descriptor per base pointer, a
// per-lane 32-bit byte offset and an SGPR/immediate constant offset, so the
// unrolled accesses of a row need no 64-bit address arithmetic.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
static constexpr int kRsrcFlags = 0x00020000; // raw buffer, 32-bit data format

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, kRsrcFlags);
}
__device__ __forceinline__ float2 bload(rsrc_t r, uint32_t voff, uint32_t soff)
{
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
// non-temporal (streaming) variant for data read exactly once
__device__ __forceinline__ float2 bload_nt(rsrc_t r, uint32_t voff, uint32_t soff)
{
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 2));
}
__device__ __forceinline__ void bstore(rsrc_t r, float2 v, uint32_t voff, uint32_t soff)
{
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 0);
}
__device__ __forceinline__ void bstore_nt(rsrc_t r, float2 v, uint32_t voff, uint32_t soff)
{
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 2);
}
template <bool NT>
__device__ __forceinline__ float bload1(rsrc_t r, uint32_t voff, uint32_t soff)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, NT ? 2 : 0));
}
template <bool NT>
__device__ __forceinline__ void bstore1(rsrc_t r, float v, uint32_t voff, uint32_t soff)
{
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, NT ? 2 : 0);
}

// Access to one line of complex values, element e at a per-lane base plus a
// constant (or scalar) offset.  IoC: interleaved complex<float> (one 64-bit
// access per value).  IoS: split storage, real and imaginary parts in two
// float arrays with the same layout (two 32-bit accesses, each coalesced).
// NTL / NTS: non-temporal loads / stores.  The row transforms write each line
// once and store it non-temporally; their loads are ordinary: non-temporal
// ones took 19.5 instead of 15.1 us for a 1000 x 4096 fastconv, 36.8 instead of
// 33.9 at 1000 x 8192 and 5.7 instead of 5.2 at 256 x 2048 (the exception is
// hier_streams_in()).
template <bool NTL = false, bool NTS = true>
struct IoCx {
  rsrc_t r;
  uint32_t v; // lane base, bytes
  __device__ __forceinline__ float2 ld(uint32_t e) const
  {
    if constexpr (NTL) return bload_nt(r, v, e * 8u);
    else return bload(r, v, e * 8u);
  }
  __device__ __forceinline__ void st(float2 x, uint32_t e) const
  {
    if constexpr (NTS) bstore_nt(r, x, v, e * 8u);
    else bstore(r, x, v, e * 8u);
  }
};
using IoC = IoCx<>;
template <bool NTL = false, bool NTS = true>
struct IoSx {
  rsrc_t re, im;
  uint32_t v; // lane base, bytes
  __device__ __forceinline__ float2 ld(uint32_t e) const
  {
    return make_float2(bload1<NTL>(re, v, e * 4u), bload1<NTL>(im, v, e * 4u));
  }
  __device__ __forceinline__ void st(float2 x, uint32_t e) const
  {
    bstore1<NTS>(re, x.x, v, e * 4u);
    bstore1<NTS>(im, x.y, v, e * 4u);
  }
};
using IoS = IoSx<>;

} // namespace ovx
