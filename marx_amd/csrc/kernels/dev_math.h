// dev_math.h -- FP64 primitives of the per-photon kernels, for arguments of
// ordinary size.
//
// The kernels are bound by the vector ALUs' issue rate, and the compiler's
// division, square root and device-library sincos and log are general: they
// scale against over- and underflow, fix up infinities and reduce arguments
// of any size.  The ones here leave that out, and each says which arguments
// it takes; where the caller cannot promise them it uses the general form.
// They start from the hardware's approximations (v_rcp_f64, v_rsq_f64, good
// to 2^-23 or better) and refine them with fused multiply-adds, whose one
// rounding makes a residual exact; the polynomials are the Taylor series.
// Largest error over 2^20 arguments against 80-bit arithmetic, in units of
// the last place, beside the general form's: division and square root 0.50
// (0.50), 1 / sqrt 0.99 (1.48 as 1 / sqrt (x)), log 0.54 (0.63), sine and
// cosine of an angle 0.75 (0.77), the polar method's sqrt (-2 log (g) / g)
// 0.90 (1.18); of a turn, 1.4e-16 in all (6.9e-16 as sincos (2 pi u), whose
// argument is rounded).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mxg {

// a b + c for a constant c, kept in scalar registers: the compiler's v_fmac
// would first copy it to vector registers, an instruction for each term of
// a polynomial
__device__ __forceinline__ double fma_k (double a, double b, double c)
{
   double d;
   asm ("v_fma_f64 %0, %1, %2, %3" : "=v" (d) : "v" (a), "v" (b), "s" (c));
   return d;
}

// 1 / b; b normal, of a size whose reciprocal is
__device__ __forceinline__ double rcp_n (double b)
{
   const double r = __builtin_amdgcn_rcp (b);
   const double e = fma (-b, r, 1.0);
   return fma (r, fma (e, e, e), r);
}

// a / b given r = rcp_n (b)
__device__ __forceinline__ double div_r (double a, double b, double r)
{
   const double q = a * r;
   return fma (fma (-b, q, a), r, q);
}

// a / b; b and the quotient normal (or a zero)
__device__ __forceinline__ double div_n (double a, double b)
{
   return div_r (a, b, rcp_n (b));
}

// a / b as div_n, and as the general form where a or b is 0, infinite or NaN
__device__ __forceinline__ double div_x (double a, double b)
{
   return __builtin_amdgcn_div_fixup (div_n (a, b), b, a);
}

// 1 / sqrt (x); x > 0 and normal
__device__ __forceinline__ double rsqrt_n (double x)
{
   const double y = __builtin_amdgcn_rsq (x);
   const double e = fma (-(x * y), y, 1.0);
   return fma (y * e, fma (0.375, e, 0.5), y);
}

// sqrt (x) and 1 / sqrt (x); x > 0 and normal
__device__ __forceinline__ double sqrt_rsqrt_n (double x, double &inv)
{
   const double y = rsqrt_n (x);
   const double g = x * y;
   inv = y;
   return fma (fma (-g, g, x), 0.5 * y, g);
}

// sqrt (x); x > 0 and normal, or 0
__device__ __forceinline__ double sqrt_n (double x)
{
   const double y = __builtin_amdgcn_rsq (x);
   double g = x * y, h = 0.5 * y;
   const double r = fma (-h, g, 0.5);
   g = fma (g, r, g);
   h = fma (h, r, h);
   g = fma (fma (-g, g, x), h, g);
   return (x == 0.0) ? 0.0 : g;
}

// sin and cos of x + tail, |x| <= pi / 4 (a little more does no harm), tail
// below an ulp of x: the Taylor series through x^17 and x^16 (truncation
// below 2e-18).  TAIL: what the squares round off is carried too.
template <bool TAIL>
__device__ __forceinline__ void sincos_poly (double x, double tail, double &s, double &c)
{
   const double z = x * x;
   double p = 1.0 / 355687428096000.0;
   p = fma_k (p, z, -1.0 / 1307674368000.0);
   p = fma_k (p, z, 1.0 / 6227020800.0);
   p = fma_k (p, z, -1.0 / 39916800.0);
   p = fma_k (p, z, 1.0 / 362880.0);
   p = fma_k (p, z, -1.0 / 5040.0);
   p = fma_k (p, z, 1.0 / 120.0);
   p = fma_k (p, z, -1.0 / 6.0);
   double q = 1.0 / 20922789888000.0;
   q = fma_k (q, z, -1.0 / 87178291200.0);
   q = fma_k (q, z, 1.0 / 479001600.0);
   q = fma_k (q, z, -1.0 / 3628800.0);
   q = fma_k (q, z, 1.0 / 40320.0);
   q = fma_k (q, z, -1.0 / 720.0);
   q = fma_k (q, z, 1.0 / 24.0);
   // 1 - z / 2 is rounded once, and what it lost goes back with the rest
   const double w = 0.5 * z, a = 1.0 - w;
   double lost = (1.0 - a) - w;
   if (TAIL)
     {
        s = x + fma (p, z * x, fma (-w, tail, tail));
        lost = fma (-x, tail, fma (-0.5, fma (x, x, -z), lost));
     }
   else
     s = x + p * z * x;
   c = a + fma (z * z, q, lost);
}

// (s, c) turned by k quarter turns
__device__ __forceinline__ void quarter_turns (int k, double s, double c, double &so, double &co)
{
   const bool odd = k & 1;
   const double a = odd ? c : s, b = odd ? s : c;
   so = (k & 2) ? -a : a;
   co = ((k + 1) & 2) ? -b : b;
}

// k mod 2^32 of a whole number |k| < 2^51 (a conversion to int ends at 2^31)
__device__ __forceinline__ int low_bits (double k)
{
   return __double2loint (k + 6755399441055744.0);      // 1.5 x 2^52
}

// sin and cos of 2 pi u, |u| < 2^20: the quarter turns are taken off
// exactly, before the product with 2 pi
__device__ __forceinline__ void sincos_turn (double u, double &s, double &c)
{
   const double k = rint (4.0 * u);
   double sx, cx;
   sincos_poly<false> (6.283185307179586477 * fma (-0.25, k, u), 0.0, sx, cx);
   quarter_turns ((int) k, sx, cx, s, c);
}

// sin and cos of x, |x| < 2^20 (to 2^50 with an absolute error below 2e-16):
// k quarter turns are taken off in two parts of pi / 2 (53 bits each: the
// first product and difference are exact in the fma), and what the second
// subtraction rounds off goes on as the tail
__device__ __forceinline__ void sincos_r (double x, double &s, double &c)
{
   const double k = rint (x * 0.63661977236758134308);
   const double r1 = fma (-k, 1.5707963267948965580, x);
   const double r = fma (-k, 6.1232339957367660e-17, r1);
   double sx, cx;
   sincos_poly<true> (r, fma (-k, 6.1232339957367660e-17, r1 - r), sx, cx);
   quarter_turns (low_bits (k), sx, cx, s, c);
}

// sin of x, |x| < 2^20
__device__ __forceinline__ double sin_r (double x)
{
   double s, c;
   sincos_r (x, s, c);
   return s;
}

// sin of any x
__device__ __forceinline__ double sin_any (double x)
{
   return (fabs (x) < 1048576.0) ? sin_r (x) : sin (x);
}

// log (x), x > 0 and normal: x = 2^e (1 + f), sqrt (1/2) <= 1 + f <
// sqrt (2), log (1 + f) = 2 atanh (f / (2 + f)) by its series (through
// the 21st power: truncation below 1e-18 of it).  The quotient and the sum
// with e log (2) keep what they round off.
__device__ __forceinline__ double log_n (double x)
{
   double m = __builtin_amdgcn_frexp_mant (x);
   int e = __builtin_amdgcn_frexp_exp (x);
   if (m < 0.70710678118654752440)
     {
        m = m + m;
        e--;
     }
   const double f = m - 1.0, t = 2.0 + f, r = rcp_n (t);
   const double s = div_r (f, t, r);
   const double z = s * s;
   double p = 2.0 / 21.0;
   p = fma_k (p, z, 2.0 / 19.0);
   p = fma_k (p, z, 2.0 / 17.0);
   p = fma_k (p, z, 2.0 / 15.0);
   p = fma_k (p, z, 2.0 / 13.0);
   p = fma_k (p, z, 2.0 / 11.0);
   p = fma_k (p, z, 2.0 / 9.0);
   p = fma_k (p, z, 2.0 / 7.0);
   p = fma_k (p, z, 2.0 / 5.0);
   p = fma_k (p, z, 2.0 / 3.0);
   // f - s (2 + f), with the rounding f - (t - 2) of t
   const double rest = fma (-s, f - (t - 2.0), fma (-s, t, f)) * r;
   const double k = (double) e, s2 = s + s;
   const double h = fma (k, 0.69314718055994528623, s2);
   const double l = fma (k, 0.69314718055994528623, -h) + s2;
   return h + (l + fma (k, 2.3190468138462995584e-17, fma (p, z * s, rest + rest)));
}

// a ^ b ^ c, one instruction on gfx950
__device__ __forceinline__ uint32_t xor3 (uint32_t a, uint32_t b, uint32_t c)
{
   return __builtin_amdgcn_bitop3_b32 (a, b, c, 0x96);
}

// ---- vectors, with fused multiply-adds ------------------------------------------

struct vec3 { double x, y, z; };

__device__ __forceinline__ double dot_f (vec3 a, vec3 b)
{
   return fma (a.z, b.z, fma (a.y, b.y, a.x * b.x));
}

__device__ __forceinline__ vec3 cross_f (vec3 a, vec3 b)
{
   vec3 c;
   c.x = fma (a.y, b.z, -(a.z * b.y));
   c.y = fma (a.z, b.x, -(a.x * b.z));
   c.z = fma (a.x, b.y, -(a.y * b.x));
   return c;
}

// x + t p
__device__ __forceinline__ vec3 along_f (vec3 x, double t, vec3 p)
{
   vec3 r;
   r.x = fma (t, p.x, x.x);
   r.y = fma (t, p.y, x.y);
   r.z = fma (t, p.z, x.z);
   return r;
}

// a x + b y
__device__ __forceinline__ vec3 lin2_f (double a, vec3 x, double b, vec3 y)
{
   vec3 r;
   r.x = fma (a, x.x, b * y.x);
   r.y = fma (a, x.y, b * y.y);
   r.z = fma (a, x.z, b * y.z);
   return r;
}

__device__ __forceinline__ vec3 scale_f (double a, vec3 x)
{
   vec3 r;
   r.x = a * x.x; r.y = a * x.y; r.z = a * x.z;
   return r;
}

// a / |a|; a not 0
__device__ __forceinline__ vec3 unit_f (vec3 a)
{
   return scale_f (rsqrt_n (dot_f (a, a)), a);
}

// a / |a| of a vector that a rotation keeps of length 1 to rounding: the
// first term of the series of 1 / sqrt about 1 is all that shows
__device__ __forceinline__ vec3 reunit_f (vec3 a)
{
   return scale_f (fma (-0.5, dot_f (a, a), 1.5), a);
}

// p turned about the unit axis n by the angle of cosine c and sine s
__device__ __forceinline__ vec3 turn_f (vec3 p, vec3 n, double c, double s)
{
   const double t = dot_f (p, n) * (1.0 - c);
   const vec3 q = cross_f (n, p);
   vec3 u;
   u.x = fma (c, p.x, fma (t, n.x, s * q.x));
   u.y = fma (c, p.y, fma (t, n.y, s * q.y));
   u.z = fma (c, p.z, fma (t, n.z, s * q.z));
   return u;
}

// ... about the x axis
__device__ __forceinline__ vec3 turn_x_f (vec3 p, double c, double s)
{
   vec3 u;
   u.x = p.x;
   u.y = fma (c, p.y, -(s * p.z));
   u.z = fma (s, p.y, c * p.z);
   return u;
}

__device__ __forceinline__ vec3 mul_m3_f (const double *m, vec3 v)
{
   vec3 r;
   r.x = fma (m[2], v.z, fma (m[1], v.y, m[0] * v.x));
   r.y = fma (m[5], v.z, fma (m[4], v.y, m[3] * v.x));
   r.z = fma (m[8], v.z, fma (m[7], v.y, m[6] * v.x));
   return r;
}

} // namespace mxg
