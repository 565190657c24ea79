// diff.hip -- the differentiable mirror: a weighted-photon HRMA trace with
// forward-mode derivatives, its focal-plane image, and the adjoint that turns
// d(loss)/d(image) into d(loss)/d(misalignment parameters).
//
// Per photon, the same steps as hrma.hip (marx/libsrc/hrma.c:984-1050,
// 411-545, 900-981; reflect.c:39-77; wfold.c:334-369) with two changes:
//  - survival weights replace the vignetting and reflectivity draws: the
//    weight is the product of the vignetting factor and, per surface, the
//    Fresnel reflectivity times the scale factor; a photon that misses a
//    surface, is shadowed by a strut or scatters past pi/4 gets weight 0;
//  - every quantity that depends on the photon's shell-pair parameters
//    (tilt az, tilt el, decenter y, decenter z, despace x) carries their
//    five derivatives (a dual number).  Draws are consumed in the same
//    order as the oracle's weighted trace; each photon's draws do not depend
//    on the parameters.
// At the focal plane (x = 0) the weight is spread bilinearly over the four
// pixels around the photon.  Weights, positions and their derivatives stay
// in HBM for the adjoint, which contracts them with d(loss)/d(image).
#include "dev_common.h"
#include "dev_store.h"

namespace mxg {

constexpr int kNP = MXG_DIFF_NPAR;

// ---- dual numbers: a value and its derivatives by N parameters ---------------------
//
// N = kNP carries all five parameters of the photon's shell pair.  N = 2
// carries the two tilts only: for a source at infinity a translation of the
// shell pair moves the photon's aperture position with it (the annulus is
// sampled about the displaced shell), so in the frame of each surface the
// path does not depend on the translations, whose derivatives are then
// fixed at the focal plane (kernel below).  N = 0 is the value-only pass.

template <int N>
struct Dual
{
   double v;
   double d[N > 0 ? N : 1];
};

template <int N> __device__ __forceinline__ Dual<N> dc (double v)
{
   Dual<N> r;
   r.v = v;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = 0.0;
   return r;
}

template <int N> __device__ __forceinline__ Dual<N> operator+ (Dual<N> a, Dual<N> b)
{
   Dual<N> r; r.v = a.v + b.v;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = a.d[j] + b.d[j];
   return r;
}
template <int N> __device__ __forceinline__ Dual<N> operator- (Dual<N> a, Dual<N> b)
{
   Dual<N> r; r.v = a.v - b.v;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = a.d[j] - b.d[j];
   return r;
}
template <int N> __device__ __forceinline__ Dual<N> operator- (Dual<N> a)
{
   Dual<N> r; r.v = -a.v;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = -a.d[j];
   return r;
}
template <int N> __device__ __forceinline__ Dual<N> operator* (Dual<N> a, Dual<N> b)
{
   Dual<N> r; r.v = a.v * b.v;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = fma (a.d[j], b.v, a.v * b.d[j]);
   return r;
}
template <int N> __device__ __forceinline__ Dual<N> operator* (double a, Dual<N> b)
{
   Dual<N> r; r.v = a * b.v;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = a * b.d[j];
   return r;
}
template <int N> __device__ __forceinline__ Dual<N> operator* (Dual<N> b, double a) { return a * b; }
template <int N> __device__ __forceinline__ Dual<N> operator/ (Dual<N> a, Dual<N> b)
{
   const double ib = rcp_n (b.v);
   Dual<N> r; r.v = div_r (a.v, b.v, ib);
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = fma (-r.v, b.d[j], a.d[j]) * ib;
   return r;
}
// a b + c
template <int N> __device__ __forceinline__ Dual<N> dfma (Dual<N> a, Dual<N> b, Dual<N> c)
{
   Dual<N> r; r.v = fma (a.v, b.v, c.v);
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = fma (a.d[j], b.v, fma (a.v, b.d[j], c.d[j]));
   return r;
}
template <int N> __device__ __forceinline__ Dual<N> dfma (double a, Dual<N> b, Dual<N> c)
{
   Dual<N> r; r.v = fma (a, b.v, c.v);
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = fma (a, b.d[j], c.d[j]);
   return r;
}

template <int N> __device__ __forceinline__ Dual<N> dsqrt (Dual<N> a)
{
   Dual<N> r; r.v = sqrt_n (a.v);
   const double f = (N > 0 && r.v > 0.0) ? 0.5 * rcp_n (r.v) : 0.0;
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = a.d[j] * f;
   return r;
}
// 1 / sqrt (a), a > 0
template <int N> __device__ __forceinline__ Dual<N> drsqrt (Dual<N> a)
{
   Dual<N> r; r.v = rsqrt_n (a.v);
   const double f = -0.5 * r.v * (r.v * r.v);
#pragma unroll
   for (int j = 0; j < N; j++) r.d[j] = a.d[j] * f;
   return r;
}
template <int N> __device__ __forceinline__ void dsincos (Dual<N> a, Dual<N> &s, Dual<N> &c)
{
   double sv, cv;
   sincos_small (a.v, &sv, &cv);
   s.v = sv; c.v = cv;
#pragma unroll
   for (int j = 0; j < N; j++) { s.d[j] = cv * a.d[j]; c.d[j] = -sv * a.d[j]; }
}

template <int N> struct DVec { Dual<N> x, y, z; };

template <int N> __device__ __forceinline__ DVec<N> dv (vec3 a)
{
   DVec<N> r; r.x = dc<N> (a.x); r.y = dc<N> (a.y); r.z = dc<N> (a.z); return r;
}
template <int N> __device__ __forceinline__ vec3 val (const DVec<N> &a) { return v3 (a.x.v, a.y.v, a.z.v); }
template <int N> __device__ __forceinline__ DVec<N> dadd (const DVec<N> &a, const DVec<N> &b)
{
   DVec<N> r; r.x = a.x + b.x; r.y = a.y + b.y; r.z = a.z + b.z; return r;
}
template <int N> __device__ __forceinline__ DVec<N> dsub (const DVec<N> &a, const DVec<N> &b)
{
   DVec<N> r; r.x = a.x - b.x; r.y = a.y - b.y; r.z = a.z - b.z; return r;
}
template <int N> __device__ __forceinline__ Dual<N> ddot (const DVec<N> &a, const DVec<N> &b)
{
   return dfma (a.z, b.z, dfma (a.y, b.y, a.x * b.x));
}
template <int N> __device__ __forceinline__ DVec<N> dcross (const DVec<N> &a, const DVec<N> &b)
{
   DVec<N> c;
   c.x = dfma (a.y, b.z, -(a.z * b.y));
   c.y = dfma (a.z, b.x, -(a.x * b.z));
   c.z = dfma (a.x, b.y, -(a.y * b.x));
   return c;
}
template <int N> __device__ __forceinline__ DVec<N> dscale (Dual<N> a, const DVec<N> &x)
{
   DVec<N> r;
   r.x = a * x.x; r.y = a * x.y; r.z = a * x.z;
   return r;
}
// a x + b y
template <int N>
__device__ __forceinline__ DVec<N> dlin2 (Dual<N> a, const DVec<N> &x, Dual<N> b, const DVec<N> &y)
{
   DVec<N> r;
   r.x = dfma (a, x.x, b * y.x);
   r.y = dfma (a, x.y, b * y.y);
   r.z = dfma (a, x.z, b * y.z);
   return r;
}

// a / |a|
template <int N> __device__ __forceinline__ DVec<N> dunit (const DVec<N> &a)
{
   return dscale (drsqrt (ddot (a, a)), a);
}

// ... of a vector that a rotation keeps of length 1 to rounding (reunit_f)
template <int N> __device__ __forceinline__ DVec<N> dreunit (const DVec<N> &a)
{
   return dscale (dfma (-0.5, ddot (a, a), dc<N> (1.5)), a);
}

// M x for a tilt matrix M(az, el): value m, derivatives dm[0] (az, tangent
// 0), dm[1] (el, tangent 1)
template <int N>
__device__ __forceinline__ Dual<N> dm3_row (const double *m, const double (*dm)[9], int row, const DVec<N> &x)
{
   const double *a = m + 3 * row;
   Dual<N> o = dfma (a[2], x.z, dfma (a[1], x.y, a[0] * x.x));
   if constexpr (N >= 2)
     for (int j = 0; j < 2; j++)
       {
          const double *b = dm[j] + 3 * row;
          o.d[j] = fma (b[2], x.z.v, fma (b[1], x.y.v, fma (b[0], x.x.v, o.d[j])));
       }
   return o;
}

template <int N>
__device__ __forceinline__ DVec<N> dm3_vmul (const double *m, const double (*dm)[9], const DVec<N> &x)
{
   DVec<N> r;
   r.x = dm3_row (m, dm, 0, x);
   r.y = dm3_row (m, dm, 1, x);
   r.z = dm3_row (m, dm, 2, x);
   return r;
}

// to_osac of surface k as a dual: d/d(decenter y, z, despace x) = -1 (only
// carried when the translations are)
template <int N> __device__ __forceinline__ DVec<N> dto_osac (const mxg_diff_shell &D, int k)
{
   DVec<N> t = dv<N> (ld3 (D.to_osac[k]));
   if constexpr (N == kNP)
     {
        t.y.d[2] = -1.0;
        t.z.d[3] = -1.0;
        t.x.d[4] = -1.0;
     }
   return t;
}

// ---- the reflectivity and its derivative by cos(theta) ---------------------------
//
// With m = n^2 - 1 and w = sqrt (m + c^2), the amplitudes are E = (c - w) /
// (c + w) across and (n^2 c - w) / (n^2 c + w) along the plane of incidence,
// w' = c / w, and from w^2 - c^2 = m
//   d|E|^2 / dc = -4 |m|^2 Re (w) / (|c + w|^4 |w|^2)
//   d|E|^2 / dc = 4 |m|^2 Re (n^2 conj ((c^2 (2 + m) - 1) w)) / (|n^2 c + w|^4 |w|^2).
// The reflectivity (reflect.c:39-77) is the mean of the two |E|^2.

struct MirrorOptics
{
   double mr, mi;                // m = n^2 - 1, n = 1 - delta + i beta
};

__device__ __forceinline__ MirrorOptics mirror_optics (double beta, double delta)
{
   MirrorOptics o;
   o.mr = fma (delta, delta - 2.0, -(beta * beta));
   o.mi = 2.0 * (1.0 - delta) * beta;
   return o;
}

// the reflectivity at cos (theta) = c; SLOPE: its derivative in dr
template <bool SLOPE>
__device__ __forceinline__ double reflectivity_at (double c, const MirrorOptics &o, double &dr)
{
   const double c2 = c * c, wr2 = fma (c, c, o.mr), wi2 = o.mi;
   // the principal square root of wr2 + i wi2 by the half-angle formulas
   double inv;
   const double mod = sqrt_n (fma (wr2, wr2, wi2 * wi2));
   const double big = sqrt_rsqrt_n (fmax (0.5 * (mod + fabs (wr2)), 1e-300), inv);
   const double small = 0.5 * wi2 * inv;
   const double wr = (wr2 >= 0.0) ? big : fabs (small);
   const double wi = (wr2 >= 0.0) ? small : copysign (big, small);
   const double i2 = wi * wi, nr = 1.0 + o.mr;
   const double d1 = c - wr, s1 = c + wr;
   const double A = fma (d1, d1, i2), B = fma (s1, s1, i2);
   const double xr = nr * c, xi = o.mi * c;
   const double e1 = xr - wr, e2 = xi - wi, f1 = xr + wr, f2 = xi + wi;
   const double C = fma (e1, e1, e2 * e2), D = fma (f1, f1, f2 * f2);
   const double ibd = rcp_n (B * D);
   const double ib = ibd * D, id = ibd * B;       // 1 / B, 1 / D
   if (SLOPE)
     {
        const double m2 = fma (o.mr, o.mr, o.mi * o.mi);
        // u = (c^2 (2 + m) - 1) w, then Re (n^2 conj (u))
        const double tr = fma (c2, 2.0 + o.mr, -1.0), ti = c2 * o.mi;
        const double ur = fma (tr, wr, -(ti * wi)), ui = fma (tr, wi, ti * wr);
        const double par = fma (nr, ur, o.mi * ui);
        dr = 2.0 * m2 * rcp_n (fmax (mod, 1e-300)) * fma (par * id, id, -(wr * ib) * ib);
     }
   return 0.5 * fma (A, ib, C * id);
}

// WFold angle at (energy, sin_alpha, r) and its derivative by sin_alpha
// (linear in e_alpha = energy sin_alpha between the bracketing tables)
__device__ __forceinline__ double wfold_d1 (const mxg_wfold &w, const float *__restrict__ fa,
                                            const double *__restrict__ da, double energy,
                                            double sin_alpha, double r, double &dval)
{
   dval = 0.0;
   if (w.n_arrays == 0) return 0.0;
   const FoldRecord *arrays = (const FoldRecord *) (da + w.arrays_off);
   if (w.n_arrays == 1) return fold_theta (arrays[0], fa, r);
   const double *e_alphas = da + w.e_alphas_off;
   double e_alpha = energy * sin_alpha;
   unsigned int i = search_w (e_alpha, e_alphas, w.n_arrays);
   if (i == w.n_arrays) i--;
   if (i == 0) i++;
   const FoldRecord f0 = arrays[i - 1], f1 = arrays[i];
   const double theta_0 = fold_theta (f0, fa, r);
   const double theta_1 = fold_theta (f1, fa, r);
   double e0 = e_alphas[i - 1], e1 = e_alphas[i];
   const double slope = div_n (theta_1 - theta_0, e1 - e0);
   dval = slope * energy;
   return fma (slope, e_alpha - e0, theta_0);
}

// ---- one photon -----------------------------------------------------------------------

// conic_hit (hrma_stage.h) on duals
template <int N>
__device__ __forceinline__ bool dconic_hit (double a, double b, double c, DVec<N> &x0, const DVec<N> &p,
                                            double xmin, double xmax)
{
   const Dual<N> t0 = -x0.x / p.x;
   const Dual<N> x_y = dfma (t0, p.y, x0.y);
   const Dual<N> x_z = dfma (t0, p.z, x0.z);
   const Dual<N> alpha = dfma (a * p.x, p.x, dc<N> (-1.0));
   const Dual<N> beta = dfma (b, p.x, -2.0 * dfma (p.y, x_y, p.z * x_z));
   const Dual<N> gamma = dfma (-x_y, x_y, dfma (-x_z, x_z, dc<N> (c)));
   Dual<N> t_plus, t_minus;
   bool minus_ok = false;
   if (alpha.v == 0.0)
     {
        if (beta.v == 0.0) return false;
        t_plus = t_minus = -gamma / beta;
     }
   else
     {
        const Dual<N> disc = dfma (beta, beta, -4.0 * (alpha * gamma));
        if (!(disc.v >= 0.0)) return false;
        const Dual<N> root = dsqrt (disc);
        const Dual<N> q = (beta.v < 0.0) ? beta - root : beta + root;
        t_plus = -2.0 * (gamma / q);
        t_minus = t_plus;
        if (fabs (p.x.v * q.v) <= 2.0001 * fmax (fabs (xmin), fabs (xmax)) * fabs (alpha.v))
          {
             t_minus = -0.5 * (q / alpha);
             const double x_minus = p.x.v * t_minus.v;
             minus_ok = (x_minus >= xmin) && (x_minus < xmax);
          }
     }
   const double x_plus = p.x.v * t_plus.v;
   const bool plus_ok = (x_plus >= xmin) && (x_plus < xmax);
   if (!(plus_ok || minus_ok)) return false;
   const bool minus = minus_ok && !(plus_ok && (x_plus >= p.x.v * t_minus.v));
   const Dual<N> t = minus ? t_minus : t_plus;
   x0.x = p.x * t;
   x0.y = dfma (p.y, t, x_y);
   x0.z = dfma (p.z, t, x_z);
   return true;
}

// reflection at x on conic k: normal blur, survival weight, specular
// reflection, WFold scatter (the rotations as in hrma_stage.h: about axes
// at right angles).  false: scattered past pi/4.
template <int N>
__device__ __forceinline__ bool dreflect_at (const mxg_hrma_cfg &h, const mxg_shell_cfg &S, int k,
                                             const DVec<N> &x, DVec<N> &p, Dual<N> &w, double energy,
                                             const MirrorOptics &optics, double corr,
                                             const float *__restrict__ fa,
                                             const double *__restrict__ da, Stream &st)
{
   DVec<N> n;
   n.x = dfma (S.conic_a[k] - 1.0, x.x, dc<N> (0.5 * S.conic_b[k]));
   n.y = -x.y;
   n.z = -x.z;
   n = dunit (n);
   if (h.use_blur)
     {
        double sn, cs;
        const Dual<N> n2 = dfma (n.y, n.y, n.z * n.z);
        const Dual<N> il = drsqrt (n2);
        sincos_turn (uniform (st), sn, cs);
        const Dual<N> cl = cs * il, sl = sn * il, sx = sl * n.x;
        DVec<N> u;
        u.x = -(sl * n2);
        u.y = dfma (sx, n.y, cl * n.z);
        u.z = dfma (sx, n.z, -(cl * n.y));
        double phi = S.blur[k] * (1.0 / 3600.0 * MXG_PI / 180.0);
        phi = phi * gaussian (st);
        sincos_small (phi, &sn, &cs);
        n = dreunit (dlin2 (dc<N> (cs), n, dc<N> (sn), dcross (u, n)));
     }
   const Dual<N> p_dot_n = ddot (p, n);
   if (h.ideal == 0)
     {
        double dr = 0.0;
        Dual<N> R;
        R.v = reflectivity_at<(N > 0)> (fabs (p_dot_n.v), optics, dr);
        const double f = (p_dot_n.v < 0.0) ? -dr : dr;
#pragma unroll
        for (int j = 0; j < N; j++) R.d[j] = f * p_dot_n.d[j];
        w = w * (R * corr);
     }
   p = dlin2 (dc<N> (1.0), p, -2.0 * p_dot_n, n);
   if (h.use_wfold == 0)
     return true;
   double r = uniform (st);
   double slope;
   double g = wfold_d1 (S.wfold[k], fa, da, energy, -p_dot_n.v, r, slope);
   Dual<N> dg = (-slope) * p_dot_n;      // d/d(params) of the angle through sin_alpha = -p.n
   dg.v = g;
   dg = dg * S.scat_factor[k];
   if (dg.v > MXG_PI / 4) return false;
   if (uniform (st) < 0.5) dg = -dg;
   Dual<N> sn, cs;
   dsincos (dg, sn, cs);
   p = dunit (dlin2 (dfma (sn, p_dot_n, cs), p, sn, n));
   return true;
}

struct ImageSpec
{
   uint32_t npix;
   double pix, cy, cz;
};

constexpr int kWin = 64;         // central window of the image accumulated in LDS

__device__ __forceinline__ void pixel_coords (const ImageSpec &sp, double y, double z, int &i0, int &j0,
                                              double &fu, double &fv)
{
   double u = (y - sp.cy) / sp.pix + 0.5 * sp.npix - 0.5;
   double v = (z - sp.cz) / sp.pix + 0.5 * sp.npix - 0.5;
   double fu0 = floor (u), fv0 = floor (v);
   // clamp far-away photons to an index range that keeps the arithmetic in int
   fu0 = fmin (fmax (fu0, -2.0), (double) sp.npix + 1.0);
   fv0 = fmin (fmax (fv0, -2.0), (double) sp.npix + 1.0);
   i0 = (int) fu0;
   j0 = (int) fv0;
   fu = u - fu0;
   fv = v - fv0;
}

// A photon up to its paraboloid intersection: its draws (source stream:
// energy; mirror stream: shell, radius, azimuth), the aperture position in
// MARX coordinates, the precollimator struts, and the intersection in the
// paraboloid's frame.  false: the photon is lost before the first
// reflection.  k_diff_enter runs it on values, k_diff_forward again with
// tangents on the photons that pass; the values come out the same.
template <int N>
struct DiffPhoton
{
   double energy;
   int si;
   Stream st;
   DVec<N> x, p, t0, t1;
};

template <int N>
__device__ __forceinline__ bool diff_enter (const mxg_hrma_cfg &h, const mxg_source_cfg &src,
                                            const double *__restrict__ da,
                                            const mxg_diff_cfg *__restrict__ dcfg, uint32_t tag,
                                            unsigned long long seed, DiffPhoton<N> &ph)
{
   Stream ss;
   stream_init (ss, seed, tag, MXG_STAGE_SOURCE, 0u);
   ph.energy = draw_energy (src, da, ss);
   stream_init (ph.st, seed, tag, MXG_STAGE_MIRROR, 0u);
   int si;
   for (;;)
     {
        double r = uniform (ph.st);
        si = -1;
        for (int k = 0; k < MXG_NUM_SHELLS; k++)
          if (r < h.shell[k].area_fraction) { si = k; break; }
        if (si >= 0) break;
     }
   ph.si = si;
   const mxg_shell_cfg &S = h.shell[si];
   const mxg_diff_shell &D = dcfg->shell[si];
   double radius = S.min_radius + (S.max_radius - S.min_radius) * uniform (ph.st);
   double theta;
   unsigned int quad;
   do
     {
        theta = uniform (ph.st);
        quad = (unsigned int) (4.0 * theta);
     }
   while (0 == (S.shutter_bitmap & (1u << quad)));
   double sn, cs;
   sincos_turn (theta - 1.0 / 8.0, sn, cs);

   ph.t0 = dto_osac<N> (D, 0);
   ph.t1 = dto_osac<N> (D, 1);
   DVec<N> &x = ph.x, &p = ph.p;
   x.x = dc<N> (D.front_position);
   if constexpr (N == kNP) x.x.d[4] = 1.0;
   x.z = dc<N> (radius * cs) - ph.t0.z;
   x.y = dc<N> (radius * sn) - ph.t0.y;
   p = dv<N> (ld3 (src.p));
   if (src.distance > 0.0)
     {
        p = dunit (dlin2 (dc<N> (1.0), x, dc<N> (src.distance), p));
     }
   if (h.use_struts && in_strut_shadow (h, val (x), val (p), rcp_n (p.x.v), h.pre_struts))
     return false;
   x = dadd (x, ph.t0);
   x = dm3_vmul (D.fwd[0], D.dfwd[0], x);
   p = dm3_vmul (D.fwd[0], D.dfwd[0], p);
   return dconic_hit (S.conic_a[0], S.conic_b[0], S.conic_c[0], x, p, S.conic_xmin[0], S.conic_xmax[0]);
}

// Every photon to its paraboloid intersection, values only: its shell, and
// those that are not lost listed, in order, for k_diff_forward, whose rows
// are dense: row q of its columns is entry q of the list.  (About half of
// the photons are lost.  With the columns by photon this kernel also wrote
// the lost ones' zeros, and the adjoint read lines half of which it did not
// need: 0.150 and 0.220 ms for 1e7 photons, now 0.137 and 0.116.)
__global__ __launch_bounds__ (kBlock)
void k_diff_enter (const mxg_config *__restrict__ cfg, const double *__restrict__ da,
                   const mxg_diff_cfg *__restrict__ dcfg, uint32_t n, uint32_t tag_start,
                   unsigned long long seed, DiffOut out, ListIO io)
{
   __shared__ uint32_t wc[2 * (kBlock / 64)];
   const mxg_hrma_cfg &h = cfg->hrma;
   const mxg_source_cfg &src = cfg->src;
   const BlockRange range = block_range (n, blockIdx.x, gridDim.x);
   SegWriter sw (io, range, wc);
   for (uint32_t base = range.lo; base < range.hi; base += kBlock)
     {
        const uint32_t i = base + threadIdx.x;
        bool keep = false;
        if (i < range.hi)
          {
             DiffPhoton<0> ph;
             keep = diff_enter<0> (h, src, da, dcfg, tag_start + i, seed, ph);
             out.shell[i] = (uint8_t) ph.si;
          }
        sw.add (keep, i);
     }
   sw.finish (io);
}

// waves per SIMD the forward kernel's registers are bounded for; timed on
// MI355X over 1e7 photons, 1 to 4 waves: 2 with tangents, 3 value only
template <int N> constexpr int kDiffWaves = (N == 0) ? 3 : 2;

// The photons listed by k_diff_enter (idx[0 .. *n_list)), with N tangents
// each (see Dual): kNP, 2 (source at infinity: the translation derivatives
// follow at the focal plane), or 0 (value only).  From the paraboloid
// intersection on: both reflections, the cap and post struts, the focal
// plane, the state, and the splat into the image (central window in LDS,
// summed per block in win_partial; the rest by global atomics).
template <int N>
__global__ __launch_bounds__ (kBlock, kDiffWaves<N>)
void k_diff_forward (const mxg_config *__restrict__ cfg, const float *__restrict__ fa,
                     const double *__restrict__ da, const mxg_diff_cfg *__restrict__ dcfg,
                     const uint32_t *__restrict__ idx, const uint32_t *__restrict__ n_list, uint32_t n,
                     uint32_t tag_start, unsigned long long seed, ImageSpec sp,
                     float *__restrict__ image, float *__restrict__ win_partial, DiffOut out)
{
   __shared__ float win[kWin * kWin];
   __shared__ double wsum[kBlock / 64];
   const int W = (sp.npix < (uint32_t) kWin) ? (int) sp.npix : kWin;
   const int wo = ((int) sp.npix - W) / 2;
   for (int k = threadIdx.x; k < W * W; k += blockDim.x) win[k] = 0.0f;
   __syncthreads ();

   const mxg_hrma_cfg &h = cfg->hrma;
   const mxg_source_cfg &src = cfg->src;
   const BlockRange range = block_range (*n_list, blockIdx.x, gridDim.x);
   double my_w = 0.0;

   for (uint32_t q = range.lo + threadIdx.x; q < range.hi; q += blockDim.x)
     {
        const uint32_t i = idx[q];
        DiffPhoton<N> ph;
        bool alive = diff_enter<N> (h, src, da, dcfg, tag_start + i, seed, ph);
        const int si = ph.si;
        const mxg_shell_cfg &S = h.shell[si];
        const mxg_diff_shell &D = dcfg->shell[si];
        DVec<N> &x = ph.x, &p = ph.p;
        Dual<N> w = dc<N> ((h.ideal == 0) ? h.vignetting : 1.0);

        double beta = 0.0, delta = 1.0, corr = 1.0;
        if (alive && (h.opt_n != 0) && (h.ideal == 0))
          {
             float ef = (float) ph.energy;
             beta = interp_f (ef, fa + h.opt_e_off, fa + h.opt_beta_off, h.opt_n);
             delta = interp_f (ef, fa + h.opt_e_off, fa + h.opt_delta_off, h.opt_n);
             if (h.use_scale)
               corr = sqrt ((double) interp_f (ef, fa + S.corr_e_off, fa + S.corr_f_off, S.corr_n));
          }
        const MirrorOptics optics = mirror_optics (beta, delta);
        for (int k = 0; (k < 2) && alive; k++)
          {
             if (k == 1)
               {
                  x = dadd (x, ph.t1);
                  x = dm3_vmul (D.fwd[1], D.dfwd[1], x);
                  p = dm3_vmul (D.fwd[1], D.dfwd[1], p);
                  if (!dconic_hit (S.conic_a[1], S.conic_b[1], S.conic_c[1], x, p, S.conic_xmin[1], S.conic_xmax[1]))
                    {
                       alive = false;
                       break;
                    }
               }
             if (!dreflect_at (h, S, k, x, p, w, ph.energy, optics, corr, fa, da, ph.st))
               {
                  alive = false;
                  break;
               }
             p = dm3_vmul (D.bwd[k], D.dbwd[k], p);
             x = dm3_vmul (D.bwd[k], D.dbwd[k], x);
             x = dsub (x, (k == 0) ? ph.t0 : ph.t1);
             if (h.use_struts && in_strut_shadow (h, val (x), val (p), rcp_n (p.x.v), (k == 0) ? h.cap_struts : h.post_struts))
               alive = false;
          }

        // focal plane
        Dual<N> yf = dc<N> (0.0), zf = dc<N> (0.0);
        double ib = 0.0;
        if (alive)
          {
             Dual<N> t = -x.x / p.x;
             yf = x.y + t * p.y;
             zf = x.z + t * p.z;
             ib = 1.0 / p.x.v;
          }
        else
          w = dc<N> (0.0);

        put_once (&out.w[q], w.v);
        put_once (&out.y[q], yf.v);
        put_once (&out.z[q], zf.v);
        if constexpr (N == kNP)
          {
#pragma unroll
             for (int j = 0; j < kNP; j++)
               {
                  out.dw[(size_t) j * n + q] = w.d[j];
                  out.dy[(size_t) j * n + q] = yf.d[j];
                  out.dz[(size_t) j * n + q] = zf.d[j];
               }
          }
        else if constexpr (N == 2)
          {
             // tilts as traced; the translations (decenter y, decenter z,
             // despace x) move the exit point by themselves and leave the
             // direction and weight alone: d(y, z) = (1, 0), (0, 1),
             // -(p_y, p_z) / p_x, dw = 0.  Only what is not a constant is
             // stored (k_diff_adjoint<true>, mxgd_diff_state): 11 doubles a
             // photon, not 18.
#pragma unroll
             for (int j = 0; j < 2; j++)
               {
                  put_once (&out.dw[(size_t) j * n + q], w.d[j]);
                  put_once (&out.dy[(size_t) j * n + q], yf.d[j]);
                  put_once (&out.dz[(size_t) j * n + q], zf.d[j]);
               }
             put_once (&out.dy[(size_t) 4 * n + q], -ib * p.y.v);
             put_once (&out.dz[(size_t) 4 * n + q], -ib * p.z.v);
          }
        put_once (&out.row_shell[q], (uint8_t) si);

        if (w.v != 0.0)
          {
             my_w += w.v;
             int i0, j0;
             double fu, fv;
             pixel_coords (sp, yf.v, zf.v, i0, j0, fu, fv);
             const double b[4] = {(1 - fu) * (1 - fv), fu * (1 - fv), (1 - fu) * fv, fu * fv};
#pragma unroll
             for (int c = 0; c < 4; c++)
               {
                  const int iy = i0 + (c & 1), iz = j0 + (c >> 1);
                  if ((iy < 0) || (iz < 0) || (iy >= (int) sp.npix) || (iz >= (int) sp.npix)) continue;
                  const float add = (float) (w.v * b[c]);
                  const int wy = iy - wo, wz = iz - wo;
                  if ((wy >= 0) && (wz >= 0) && (wy < W) && (wz < W))
                    atomicAdd (&win[wz * W + wy], add);
                  else
                    atomicAdd (&image[(size_t) iz * sp.npix + iy], add);
               }
          }
     }

   // per-block summed weight and the window
   for (int off = 32; off > 0; off >>= 1) my_w += __shfl_xor (my_w, off);
   if (__lane_id () == 0) wsum[threadIdx.x >> 6] = my_w;
   __syncthreads ();
   if (threadIdx.x == 0)
     {
        double s = 0.0;
        for (int k = 0; k < kBlock / 64; k++) s += wsum[k];
        out.block_w[blockIdx.x] = s;
     }
   for (int k = threadIdx.x; k < W * W; k += blockDim.x)
     win_partial[(size_t) blockIdx.x * (kWin * kWin) + k] = win[k];
}

// image window = sum of the blocks' windows in a fixed order: slice q
// (blockIdx.y) sums blocks q, q + kSlices, ... per pixel into slice_sum; then
// k_diff_window_final adds the slices in order
constexpr int kSlices = 64;

__global__ __launch_bounds__ (kBlock)
void k_diff_window (const float *__restrict__ win_partial, uint32_t nblocks, ImageSpec sp,
                    float *__restrict__ slice_sum)
{
   const int W = (sp.npix < (uint32_t) kWin) ? (int) sp.npix : kWin;
   const int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= W * W) return;
   float s = 0.0f;
   for (uint32_t b = blockIdx.y; b < nblocks; b += kSlices) s += win_partial[(size_t) b * (kWin * kWin) + k];
   slice_sum[(size_t) blockIdx.y * (kWin * kWin) + k] = s;
}

__global__ __launch_bounds__ (kBlock)
void k_diff_window_final (const float *__restrict__ slice_sum, ImageSpec sp, float *__restrict__ image)
{
   const int W = (sp.npix < (uint32_t) kWin) ? (int) sp.npix : kWin;
   const int wo = ((int) sp.npix - W) / 2;
   const int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= W * W) return;
   float s = 0.0f;
   for (int q = 0; q < kSlices; q++) s += slice_sum[(size_t) q * (kWin * kWin) + k];
   const int wy = k % W, wz = k / W;
   image[(size_t) (wz + wo) * sp.npix + (wy + wo)] = s;
}

__global__ void k_zero_f (float *__restrict__ a, size_t n)
{
   size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
   const size_t stride = (size_t) gridDim.x * blockDim.x;
   for (; i < n; i += stride) a[i] = 0.0f;
}

// per-block partial gradients: 4 shell pairs x kNP parameters.  TILTS: the
// forward pass carried the tilts only, and the translations' constant
// derivatives are not in memory: bound by the columns it reads, 89 bytes a
// photon instead of 145 (1e7 photons, 4.77e6 rows: 0.297 -> 0.220 ms, and 0.116
// on dense rows).
template <bool TILTS>
__global__ __launch_bounds__ (kBlock)
void k_diff_adjoint (uint32_t n, const uint32_t *__restrict__ n_rows, DiffOut in, ImageSpec sp, const float *__restrict__ g,
                     double *__restrict__ partial)
{
   constexpr int kG = MXG_NUM_SHELLS * kNP;
   __shared__ double red[kBlock / 64][kG];
   double acc[kG];
#pragma unroll
   for (int q = 0; q < kG; q++) acc[q] = 0.0;
   const BlockRange range = block_range (*n_rows, blockIdx.x, gridDim.x);
   const double inv_pix = 1.0 / sp.pix;

   for (uint32_t i = range.lo + threadIdx.x; i < range.hi; i += blockDim.x)
     {
        // a photon of weight 0 (lost, or vignetted to nothing) adds nothing
        const double w = in.w[i];
        if (w == 0.0) continue;
        double dw[kNP], dy[kNP], dz[kNP];
#pragma unroll
        for (int j = 0; j < kNP; j++)
          {
             if (TILTS && (j > 1))
               {
                  dw[j] = 0.0;
                  dy[j] = (j == 2) ? 1.0 : (j == 3) ? 0.0 : in.dy[(size_t) j * n + i];
                  dz[j] = (j == 2) ? 0.0 : (j == 3) ? 1.0 : in.dz[(size_t) j * n + i];
                  continue;
               }
             dw[j] = in.dw[(size_t) j * n + i];
             dy[j] = in.dy[(size_t) j * n + i];
             dz[j] = in.dz[(size_t) j * n + i];
          }
        int i0, j0;
        double fu, fv;
        pixel_coords (sp, in.y[i], in.z[i], i0, j0, fu, fv);
        // bilinear weights and their derivatives by u and v
        const double b[4] = {(1 - fu) * (1 - fv), fu * (1 - fv), (1 - fu) * fv, fu * fv};
        const double bu[4] = {-(1 - fv), (1 - fv), -fv, fv};
        const double bv[4] = {-(1 - fu), -fu, (1 - fu), fu};
        double gsum = 0.0, gu = 0.0, gv = 0.0;
#pragma unroll
        for (int c = 0; c < 4; c++)
          {
             const int iy = i0 + (c & 1), iz = j0 + (c >> 1);
             if ((iy < 0) || (iz < 0) || (iy >= (int) sp.npix) || (iz >= (int) sp.npix)) continue;
             const double gc = (double) g[(size_t) iz * sp.npix + iy];
             gsum += gc * b[c];
             gu += gc * bu[c];
             gv += gc * bv[c];
          }
        const int s = in.row_shell[i];
#pragma unroll
        for (int j = 0; j < kNP; j++)
          {
             const double c = gsum * dw[j] + w * inv_pix * (gu * dy[j] + gv * dz[j]);
#pragma unroll
             for (int k = 0; k < MXG_NUM_SHELLS; k++)
               acc[k * kNP + j] += (s == k) ? c : 0.0;
          }
     }
   const int wave = threadIdx.x >> 6;
#pragma unroll
   for (int q = 0; q < kG; q++)
     {
        double v = acc[q];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor (v, off);
        if (__lane_id () == 0) red[wave][q] = v;
     }
   __syncthreads ();
   if (threadIdx.x < kG)
     {
        double s = 0.0;
        for (int k = 0; k < kBlock / 64; k++) s += red[k][threadIdx.x];
        partial[(size_t) blockIdx.x * kG + threadIdx.x] = s;
     }
}

// out[q] = sum over b of partial[b * width + q], one block per q, in a fixed
// order: thread t sums b = t, t + kBlock, ...; then a tree over the threads
__global__ __launch_bounds__ (kBlock)
void k_diff_sum (const double *__restrict__ partial, uint32_t nblocks, double *__restrict__ out,
                 uint32_t width)
{
   __shared__ double red[kBlock];
   const uint32_t q = blockIdx.x;
   double s = 0.0;
   for (uint32_t b = threadIdx.x; b < nblocks; b += kBlock) s += partial[(size_t) b * width + q];
   red[threadIdx.x] = s;
   __syncthreads ();
   for (int half = kBlock / 2; half > 0; half >>= 1)
     {
        if ((int) threadIdx.x < half) red[threadIdx.x] += red[threadIdx.x + half];
        __syncthreads ();
     }
   if (threadIdx.x == 0) out[q] = red[0];
}

hipError_t launch_diff_forward (const mxg_config *cfg, const float *fa, const double *da,
                                const mxg_diff_cfg *dcfg, uint32_t n, uint32_t tag_start,
                                unsigned long long seed, const mxg_image_spec *spec, float *image,
                                float *win_partial, float *slice_sum, DiffOut out, const ListIO &enter,
                                uint32_t grid, double *wsum_dev, int tangents, hipStream_t st,
                                hipEvent_t *ev)
{
   ImageSpec sp = {spec->npix, spec->pixel_size, spec->center_y, spec->center_z};
   const size_t npix2 = (size_t) spec->npix * spec->npix;
   hipLaunchKernelGGL (k_zero_f, dim3 (256), dim3 (kBlock), 0, st, image, npix2);
   if (ev) (void) hipEventRecord (ev[0], st);
   hipLaunchKernelGGL (k_diff_enter, dim3 (enter.grid), dim3 (kBlock), 0, st, cfg, da, dcfg, n, tag_start,
                       seed, out, enter);
   hipError_t e = launch_compact (enter, st);
   if (e != hipSuccess) return e;
   if (ev) (void) hipEventRecord (ev[1], st);
   if (ev) (void) hipEventRecord (ev[2], st);
   const uint32_t *idx = enter.idx_out, *n_list = enter.n_out;
   if (tangents == kNP)
     hipLaunchKernelGGL (k_diff_forward<kNP>, dim3 (grid), dim3 (kBlock), 0, st, cfg, fa, da, dcfg, idx,
                         n_list, n, tag_start, seed, sp, image, win_partial, out);
   else if (tangents == 2)
     hipLaunchKernelGGL (k_diff_forward<2>, dim3 (grid), dim3 (kBlock), 0, st, cfg, fa, da, dcfg, idx,
                         n_list, n, tag_start, seed, sp, image, win_partial, out);
   else
     hipLaunchKernelGGL (k_diff_forward<0>, dim3 (grid), dim3 (kBlock), 0, st, cfg, fa, da, dcfg, idx,
                         n_list, n, tag_start, seed, sp, image, win_partial, out);
   if (ev) (void) hipEventRecord (ev[3], st);
   const int W = (spec->npix < (uint32_t) kWin) ? (int) spec->npix : kWin;
   const uint32_t wblocks = (W * W + kBlock - 1) / kBlock;
   hipLaunchKernelGGL (k_diff_window, dim3 (wblocks, kSlices), dim3 (kBlock), 0, st, win_partial, grid, sp,
                       slice_sum);
   hipLaunchKernelGGL (k_diff_window_final, dim3 (wblocks), dim3 (kBlock), 0, st, slice_sum, sp, image);
   hipLaunchKernelGGL (k_diff_sum, dim3 (1), dim3 (kBlock), 0, st, out.block_w, grid, wsum_dev, 1u);
   return hipGetLastError ();
}

hipError_t launch_diff_adjoint (uint32_t n, const uint32_t *n_rows, DiffOut in, int tangents, const mxg_image_spec *spec, const float *g,
                                double *partial, uint32_t grid, double *grad_dev, hipStream_t st,
                                hipEvent_t *ev)
{
   ImageSpec sp = {spec->npix, spec->pixel_size, spec->center_y, spec->center_z};
   if (ev) (void) hipEventRecord (ev[0], st);
   void (*adjoint) (uint32_t, const uint32_t *, DiffOut, ImageSpec, const float *, double *)
     = (tangents == 2) ? k_diff_adjoint<true> : k_diff_adjoint<false>;
   hipLaunchKernelGGL (adjoint, dim3 (grid), dim3 (kBlock), 0, st, n, n_rows, in, sp, g, partial);
   if (ev) (void) hipEventRecord (ev[1], st);
   hipLaunchKernelGGL (k_diff_sum, dim3 (MXG_NUM_SHELLS * kNP), dim3 (kBlock), 0, st, partial, grid,
                       grad_dev, (uint32_t) (MXG_NUM_SHELLS * kNP));
   return hipGetLastError ();
}

} // namespace mxg
