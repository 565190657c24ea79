// hrma_stage.h -- the per-photon work of the HRMA stage (marx/libsrc/hrma.c),
// shared by the stage kernels (hrma.hip) and the chunk kernels
// (passes.hip).
//
// Per photon (the operations of marx/libsrc/hrma.c:1161-1341):
//   vignetting draw -> aperture sampling by cumulative shell area, radius and
//   shutter-checked azimuth (hrma.c:984-1050) -> paraboloid: conic
//   intersection (hrma.c:411-478), normal blur (:1054-1093), Fresnel
//   reflectivity draw (reflect.c:39-77), specular reflection, WFold scatter
//   (wfold.c:334-369) -> cap struts -> hyperboloid: the same -> post-collimator
//   struts.  Geometry is FP64.
//
// The mirror's work is split in two at the paraboloid hit (hrma_enter_core,
// hrma_reflect_core).  The stream position handed on is the number of words
// drawn; no Gaussian variate is pending there.  (A second split at the
// hyperboloid hit, each part on the photons still alive, measured 37 percent
// slower: the second kernel repeats the stream resumption, the table lookups
// and the LDS staging.)
#pragma once

#include <string.h>
#include "dev_common.h"
#include "dev_store.h"

namespace mxg {

// The hit of a ray on the quadric x^2+y^2+z^2 = a x^2 + b x + c between
// xmin <= x < xmax (the larger valid root in x); ipx = rcp_n (p.x).  On
// success x0 becomes the hit; on a miss x0 is unchanged and false is
// returned.  The second root, -q / (2 alpha) of alpha t^2 + beta t + gamma,
// is formed only where it can lie between the limits: alpha is of the order
// of the squared angle to the axis, so it hardly ever does.
__device__ __forceinline__ bool conic_hit (double a, double b, double c, vec3 &x0, vec3 p, double ipx,
                                           double xmin, double xmax)
{
   const double t0 = div_r (-x0.x, p.x, ipx);
   const double x_y = fma (t0, p.y, x0.y);
   const double x_z = fma (t0, p.z, x0.z);
   const double alpha = fma (a * p.x, p.x, -1.0);
   const double beta = fma (b, p.x, -2.0 * fma (p.y, x_y, p.z * x_z));
   const double gamma = fma (-x_y, x_y, fma (-x_z, x_z, c));
   double t_plus, t_minus;
   bool minus_ok = false;

   if (alpha == 0.0)
     {
        if (beta == 0.0) return false;
        t_plus = t_minus = -div_n (gamma, beta);
     }
   else
     {
        const double disc = fma (beta, beta, -4.0 * alpha * gamma);
        if (!(disc >= 0.0)) return false;
        const double q = beta + copysign (sqrt_n (disc), beta);
        t_plus = -2.0 * div_n (gamma, q);
        t_minus = t_plus;
        if (fabs (p.x * q) <= 2.0001 * fmax (fabs (xmin), fabs (xmax)) * fabs (alpha))
          {
             t_minus = -0.5 * div_n (q, alpha);
             const double x_minus = p.x * t_minus;
             minus_ok = (x_minus >= xmin) && (x_minus < xmax);
          }
     }

   const double x_plus = p.x * t_plus;
   const bool plus_ok = (x_plus >= xmin) && (x_plus < xmax);
   if (!(plus_ok || minus_ok)) return false;
   const double t = (minus_ok && !(plus_ok && (x_plus >= p.x * t_minus))) ? t_minus : t_plus;
   x0.x = p.x * t;
   x0.y = fma (p.y, t, x_y);
   x0.z = fma (p.z, t, x_z);
   return true;
}

// inward unit normal of the quadric at a point on it (hrma.c:470-476)
__device__ __forceinline__ vec3 conic_normal (double a, double b, vec3 x)
{
   return unit_f (v3 (fma (a - 1.0, x.x, 0.5 * b), -x.y, -x.z));
}

// The normal n turned by a Gaussian angle about a random direction u in the
// surface (hrma.c:1054-1093).  u is (0, n_z, -n_y) / |(n_y, n_z)| turned
// about n by a uniform azimuth; the two are at right angles, and u and n are,
// so the rotations have no component along their axes, and they keep the
// length 1 to rounding.
__device__ __forceinline__ void blur_normal (vec3 &n, double blur, RingStream &st)
{
   const double n2 = fma (n.y, n.y, n.z * n.z);
   const double il = rsqrt_n (n2);
   double s, c;
   need (st, 1);
   sincos_turn (take (st), s, c);
   const double cl = c * il, sl = s * il, sx = sl * n.x;
   const vec3 u = v3 (-(sl * n2), fma (sx, n.y, cl * n.z), fma (sx, n.z, -(cl * n.y)));
   double phi = blur * (1.0 / 3600.0 * MXG_PI / 180.0);
   phi = phi * gaussian (st);
   sincos_small (phi, &s, &c);
   n = reunit_f (lin2_f (c, n, s, cross_f (u, n)));
}

// The photon's index of refraction at the mirror, n = 1 - delta + i beta,
// as the Fresnel draw uses it: the real and imaginary part of n^2, and the
// real part less one (from delta and beta: no cancellation); corr: the
// square root of its shell's area correction.
struct MirrorIndex
{
   double n2r, n2i, n2r1, corr;
};

// The Fresnel draw u against reflectivity times corr (reflect.c:39-77):
// true when absorbed.  The reflectivity is the mean of A / B = |c - w|^2 /
// |c + w|^2 and C / D = |n^2 c - w|^2 / |n^2 c + w|^2 with c the cosine of
// the angle to the normal and w = sqrt (n^2 - 1 + c^2); the draw is compared
// without the divisions.
__device__ __forceinline__ bool fresnel_absorbs (double u, double c, const MirrorIndex &m)
{
   const double wr = fma (c, c, m.n2r1), wi = m.n2i;
   // the principal square root by the half-angle formulas
   double inv;
   const double mod = sqrt_n (fma (wr, wr, wi * wi));
   const double big = sqrt_rsqrt_n (fmax (0.5 * (mod + fabs (wr)), 1e-300), inv);
   const double small = 0.5 * wi * inv;
   const double re = (wr >= 0.0) ? big : fabs (small);
   const double im = (wr >= 0.0) ? small : copysign (big, small);
   const double i2 = im * im;
   const double d1 = c - re, s1 = c + re;
   const double A = fma (d1, d1, i2), B = fma (s1, s1, i2);
   const double xr = m.n2r * c, xi = m.n2i * c;
   const double dr = xr - re, di = xi - im, sr = xr + re, si = xi + im;
   const double C = fma (dr, dr, di * di), D = fma (sr, sr, si * si);
   return 2.0 * u * (B * D) >= fma (A, D, C * B) * m.corr;
}

// Reflection at a surface point x already on conic k of shell S: normal
// blur, Fresnel draw, specular reflection, WFold scatter (hrma.c:488-545).
// 0 reflected, -1 absorbed or scattered out.
__device__ __forceinline__ int reflect_at (const mxg_hrma_cfg &h, const mxg_shell_cfg &S, int k,
                                           vec3 x, vec3 &p, double energy, const MirrorIndex &m,
                                           const float *__restrict__ fa,
                                           const double *__restrict__ da,
                                           const float *__restrict__ e_alphas,
                                           const float *__restrict__ ea_cnt, RingStream &st)
{
   vec3 normal = conic_normal (S.conic_a[k], S.conic_b[k], x);
   if (h.use_blur)
     blur_normal (normal, S.blur[k], st);
   const double p_dot_n = dot_f (p, normal);
   if (h.ideal == 0)
     {
        need (st, 1);
        if (fresnel_absorbs (take (st), fabs (p_dot_n), m)) return -1;
     }
   p = along_f (p, -2.0 * p_dot_n, normal);
   if (h.use_wfold == 0)
     return 0;
   // a block for every lane with room: usually the scatter's two words here
   // and four more for the other surface
   top_up (st);
   need (st, 2);
   const double r = take (st);
   double dg = wfold_interp (S.wfold[k], fa, da, e_alphas, energy, -p_dot_n, r, &S.ea_bucket[k], ea_cnt);
   dg *= S.scat_factor[k];
   if (dg > MXG_PI / 4) return -1;
   if (take (st) < 0.5) dg = -dg;
   // p turned by dg about p x n, which is at right angles to p and not of
   // length 1: cos p + sin (p x n) x p, with (p x n) x p = n |p|^2 - p (p . n)
   // and p . n = -p_dot_n after the reflection (|p| is 1 unless a caller's
   // list holds other directions)
   double sn, cs;
   sincos_small (dg, &sn, &cs);
   p = unit_f (lin2_f (fma (sn, p_dot_n, cs), p, sn * dot_f (p, p), normal));
   return 0;
}

// Offsets (in floats) of the tables staged in LDS by k_hrma_reflect.
struct HrmaLds
{
   uint32_t opt;                  // energies, betas, deltas: 3 * opt_n
   uint32_t corr_e[MXG_NUM_SHELLS], corr_f[MXG_NUM_SHELLS];
   uint32_t ea[MXG_NUM_SHELLS][2];  // e_alpha of each WFold table (float32 on disk: exact)
   // the bucket counts of the searched tables (mxg_bucket)
   uint32_t bk_opt, bk_corr[MXG_NUM_SHELLS], bk_ea[MXG_NUM_SHELLS][2];
   uint32_t floats;               // staged floats after the configuration copy
   // bit k: some shell's tilt matrix of surface k is not the identity (with
   // the standard geometry file the paraboloids' all are, and the products
   // with them are left out)
   uint32_t tilted;
};

// HrmaLds::tilted of configuration h (host side)
inline uint32_t hrma_tilted (const mxg_hrma_cfg &h)
{
   uint32_t t = 0;
   for (int sh = 0; sh < MXG_NUM_SHELLS; sh++)
     for (int k = 0; k < 2; k++)
       for (int q = 0; q < 9; q++)
         {
            const double one = (q % 4 == 0) ? 1.0 : 0.0;
            if ((h.shell[sh].fwd[k][q] != one) || (h.shell[sh].bwd[k][q] != one)) t |= 1u << k;
         }
   return t;
}

// Dynamic LDS of the reflection: the configuration copy, a copy of the
// layout at kHrmaLayOff (the reflection reads a table's offset by the
// photon's shell from LDS, instead of holding every shell's offsets in
// scalar registers and selecting per lane), the tables from kHrmaTabOff.
constexpr size_t kHrmaLayOff = (sizeof (mxg_hrma_cfg) + 15) & ~(size_t) 15;
constexpr size_t kHrmaTabOff = (kHrmaLayOff + sizeof (HrmaLds) + 15) & ~(size_t) 15;

// The LDS layout of the reflection tables for configuration h, whose e_alpha
// values are in da (host side).  WFold tables on the same e_alpha values (the
// standard ones all are) share them, which lets a CU hold four blocks of the
// reflection with their streams instead of three.
inline HrmaLds hrma_lds_layout (const mxg_hrma_cfg &h, const double *da)
{
   HrmaLds lay;
   uint32_t f = 0;
   lay.opt = f; f += 3 * h.opt_n;
   lay.bk_opt = f; f += bucket_floats (h.opt_bucket);
   for (int sh = 0; sh < MXG_NUM_SHELLS; sh++)
     {
        const mxg_shell_cfg &S = h.shell[sh];
        lay.corr_e[sh] = f; f += S.corr_n;
        lay.corr_f[sh] = f; f += S.corr_n;
        lay.bk_corr[sh] = f; f += bucket_floats (S.corr_bucket);
        for (int k = 0; k < 2; k++)
          {
             int same = -1;
             for (int q = 0; (q < 2 * sh + k) && (same < 0); q++)
               {
                  const mxg_wfold &o = h.shell[q / 2].wfold[q % 2], &w = S.wfold[k];
                  if ((o.n_arrays == w.n_arrays)
                      && !memcmp (da + o.e_alphas_off, da + w.e_alphas_off, w.n_arrays * sizeof (double)))
                    same = q;
               }
             if (same >= 0)
               {
                  lay.ea[sh][k] = lay.ea[same / 2][same % 2];
                  lay.bk_ea[sh][k] = lay.bk_ea[same / 2][same % 2];
                  continue;
               }
             lay.ea[sh][k] = f;
             f += S.wfold[k].n_arrays;
             lay.bk_ea[sh][k] = f;
             f += bucket_floats (S.ea_bucket[k]);
          }
     }
   lay.floats = f;
   lay.tilted = hrma_tilted (h);
   return lay;
}

// The LDS image of the mirror configuration and the reflection tables (the
// binary-search targets of every photon), made by the host from the arenas
// fa, da: the configuration at 0, lay at kHrmaLayOff, the tables at
// kHrmaTabOff + the offsets of lay: hrma_image_bytes of it, a multiple of 16.
inline size_t hrma_image_bytes (const HrmaLds &lay)
{
   return (kHrmaTabOff + (size_t) lay.floats * sizeof (float) + 15) & ~(size_t) 15;
}

inline void hrma_image (const mxg_hrma_cfg &h, const float *fa, const double *da, const HrmaLds &lay,
                        unsigned char *img)
{
   memset (img, 0, hrma_image_bytes (lay));
   memcpy (img, &h, sizeof (h));
   memcpy (img + kHrmaLayOff, &lay, sizeof (lay));
   float *tab = (float *) (img + kHrmaTabOff);
   auto put = [&] (uint32_t at, uint32_t off, uint32_t n) { if (n) memcpy (tab + at, fa + off, n * sizeof (float)); };
   put (lay.opt, h.opt_e_off, h.opt_n);
   put (lay.opt + h.opt_n, h.opt_beta_off, h.opt_n);
   put (lay.opt + 2 * h.opt_n, h.opt_delta_off, h.opt_n);
   put (lay.bk_opt, h.opt_bucket.off, bucket_floats (h.opt_bucket));
   for (int sh = 0; sh < MXG_NUM_SHELLS; sh++)
     {
        const mxg_shell_cfg &S = h.shell[sh];
        put (lay.corr_e[sh], S.corr_e_off, S.corr_n);
        put (lay.corr_f[sh], S.corr_f_off, S.corr_n);
        put (lay.bk_corr[sh], S.corr_bucket.off, bucket_floats (S.corr_bucket));
        for (int k = 0; k < 2; k++)
          {
             for (uint32_t w = 0; w < S.wfold[k].n_arrays; w++)
               tab[lay.ea[sh][k] + w] = (float) da[S.wfold[k].e_alphas_off + w];
             put (lay.bk_ea[sh][k], S.ea_bucket[k].off, bucket_floats (S.ea_bucket[k]));
          }
     }
}

// The source-to-paraboloid part of the mirror for an unabsorbed photon with
// tag `tag` and direction p (tilted: HrmaLds): vignetting, aperture, precollimator struts,
// frame change and the paraboloid intersection.  False when vignetting
// blocks the photon (nothing else is drawn); else true, with its position
// x, direction p, shell si and the mirror's marks added to flags; hit: it
// hit the paraboloid; its random-stream position in rng (3 words, 4 with
// vignetting, unless a draw was repeated).
__device__ __forceinline__ bool hrma_enter_core (const mxg_hrma_cfg &h, uint32_t tilted, uint32_t tag,
                                                 double source_distance,
                                                 unsigned long long seed, uint32_t source_id, vec3 &x,
                                                 vec3 &p, int &si, uint32_t &flags, bool &hit, uint32_t &rng)
{
   hit = false;
   uint32_t w0, w1, w2, w3;
   philox (tag, MXG_STAGE_MIRROR, 0u, source_id, (uint32_t) seed, (uint32_t) (seed >> 32), w0, w1, w2, w3);
   const double unit = 1.0 / ((double) 0xFFFFFFFFu);
   if (h.ideal == 0)
     {
        if ((double) w0 * unit > h.vignetting) return false;
        w0 = w1;
        w1 = w2;
        w2 = w3;
     }

   // aperture: shell by cumulative area, radius, open quadrant
   const double r = (double) w0 * unit;
   si = 0;
   for (int k = 0; k < MXG_NUM_SHELLS - 1; k++) si += (r >= h.shell[k].area_fraction) ? 1 : 0;
   bool ok = r < h.shell[MXG_NUM_SHELLS - 1].area_fraction;
   double u_radius = (double) w1 * unit, theta = (double) w2 * unit;
   ok = ok && (0 != (h.shell[si].shutter_bitmap & (1u << (unsigned int) (4.0 * theta))));
   rng = h.ideal ? 3u : 4u;
   if (!ok)
     {
        // a draw outside the open aperture is repeated: the draws again, as
        // the stream takes them
        Stream st;
        stream_init (st, seed, tag, MXG_STAGE_MIRROR, source_id);
        if (h.ideal == 0) (void) uniform (st);
        for (si = -1; si < 0; )
          {
             const double q = uniform (st);
             for (int k = 0; k < MXG_NUM_SHELLS; k++)
               if (q < h.shell[k].area_fraction) { si = k; break; }
          }
        u_radius = uniform (st);
        do theta = uniform (st);
        while (0 == (h.shell[si].shutter_bitmap & (1u << (unsigned int) (4.0 * theta))));
        rng = 4u * st.c2 - 4u + (uint32_t) st.pos;
     }
   const mxg_shell_cfg &S = h.shell[si];
   const double radius = S.min_radius + (S.max_radius - S.min_radius) * u_radius;
   double sn, cs;
   sincos_turn (theta - 1.0 / 8.0, sn, cs);
   x.z = radius * cs;
   x.y = radius * sn;
   x.x = S.front_position;
   x.z -= S.to_osac[0][2];
   x.y -= S.to_osac[0][1];
   if (source_distance > 0.0)
     {
        p = ax1_bx2 (1.0, x, source_distance, p);
        normalize (p);
     }
   double ipx = rcp_n (p.x);
   if (h.use_struts && in_strut_shadow (h, x, p, ipx, h.pre_struts))
     flags |= PHOTON_MIRROR_VBLOCKED;

   x = add (x, ld3 (S.to_osac[0]));
   if (tilted & 1u)
     {
        x = mul_m3_f (S.fwd[0], x);
        p = mul_m3_f (S.fwd[0], p);
        ipx = rcp_n (p.x);
     }

   if (!conic_hit (S.conic_a[0], S.conic_b[0], S.conic_c[0], x, p, ipx, S.conic_xmin[0], S.conic_xmax[0]))
     flags |= PHOTON_UNREFLECTED;
   else
     hit = true;
   return true;
}

// k_hrma_enter's work for photon id of the store (hrma_enter_core).  True
// when the photon hit the paraboloid (its stream position is saved in
// rng_pos[id] for hrma_reflect_one).  FRESH: the photon is as the source
// made it without its position, shell and flags (flags zero, not read);
// they are written here, the position and shell zero when vignetting
// blocks it.
template <bool FRESH = false>
__device__ __forceinline__ bool hrma_enter_one (const mxg_hrma_cfg &h, uint32_t tilted, Soa s, uint32_t id,
                                                uint32_t *__restrict__ rng_pos, double source_distance,
                                                unsigned long long seed, uint32_t source_id)
{
   bool keep = false;
   uint32_t flags = FRESH ? 0u : at (s.flags, id);
   if ((flags & BAD_PHOTON_MASK) == 0)
     {
        vec3 x, p = v3 (at (s.p0, id), at (s.p1, id), at (s.p2, id));
        int si;
        uint32_t rng = 0;
        if (!hrma_enter_core (h, tilted, at (s.tag, id), source_distance, seed, source_id, x, p, si, flags, keep, rng))
          {
             at (s.flags, id) = flags | PHOTON_MIRROR_VBLOCKED;
             if (FRESH)
               {
                  at (s.x0, id) = 0.0; at (s.x1, id) = 0.0; at (s.x2, id) = 0.0;
                  at (s.shell, id) = 0;
               }
          }
        else
          {
             if (keep) rng_pos[id] = rng;
             at (s.x0, id) = x.x; at (s.x1, id) = x.y; at (s.x2, id) = x.z;
             at (s.p0, id) = p.x; at (s.p1, id) = p.y; at (s.p2, id) = p.z;
             at (s.shell, id) = (uint8_t) si;
             at (s.flags, id) = flags;
          }
     }
   return keep;
}

// The photon's optical constants and the square root of its shell's area
// correction factor, interpolated at its energy from the tables in LDS (the
// same values at both surfaces).
__device__ __forceinline__ MirrorIndex mirror_index (const mxg_hrma_cfg &h, const mxg_shell_cfg &S, int si,
                                                     const float *ltab, const HrmaLds &lay, double energy)
{
   double beta = 0.0, delta = 1.0;
   MirrorIndex m;
   m.corr = 1.0;
   if (h.opt_n != 0)
     {
        const float *opt_e = ltab + lay.opt;
        float ef = (float) energy, fb, fd;
        interp_f2b (ef, opt_e, opt_e + h.opt_n, opt_e + 2 * h.opt_n, h.opt_n, h.opt_bucket, ltab + lay.bk_opt,
                    fb, fd);
        beta = fb;
        delta = fd;
        if (h.use_scale)
          m.corr = sqrt_n (interp_fb (ef, ltab + lay.corr_e[si], ltab + lay.corr_f[si], S.corr_n, S.corr_bucket,
                                      ltab + lay.bk_corr[si]));
     }
   m.n2r1 = fma (delta, delta - 2.0, -(beta * beta));
   m.n2r = 1.0 + m.n2r1;
   m.n2i = 2.0 * (1.0 - delta) * beta;
   return m;
}

// From the paraboloid hit on: reflection, cap struts, hyperboloid,
// post-collimator struts, for the photon with tag `tag`, shell si, position x
// on the paraboloid and direction p, its stream at word rng (ring: RingStream).  ltab: the tables
// staged in LDS at the offsets lay.  True when the photon leaves the mirror.
__device__ __forceinline__ bool hrma_reflect_core (const mxg_hrma_cfg &h, const float *ltab, const HrmaLds &lay,
                                                   const float *__restrict__ fa, const double *__restrict__ da,
                                                   uint32_t *ring, uint32_t tag, int si, double energy, uint32_t rng,
                                                   unsigned long long seed, uint32_t source_id, vec3 &x, vec3 &p,
                                                   uint32_t &flags)
{
   const mxg_shell_cfg &S = h.shell[si];
   RingStream st;
   ring_init (st, ring, seed, tag, MXG_STAGE_MIRROR, source_id, rng);
   ring_fill (st);
   top_up (st);
   const MirrorIndex m = mirror_index (h, S, si, ltab, lay, energy);
   const uint32_t tilted = __builtin_amdgcn_readfirstlane (lay.tilted);

   if (0 != reflect_at (h, S, 0, x, p, energy, m, fa, da, ltab + lay.ea[si][0], ltab + lay.bk_ea[si][0], st))
     flags |= PHOTON_UNREFLECTED;
   else
     {
        if (tilted & 1u)
          {
             p = mul_m3_f (S.bwd[0], p);
             x = mul_m3_f (S.bwd[0], x);
          }
        x = sub (x, ld3 (S.to_osac[0]));
        double ipx = rcp_n (p.x);
        if (h.use_struts && in_strut_shadow (h, x, p, ipx, h.cap_struts))
          flags |= PHOTON_MIRROR_VBLOCKED;
        else
          {
             x = add (x, ld3 (S.to_osac[1]));
             if (tilted & 2u)
               {
                  p = mul_m3_f (S.fwd[1], p);
                  x = mul_m3_f (S.fwd[1], x);
                  ipx = rcp_n (p.x);
               }
             if (!conic_hit (S.conic_a[1], S.conic_b[1], S.conic_c[1], x, p, ipx, S.conic_xmin[1], S.conic_xmax[1])
                 || (0 != reflect_at (h, S, 1, x, p, energy, m, fa, da,
                                      ltab + lay.ea[si][1], ltab + lay.bk_ea[si][1], st)))
               flags |= PHOTON_UNREFLECTED;
             else
               {
                  if (tilted & 2u)
                    {
                       p = mul_m3_f (S.bwd[1], p);
                       x = mul_m3_f (S.bwd[1], x);
                    }
                  x = sub (x, ld3 (S.to_osac[1]));
                  if (h.use_struts && in_strut_shadow (h, x, p, rcp_n (p.x), h.post_struts))
                    flags |= PHOTON_MIRROR_VBLOCKED;
               }
          }
     }
   return (flags & BAD_PHOTON_MASK) == 0;
}

// k_hrma_reflect's work for photon id of the middle list (hrma_reflect_core
// on the store's columns).  True when the photon leaves the mirror, its
// columns then also in o.  HANDOFF: such photons go on to the grating
// through o, and the grating stores their x, p and flags; only the photons
// the mirror drops have theirs stored here.
template <bool HANDOFF = false>
__device__ __forceinline__ bool hrma_reflect_one (const mxg_hrma_cfg &h, const float *ltab, const HrmaLds &lay,
                                                  const float *__restrict__ fa, const double *__restrict__ da,
                                                  uint32_t *ring, Soa s, uint32_t id,
                                                  const uint32_t *__restrict__ rng_pos,
                                                  unsigned long long seed, uint32_t source_id, PhotonOut &o)
{
   uint32_t flags = at (s.flags, id);
   const int si = at (s.shell, id);
   const uint32_t tag = at (s.tag, id);
   vec3 x = v3 (at (s.x0, id), at (s.x1, id), at (s.x2, id));
   vec3 p = v3 (at (s.p0, id), at (s.p1, id), at (s.p2, id));
   const double energy = at (s.energy, id);
   const bool keep = hrma_reflect_core (h, ltab, lay, fa, da, ring, tag, si, energy, rng_pos[id], seed, source_id, x,
                                        p, flags);
   if (!(HANDOFF && keep)) store_path (s, id, x, p, flags);
   o.x0 = x.x; o.x1 = x.y; o.x2 = x.z;
   o.p0 = p.x; o.p1 = p.y; o.p2 = p.z;
   o.energy = energy;
   o.tag = tag;
   o.flags = flags;
   o.shell = si;
   return keep;
}

} // namespace mxg
