// hrma_stage.h -- the per-photon work of the HRMA stage (marx/libsrc/hrma.c),
// shared by the stage kernels (hrma.hip) and the one-launch batch pass
// (persist.hip).
//
// Per photon (the operations of marx/libsrc/hrma.c:1161-1341):
//   vignetting draw -> aperture sampling by cumulative shell area, radius and
//   shutter-checked azimuth (hrma.c:984-1050) -> paraboloid: conic
//   intersection (hrma.c:411-478), normal blur (:1054-1093), Fresnel
//   reflectivity draw (reflect.c:39-77), specular reflection, WFold scatter
//   (wfold.c:334-369) -> cap struts -> hyperboloid: the same -> post-collimator
//   struts.  Geometry is FP64.
//
// The mirror's work is split in two at the paraboloid hit (hrma_enter_one,
// hrma_reflect_one).  The stream position is the Philox block counter c2
// and the index of the next unused word of the current block, packed as
// (c2 << 3) | pos.  No Gaussian variate is pending at the split (none is
// drawn before it), and the buffered block is recomputed from c2 - 1 on
// resumption.  (A second split at the hyperboloid hit, each part on the
// photons still alive, measured 37 percent slower: the second kernel
// repeats the stream resumption, the table lookups and the LDS staging.)
#pragma once

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
__device__ __forceinline__ void blur_normal (vec3 &n, double blur, Stream &st)
{
   const double n2 = fma (n.y, n.y, n.z * n.z);
   const double il = rsqrt_n (n2);
   double s, c;
   sincos_turn (uniform (st), s, c);
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
                                           const float *__restrict__ ea_cnt, Stream &st)
{
   vec3 normal = conic_normal (S.conic_a[k], S.conic_b[k], x);
   if (h.use_blur)
     blur_normal (normal, S.blur[k], st);
   const double p_dot_n = dot_f (p, normal);
   if ((h.ideal == 0) && fresnel_absorbs (uniform (st), fabs (p_dot_n), m))
     return -1;
   p = along_f (p, -2.0 * p_dot_n, normal);
   if (h.use_wfold == 0)
     return 0;
   double r = uniform (st);
   double dg = wfold_interp (S.wfold[k], fa, da, e_alphas, energy, -p_dot_n, r, &S.ea_bucket[k], ea_cnt);
   dg *= S.scat_factor[k];
   if (dg > MXG_PI / 4) return -1;
   if (uniform (st) < 0.5) dg = -dg;
   // p turned by dg about p x n, which is at right angles to p and not of
   // length 1: cos p + sin (p x n) x p, with (p x n) x p = n - p (p . n)
   // and p . n = -p_dot_n after the reflection
   double sn, cs;
   sincos_small (dg, &sn, &cs);
   p = unit_f (lin2_f (fma (sn, p_dot_n, cs), p, sn, normal));
   return 0;
}

// Copies the mirror configuration (a multiple of 4 bytes) into LDS.
__device__ __forceinline__ void stage_hrma_cfg (const mxg_config *__restrict__ cfg, unsigned char *lds)
{
   constexpr uint32_t cfg_words = sizeof (mxg_hrma_cfg) / 4;
   const uint32_t *src = (const uint32_t *) &cfg->hrma;
   uint32_t *dst = (uint32_t *) lds;
   for (uint32_t w = threadIdx.x; w < cfg_words; w += blockDim.x) dst[w] = src[w];
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

// The LDS layout of the reflection tables for configuration h (host side).
inline HrmaLds hrma_lds_layout (const mxg_hrma_cfg &h)
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

// bucket counts of table b from the float arena into LDS at dst
__device__ __forceinline__ void stage_bucket (const mxg_bucket &b, const float *__restrict__ fa, float *dst)
{
   if (!b.ok) return;
   for (uint32_t w = threadIdx.x; w <= b.nb; w += blockDim.x) dst[w] = fa[b.off + w];
}

// Stages the mirror configuration and the reflection tables (the
// binary-search targets of every photon) in LDS: the configuration copy at
// lds, lay at lds + kHrmaLayOff, the tables at ltab (lds + kHrmaTabOff) +
// the offsets of lay.  The caller synchronises.
__device__ __forceinline__ void stage_hrma_tables (const mxg_config *__restrict__ cfg, const float *__restrict__ fa,
                                                   const double *__restrict__ da, const HrmaLds &lay,
                                                   unsigned char *lds, float *ltab)
{
   stage_hrma_cfg (cfg, lds);
   if (threadIdx.x == 0) *(HrmaLds *) (lds + kHrmaLayOff) = lay;
   {
      const mxg_hrma_cfg &gh = cfg->hrma;
      for (uint32_t w = threadIdx.x; w < gh.opt_n; w += blockDim.x)
        {
           ltab[lay.opt + w] = fa[gh.opt_e_off + w];
           ltab[lay.opt + gh.opt_n + w] = fa[gh.opt_beta_off + w];
           ltab[lay.opt + 2 * gh.opt_n + w] = fa[gh.opt_delta_off + w];
        }
      stage_bucket (gh.opt_bucket, fa, ltab + lay.bk_opt);
      for (int sh = 0; sh < MXG_NUM_SHELLS; sh++)
        {
           const mxg_shell_cfg &S = gh.shell[sh];
           for (uint32_t w = threadIdx.x; w < S.corr_n; w += blockDim.x)
             {
                ltab[lay.corr_e[sh] + w] = fa[S.corr_e_off + w];
                ltab[lay.corr_f[sh] + w] = fa[S.corr_f_off + w];
             }
           stage_bucket (S.corr_bucket, fa, ltab + lay.bk_corr[sh]);
           for (int k = 0; k < 2; k++)
             {
                for (uint32_t w = threadIdx.x; w < S.wfold[k].n_arrays; w += blockDim.x)
                  ltab[lay.ea[sh][k] + w] = (float) da[S.wfold[k].e_alphas_off + w];
                stage_bucket (S.ea_bucket[k], fa, ltab + lay.bk_ea[sh][k]);
             }
        }
   }
}

// The source-to-paraboloid part of the mirror for an unabsorbed photon with
// tag `tag` and direction p (tilted: HrmaLds): vignetting, aperture, precollimator struts,
// frame change and the paraboloid intersection.  False when vignetting
// blocks the photon (nothing else is drawn); else true, with its position
// x, direction p, shell si and the mirror's marks added to flags; *hit: it
// hit the paraboloid, its random-stream position in *rng.
__device__ __forceinline__ bool hrma_enter_core (const mxg_hrma_cfg &h, uint32_t tilted, uint32_t tag,
                                                 double source_distance,
                                                 unsigned long long seed, uint32_t source_id, vec3 &x,
                                                 vec3 &p, int &si, uint32_t &flags, bool &hit, uint32_t &rng)
{
   Stream st;
   stream_init (st, seed, tag, MXG_STAGE_MIRROR, source_id);
   hit = false;
   if ((h.ideal == 0) && (uniform (st) > h.vignetting))
     return false;

   // aperture: shell by cumulative area, radius, open quadrant
   for (;;)
     {
        double r = uniform (st);
        si = -1;
        for (int k = 0; k < MXG_NUM_SHELLS; k++)
          if (r < h.shell[k].area_fraction) { si = k; break; }
        if (si >= 0) break;
     }
   const mxg_shell_cfg &S = h.shell[si];
   double radius = S.min_radius + (S.max_radius - S.min_radius) * uniform (st);
   double theta;
   unsigned int quad;
   do
     {
        theta = uniform (st);
        quad = (unsigned int) (4.0 * theta);
     }
   while (0 == (S.shutter_bitmap & (1u << quad)));
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
     {
        hit = true;
        rng = (st.c2 << 3) | (uint32_t) st.pos;
     }
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
   uint32_t flags = FRESH ? 0u : s.flags[id];
   if ((flags & BAD_PHOTON_MASK) == 0)
     {
        vec3 x, p = v3 (s.p0[id], s.p1[id], s.p2[id]);
        int si;
        uint32_t rng = 0;
        if (!hrma_enter_core (h, tilted, s.tag[id], source_distance, seed, source_id, x, p, si, flags, keep, rng))
          {
             s.flags[id] = flags | PHOTON_MIRROR_VBLOCKED;
             if (FRESH)
               {
                  s.x0[id] = 0.0; s.x1[id] = 0.0; s.x2[id] = 0.0;
                  s.shell[id] = 0;
               }
          }
        else
          {
             if (keep) rng_pos[id] = rng;
             s.x0[id] = x.x; s.x1[id] = x.y; s.x2[id] = x.z;
             s.p0[id] = p.x; s.p1[id] = p.y; s.p2[id] = p.z;
             s.shell[id] = (uint8_t) si;
             s.flags[id] = flags;
          }
     }
   return keep;
}

// The stream of photon id at the mirror's split, saved by hrma_enter_one.
__device__ __forceinline__ void resume_stream (Stream &st, const uint32_t *__restrict__ rng_pos, uint32_t id)
{
   const uint32_t w = rng_pos[id];
   st.c2 = w >> 3;
   st.pos = (int) (w & 7u);
   if (st.pos < 4)
     {
        // the block again, less the words already used
        philox (st.c0, st.c1, st.c2 - 1u, st.c3, st.k0, st.k1, st.b0, st.b1, st.b2, st.b3);
        for (int k = 0; k < st.pos; k++)
          {
             st.b0 = st.b1;
             st.b1 = st.b2;
             st.b2 = st.b3;
          }
     }
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

// k_hrma_reflect's work for photon id of the middle list: paraboloid
// reflection, cap struts, hyperboloid, post-collimator struts.  ltab: the
// tables staged in LDS at the offsets lay.  True when the photon leaves the
// mirror, its columns then also in o.  HANDOFF: such photons go on to the
// grating through o, and the grating stores their x, p and flags; only the
// photons the mirror drops have theirs stored here.
template <bool HANDOFF = false>
__device__ __forceinline__ bool hrma_reflect_one (const mxg_hrma_cfg &h, const float *ltab, const HrmaLds &lay,
                                                  const float *__restrict__ fa, const double *__restrict__ da,
                                                  Soa s, uint32_t id, const uint32_t *__restrict__ rng_pos,
                                                  unsigned long long seed, uint32_t source_id, PhotonOut &o)
{
   uint32_t flags = s.flags[id];
   const int si = s.shell[id];
   const mxg_shell_cfg &S = h.shell[si];
   Stream st;
   const uint32_t tag = s.tag[id];
   stream_init (st, seed, tag, MXG_STAGE_MIRROR, source_id);
   resume_stream (st, rng_pos, id);
   vec3 x = v3 (s.x0[id], s.x1[id], s.x2[id]);
   vec3 p = v3 (s.p0[id], s.p1[id], s.p2[id]);
   const double energy = s.energy[id];
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
   const bool keep = (flags & BAD_PHOTON_MASK) == 0;
   if (!(HANDOFF && keep))
     {
        s.x0[id] = x.x; s.x1[id] = x.y; s.x2[id] = x.z;
        s.p0[id] = p.x; s.p1[id] = p.y; s.p2[id] = p.z;
        s.flags[id] = flags;
     }
   o.x0 = x.x; o.x1 = x.y; o.x2 = x.z;
   o.p0 = p.x; o.p1 = p.y; o.p2 = p.z;
   o.energy = energy;
   o.tag = tag;
   o.flags = flags;
   o.shell = si;
   return keep;
}

} // namespace mxg
