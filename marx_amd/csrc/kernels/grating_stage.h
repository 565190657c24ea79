// grating_stage.h -- the per-photon work of the HETG / LETG stage, shared by
// the stage kernel (grating.hip) and the chunk kernels (passes.hip).
//
// Per photon (the operations of marx/libsrc/diffract.c:974-1130):
//   grating vignetting draw -> rotate about X into the grating frame ->
//   Rowland-torus intersection by Newton on the quartic (:622-687) ->
//   order draw against the cumulative efficiency table interpolated at the
//   photon energy (the per-photon form of the shell-major
//   JDMinterpolate_n_fvector pass, finterpo.c:134-193) -> facet basis,
//   sector lookup, dtheta and dP/P blur, grating equation (:706-823) ->
//   LETG: fine support grating once, coarse three times (:917-970, 1081-1122)
//   -> rotate back.  Efficiency tables are energy-major so the order walk of
//   one lane touches two contiguous rows.
#pragma once

#include <string.h>
#include "dev_common.h"
#include "dev_store.h"

namespace mxg {

// The root of the quartic t^4 + a t^3 + b t^2 + c t + d by Newton's method
// from t0, as the reference takes it (at most ten steps, to 1e-4 between
// the last two: the root is then good to the square of that over its size).
__device__ __forceinline__ bool newtons_quartic (double a, double b, double c, double d, double t0, double &tp)
{
   const double a2 = 2.0 * a, a3 = 3.0 * a, b2 = 2.0 * b;
   for (int it = 0; it < 10; it++)
     {
        const double t2 = t0 * t0;
        const double num = fma (t2, fma (3.0, t2, fma (a2, t0, b)), -d);
        const double den = fma (t2, fma (4.0, t0, a3), fma (b2, t0, c));
        const double t = div_n (num, den);
        if (fabs (t - t0) < 1.0e-4)
          {
             tp = t;
             return true;
          }
        t0 = t;
     }
   return false;
}

// the hit of a ray on the Rowland torus (diffract.c:622-687)
__device__ __forceinline__ bool torus_intersect (vec3 &x0, vec3 p, double rowland)
{
   const double t = -div_n (x0.x, p.x);
   x0.x = 0.0;
   x0.y = fma (p.y, t, x0.y);
   x0.z = fma (p.z, t, x0.z);
   const double pxpz = fma (p.x, p.x, p.z * p.z);
   const double x2 = fma (x0.z, x0.z, x0.y * x0.y);
   const double r2 = rowland * rowland;
   const double a = 4.0 * fma (p.z, x0.z, p.y * x0.y);
   const double pdotx = 0.25 * a;
   const double b = fma (2.0, x2, fma (a, pdotx, -(r2 * pxpz)));
   const double c = fma (a, x2, -2.0 * r2 * p.z * x0.z);
   const double d = fma (x2, x2, -(r2 * x0.z * x0.z));
   double root;
   if (!newtons_quartic (a, b, c, d, -rowland * sqrt_n (pxpz), root))
     return false;
   x0 = along_f (x0, root, p);
   return true;
}

// Order draw: first k with r <= cumulative efficiency(E); -1 when none.
// The bracket is the one the reference's merge walk over sorted energies
// reaches: the first j >= 1 with E[j] >= e, else the last interval.  E:
// the grating's energies, bcnt: their bucket counts (LDS or the arena).
__device__ __forceinline__ int draw_order (const mxg_grating &g, const float *__restrict__ fa,
                                           const float *E, const float *bcnt, double e, double r)
{
   const unsigned int ne = g.num_energies, no = g.num_orders;
   unsigned int lo = 1, hi = ne - 1;
   const mxg_bucket &b = g.e_bucket;
   const float ef = (float) e;         // e holds a float value
   if (b.ok && (ef > E[0]))
     {
        // the first entry >= e of a strictly increasing table, from the
        // bucket that holds e (mxg_bucket); the bisection below then starts
        // on the answer clamped to [1, ne - 1]
        const uint64_t k = ((uint64_t) __float_as_uint (ef) - b.base) >> b.shift;
        const uint32_t j = (k < b.nb) ? (uint32_t) k : b.nb - 1;
        unsigned int l = (unsigned int) bcnt[j], h = (unsigned int) bcnt[j + 1];
        while (l < h)
          {
             unsigned int mid = (l + h) >> 1;
             if (E[mid] < ef) l = mid + 1;
             else h = mid;
          }
        lo = hi = (l < 1) ? 1u : ((l > ne - 1) ? ne - 1 : l);
     }
   while (lo < hi)
     {
        unsigned int mid = (lo + hi) >> 1;
        if (e > (double) E[mid]) lo = mid + 1;
        else hi = mid;
     }
   const unsigned int count = lo;
   const double x_0 = E[count - 1], x_1 = E[count];
   const double dx_10 = x_1 - x_0;
   const float *y0 = fa + g.cum_eff_off + (count - 1) * no;
   const float *y1 = y0 + no;
   // Inside its interval the interpolated value of order k lies between
   // y0[k] and y1[k] (every step of it rounds within those bounds), so the
   // division is needed only for an order whose bounds straddle r; outside
   // (extrapolation) every order is interpolated.
   const bool inside = (e >= x_0) && (e <= x_1);
   unsigned int k0 = 0;
   if (inside && g.cum_sorted)
     {
        // rows that rise with the order: the bounds do too, so every order
        // before the first whose upper bound reaches r fails, found by
        // bisection
        unsigned int l = 0, h = no;
        while (l < h)
          {
             const unsigned int mid = (l + h) >> 1;
             if (r > (double) fmaxf (y0[mid], y1[mid])) l = mid + 1;
             else h = mid;
          }
        k0 = l;
     }
   for (unsigned int k = k0; k < no; k++)
     {
        const float ya = y0[k], yb = y1[k];
        if (inside)
          {
             if (r > (double) fmaxf (ya, yb)) continue;
             if (r <= (double) fminf (ya, yb)) return (int) k;
          }
        float v;
        if (dx_10 == 0.0)
          v = ya;
        else
          {
             const double a = ya, b = yb, num = (b - a) * (e - x_0);
             v = (float) (a + (inside ? div_n (num, dx_10) : num / dx_10));   // outside, e may be infinite
          }
        if (r <= (double) v)
          return (int) k;
     }
   return -1;
}

// nsec, sec: the shell's sector count and its six columns (LDS or the
// arena), nsec = 0 without a sector table
__device__ __forceinline__ int diffract_photon (const mxg_grating &g, unsigned int nsec, const double *sec,
                                                double theta, double energy, vec3 x, vec3 &p, int order,
                                                Stream &st)
{
   // the general division: a list's energy may be 0, whose photons no order
   // but the zeroth lets pass, or infinite
   const double n_lambda_over_d = (double) order * (2.0 * MXG_PI * MXG_HBAR_C) / (g.period * energy);
   // the facet's normal -x / |x|, and the directions along (l, in the x-z
   // plane) and across (d) its grooves: n . l = 0, so d has length 1
   vec3 n = unit_f (x);
   n.x = -n.x; n.y = -n.y; n.z = -n.z;
   const double il = rsqrt_n (fma (n.x, n.x, n.z * n.z));
   vec3 l = v3 (n.z * il, 0.0, -n.x * il);
   vec3 d = cross_f (n, l);
   double dtheta, dp_over_p;

   if (nsec > 0)
     {
        const double *min_a = sec;
        const double *max_a = min_a + nsec;
        double sector = atan2 (x.y, x.z);
        if (sector < 0) sector = 2 * MXG_PI + sector;
        unsigned int sn = search_d (sector, min_a, nsec) - 1;
        if (sn >= nsec) return -1;
        if ((max_a[sn] <= sector) || (min_a[sn] > sector))
          return -1;
        dtheta = min_a[2 * nsec + sn] + min_a[3 * nsec + sn] * gaussian (st);
        dp_over_p = min_a[4 * nsec + sn] + min_a[5 * nsec + sn] * gaussian (st);
     }
   else
     {
        dtheta = g.theta_blur * gaussian (st);
        dp_over_p = g.dp_over_p * gaussian (st);
     }

   theta -= dtheta;
   if (theta != 0.0)
     {
        double s, c;
        sincos_small (theta, &s, &c);
        const vec3 l_tmp = l, d_tmp = d;
        l = lin2_f (c, l_tmp, s, d_tmp);
        d = lin2_f (-s, l_tmp, c, d_tmp);
     }

   const double p_d = n_lambda_over_d + dot_f (p, d);
   const double p_l = dot_f (p, l);
   const double pn2 = fma (-p_d, p_d, fma (-p_l, p_l, 1.0));
   if (pn2 < 0.0) return -1;
   double ipn;
   const double p_n = sqrt_rsqrt_n (fmax (pn2, 1e-300), ipn);
   p = along_f (lin2_f (p_d, d, p_n, n), p_l, l);
   if (dp_over_p == 0) return 0;
   // dp = -f d + f (p_d / p_n) n
   const double f = n_lambda_over_d * dp_over_p;
   p = unit_f (along_f (along_f (p, -f, d), f * (p_d * ipn), n));
   return 0;
}

// The small tables of grating g (energies, their bucket counts, orders)
// and its shell's sector columns, where the order draw and the diffraction
// search them.
struct GratingTabs
{
   const float *E, *bcnt, *orders;
   const double *sec;
   unsigned int nsec;
};

// one order draw plus diffraction off grating g; returns 0 or -1
__device__ __forceinline__ int diffract_from (const mxg_grating &g, const GratingTabs &t,
                                              const float *__restrict__ fa, double theta,
                                              double energy, double ef, vec3 x, vec3 &p,
                                              int8_t &order_out, Stream &st)
{
   double r = uniform (st);
   int k = draw_order (g, fa, t.E, t.bcnt, ef, r);
   if (k < 0) return -1;
   int order = (int) t.orders[k];
   order_out = (int8_t) order;
   return diffract_photon (g, t.nsec, t.sec, theta, energy, x, p, order, st);
}

// The search tables of the grating stage staged in LDS by k_grating:
// offsets in floats from the table area of gratings 0-3 (by shell), 4 (the
// LETG fine support grating) and 5 (coarse), and of each shell's sector
// columns (doubles, at even offsets).
struct GratingLds
{
   uint32_t e[6], bk[6], ord[6];
   uint32_t sec[MXG_NUM_SHELLS];
   uint32_t floats;
};

// Dynamic LDS of k_grating: the layout at 0, the tables from kGratingTabOff.
constexpr size_t kGratingTabOff = (sizeof (GratingLds) + 15) & ~(size_t) 15;

__host__ __device__ inline const mxg_grating &grating_of (const mxg_grating_cfg &gc, int k)
{
   return (k < MXG_NUM_SHELLS) ? gc.g[k] : ((k == MXG_NUM_SHELLS) ? gc.fine : gc.coarse);
}

// The LDS layout of configuration gc's search tables (host side); letg:
// with the support gratings.
inline GratingLds grating_lds_layout (const mxg_grating_cfg &gc, bool letg)
{
   GratingLds lay = {};
   uint32_t f = 0;
   for (int k = 0; k < 6; k++)
     {
        if ((k >= MXG_NUM_SHELLS) && !(letg && ((k == MXG_NUM_SHELLS) ? gc.has_fine : gc.has_coarse)))
          continue;
        const mxg_grating &g = grating_of (gc, k);
        lay.e[k] = f; f += g.num_energies;
        lay.bk[k] = f; f += bucket_floats (g.e_bucket);
        lay.ord[k] = f; f += g.num_orders;
     }
   for (int sh = 0; sh < MXG_NUM_SHELLS; sh++)
     {
        f = (f + 1) & ~1u;
        lay.sec[sh] = f;
        f += 2 * 6 * gc.sectors[sh].n;
     }
   lay.floats = f;
   return lay;
}

// The LDS image of the tables of lay, made by the host from the arenas fa,
// da: lay at 0, the tables at kGratingTabOff (letg as for the layout),
// grating_image_bytes of it, a multiple of 16.
inline size_t grating_image_bytes (const GratingLds &lay)
{
   return (kGratingTabOff + (size_t) lay.floats * sizeof (float) + 15) & ~(size_t) 15;
}

inline void grating_image (const mxg_grating_cfg &gc, const float *fa, const double *da, const GratingLds &lay,
                           bool letg, unsigned char *img)
{
   memset (img, 0, grating_image_bytes (lay));
   memcpy (img, &lay, sizeof (lay));
   float *tab = (float *) (img + kGratingTabOff);
   auto put = [&] (uint32_t at, uint32_t off, uint32_t n) { if (n) memcpy (tab + at, fa + off, n * sizeof (float)); };
   for (int k = 0; k < 6; k++)
     {
        if ((k >= MXG_NUM_SHELLS) && !(letg && ((k == MXG_NUM_SHELLS) ? gc.has_fine : gc.has_coarse)))
          continue;
        const mxg_grating &g = grating_of (gc, k);
        put (lay.e[k], g.energies_off, g.num_energies);
        put (lay.bk[k], g.e_bucket.off, bucket_floats (g.e_bucket));
        put (lay.ord[k], g.orders_off, g.num_orders);
     }
   for (int sh = 0; sh < MXG_NUM_SHELLS; sh++)
     if (gc.sectors[sh].n)
       memcpy (tab + lay.sec[sh], da + gc.sectors[sh].off, 6 * gc.sectors[sh].n * sizeof (double));
}

// The tables of grating k (0-3 by shell, 4 fine, 5 coarse) and, for k < 4,
// of shell k's sectors: from LDS (STAGED: layout L, tables ltab) or from the
// arenas.
template <bool STAGED>
__device__ __forceinline__ GratingTabs grating_tabs (const mxg_grating_cfg &gc, int k, const float *__restrict__ fa,
                                                     const double *__restrict__ da, const GratingLds *L,
                                                     const float *ltab)
{
   GratingTabs t;
   const mxg_grating &g = grating_of (gc, k);
   const bool shell = k < MXG_NUM_SHELLS;
   t.nsec = shell ? gc.sectors[k].n : 0u;
   if constexpr (STAGED)
     {
        t.E = ltab + L->e[k];
        t.bcnt = ltab + L->bk[k];
        t.orders = ltab + L->ord[k];
        t.sec = shell ? (const double *) (ltab + L->sec[k]) : nullptr;
     }
   else
     {
        t.E = fa + g.energies_off;
        t.bcnt = fa + g.e_bucket.off;
        t.orders = fa + g.orders_off;
        t.sec = shell ? da + gc.sectors[k].off : nullptr;
     }
   return t;
}

// The stream of a photon after its vignetting and order draws.
__device__ __forceinline__ void resume_diffraction (Stream &st, unsigned long long seed, uint32_t tag,
                                                    uint32_t source_id)
{
   uint32_t w0, w1;
   stream_init (st, seed, tag, MXG_STAGE_GRATING, source_id);
   philox (st.c0, st.c1, 0u, st.c3, st.k0, st.k1, w0, w1, st.b0, st.b1);
   st.c2 = 1;
   st.pos = 2;
}

// The grating stage of one photon in two parts, at the order draw: most
// photons find no order (four in five for HETG), and what follows costs
// more than what comes before.
enum GratingStep
{
   GRATING_VIGNETTED,           // flags only: the photon keeps its path
   GRATING_NO_ORDER,            // its path is final
   GRATING_DIFFRACTS            // on the torus, in the grating's frame, with an order
};

// The vignetting draw, the frame rotation, the Rowland torus and the order
// draw of a photon of shell `shell`.  STAGED: the search tables are read from
// LDS (layout L, tables ltab, as k_grating stages them), else from the
// arenas.
template <bool STAGED>
__device__ __forceinline__ GratingStep grating_enter_core (const mxg_grating_cfg &gc, const float *__restrict__ fa,
                                                           const double *__restrict__ da, const GratingLds *L,
                                                           const float *ltab, int shell, double energy, vec3 &x,
                                                           vec3 &p, uint32_t &flags, int8_t &order, Stream &st)
{
   const mxg_grating &g = gc.g[shell];
   if (uniform (st) > g.vig)
     {
        flags |= PHOTON_MIRROR_VBLOCKED;
        return GRATING_VIGNETTED;
     }
   x = turn_x_f (x, g.disp_cos, -g.disp_sin);
   p = turn_x_f (p, g.disp_cos, -g.disp_sin);
   if (!torus_intersect (x, p, gc.rowland[shell]))
     flags |= PHOTON_UNDIFFRACTED;
   const GratingTabs t = grating_tabs<STAGED> (gc, shell, fa, da, L, ltab);
   const int k = draw_order (g, fa, t.E, t.bcnt, (double) (float) energy, uniform (st));
   if (k >= 0)
     {
        order = (int8_t) (int) t.orders[k];
        return GRATING_DIFFRACTS;
     }
   flags |= PHOTON_UNDIFFRACTED;
   x = turn_x_f (x, g.disp_cos, g.disp_sin);
   p = turn_x_f (p, g.disp_cos, g.disp_sin);
   return GRATING_NO_ORDER;
}

// A GRATING_DIFFRACTS photon from there on: the diffraction, for LETG the
// support gratings (their orders to sup), and the rotation back.  True when
// it leaves the grating alive.
template <bool LETG, bool STAGED>
__device__ __forceinline__ bool grating_leave_core (const mxg_grating_cfg &gc, const float *__restrict__ fa,
                                                    const double *__restrict__ da, const GratingLds *L,
                                                    const float *ltab, int shell, double energy, int8_t order,
                                                    vec3 &x, vec3 &p, uint32_t &flags, int8_t *const *sup,
                                                    uint32_t id, Stream &st)
{
   const mxg_grating &g = gc.g[shell];
   const GratingTabs t = grating_tabs<STAGED> (gc, shell, fa, da, L, ltab);
   if (-1 == diffract_photon (g, t.nsec, t.sec, 0.0, energy, x, p, (int) order, st))
     flags |= PHOTON_UNDIFFRACTED;
   if constexpr (LETG)
     {
        const double ef = (double) (float) energy;
        for (int pass = 0; pass < 4; pass++)
          {
             const bool fine = (pass == 0);
             if (fine ? !gc.has_fine : !gc.has_coarse) continue;
             if (flags & BAD_PHOTON_MASK) continue;
             const double theta = (pass == 0) ? MXG_PI / 2.0
               : (pass == 1) ? MXG_PI / 3.0
               : (pass == 2) ? 2.0 * MXG_PI / 3.0 : 0.0;
             int8_t so = at (sup[pass], id);
             if (-1 == diffract_from (fine ? gc.fine : gc.coarse,
                                      grating_tabs<STAGED> (gc, fine ? MXG_NUM_SHELLS : MXG_NUM_SHELLS + 1, fa, da, L,
                                                            ltab),
                                      fa, theta, energy, ef, x, p, so, st))
               flags |= PHOTON_UNDIFFRACTED;
             at (sup[pass], id) = so;
          }
     }
   x = turn_x_f (x, g.disp_cos, g.disp_sin);
   p = turn_x_f (p, g.disp_cos, g.disp_sin);
   return (flags & BAD_PHOTON_MASK) == 0;
}

// k_grating's work for photon id: both parts on the store's columns.  True
// when the photon leaves the grating stage alive, its columns then also in o.
// RELAY: its incoming x, p, energy, tag, flags and shell are read from row
// `slot` of *relay instead of the store, where the mirror left x, p and
// flags for this stage to write (a vignetted photon's as they came).
// HANDOFF: the photons it keeps go on to the detector through o, and the
// detector stores their x, p and flags; only the photons it drops have
// theirs stored here.  STAGED: as grating_enter_core.
template <bool LETG, bool RELAY = false, bool HANDOFF = false, bool STAGED = false>
__device__ __forceinline__ bool grating_one (const mxg_grating_cfg &gc, const float *__restrict__ fa,
                                             const double *__restrict__ da, Soa s, uint32_t id,
                                             unsigned long long seed, uint32_t source_id, PhotonOut &o,
                                             const Relay *relay = nullptr, uint32_t slot = 0,
                                             const GratingLds *L = nullptr, const float *ltab = nullptr)
{
   bool keep = false;
   uint32_t flags = RELAY ? at (relay->flags, slot) : at (s.flags, id);
   if ((flags & BAD_PHOTON_MASK) == 0)
     {
        Stream st;
        const uint32_t tag = RELAY ? at (relay->tag, slot) : at (s.tag, id);
        stream_init (st, seed, tag, MXG_STAGE_GRATING, source_id);
        const int shell = RELAY ? (int) at (relay->shell, slot) : (int) at (s.shell, id);
        vec3 x = RELAY ? v3 (at (relay->x0, slot), at (relay->x1, slot), at (relay->x2, slot)) : v3 (at (s.x0, id), at (s.x1, id), at (s.x2, id));
        vec3 p = RELAY ? v3 (at (relay->p0, slot), at (relay->p1, slot), at (relay->p2, slot)) : v3 (at (s.p0, id), at (s.p1, id), at (s.p2, id));
        const double energy = RELAY ? at (relay->energy, slot) : at (s.energy, id);
        int8_t order = 0;
        const GratingStep step = grating_enter_core<STAGED> (gc, fa, da, L, ltab, shell, energy, x, p, flags, order, st);
        if (step == GRATING_DIFFRACTS)
          {
             at (s.order, id) = order;
             keep = grating_leave_core<LETG, STAGED> (gc, fa, da, L, ltab, shell, energy, order, x, p, flags, s.sup, id,
                                                      st);
          }
        if (!RELAY && (step == GRATING_VIGNETTED)) at (s.flags, id) = flags;
        else if (!(HANDOFF && keep)) store_path (s, id, x, p, flags);
        o.x0 = x.x; o.x1 = x.y; o.x2 = x.z;
        o.p0 = p.x; o.p1 = p.y; o.p2 = p.z;
        o.energy = energy;
        o.tag = tag;
        o.flags = flags;
        o.shell = shell;
     }
   return keep;
}

} // namespace mxg
