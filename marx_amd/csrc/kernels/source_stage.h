// source_stage.h -- the per-photon work of photon creation shared by the
// source kernels (source.hip) and the chunk kernels (passes.hip).
#pragma once

#include "dev_common.h"
#include "dev_store.h"

namespace mxg {

// every column of photon i set as a fresh photon of the given energy,
// direction, time and tag, with no dither offsets; a column that a later
// step writes is left out (with_t, with_p, with_dith false; with_entry
// false: the position, shell and flags, which the mirror's entry writes
// for every photon it is given as fresh).  The columns that no later stage
// reads, or few photons of, are left out of the cache, which then holds those
// that the next stages read and write again.
__device__ __forceinline__ void init_photon (Soa s, uint32_t i, double energy, vec3 p, double t,
                                             uint32_t tag, bool with_t = true, bool with_p = true,
                                             bool with_dith = true, bool with_entry = true)
{
   at (s.energy, i) = energy;
   if (with_p)
     {
        at (s.p0, i) = p.x; at (s.p1, i) = p.y; at (s.p2, i) = p.z;
     }
   if (with_entry)
     {
        at (s.x0, i) = 0.0; at (s.x1, i) = 0.0; at (s.x2, i) = 0.0;
        at (s.flags, i) = 0u;
        at (s.shell, i) = 0;
     }
   if (with_t) put_once (&at (s.t, i), t);
   put_once (&at (s.ypix, i), 0.0f); put_once (&at (s.zpix, i), 0.0f);
   put_once (&at (s.upix, i), 0.0f); put_once (&at (s.vpix, i), 0.0f);
   if (with_dith)
     for (int q = 0; q < 6; q++) put_once (&at (s.dith[q], i), 0.0f);
   put_once (&at (s.pi, i), 0.0f);
   put_once (&at (s.pha, i), (int16_t) 0);
   put_once (&at (s.ccd, i), (int8_t) 0); put_once (&at (s.region, i), (int8_t) 0); put_once (&at (s.order, i), (int8_t) 0);
   for (int q = 0; q < 4; q++) put_once (&at (s.sup[q], i), (int8_t) 0);
   put_once (&at (s.tag, i), tag);
}

// the dither state of photon i: the three pointing offsets d (ra, dec,
// roll), the other three columns zero
__device__ __forceinline__ void store_dith (Soa s, uint32_t i, const float d[3])
{
   for (int q = 0; q < 3; q++)
     {
        put_once (&at (s.dith[q], i), d[q]);
        put_once (&at (s.dith[q + 3], i), 0.0f);
     }
}

// a / |a|, of a vector that a rotation made from a unit vector or, GIVEN, from
// one of any length
template <bool GIVEN>
__device__ __forceinline__ vec3 unit_of (vec3 a)
{
   return GIVEN ? unit_given (a) : reunit_f (a);
}

// The direction of a photon of the configured source shape about the source
// direction p (p_normal: a unit vector normal to p; line_normal and
// line_alpha: the rotation of -x onto p): a point source's p; uniform over
// a disk (s-disk.c:95-106); a Gaussian or beta-model profile
// (s-gauss.c:121-137, s-beta.c:108-124); uniform along a line
// (s-line.c:89-98); a pixel of an image drawn from its cumulative
// distribution (fa + image_off), uniform within the pixel, the image centre
// at -x rotated onto the source direction (s-image.c:284-324).  The angles may
// be of any size: a beta profile of beta near 1/2 has tails of 1e6 radians and
// far more.  The draws
// follow the energy in the source stream.  GIVEN: p is the caller's and need
// not be of length 1 (a batch's directions); the result is.
template <bool GIVEN>
__device__ __forceinline__ vec3 extended_direction (const mxg_source_cfg &src, const float *__restrict__ fa,
                                                    vec3 p, vec3 p_normal, vec3 line_normal, double line_alpha,
                                                    Stream &st)
{
   double sn, cs;
   if (src.type == MXG_SOURCE_DISK)
     {
        sincos_turn (uniform (st), sn, cs);
        const vec3 normal = unit_of<GIVEN> (turn_f (p_normal, p, cs, sn));
        double x0 = src.disk_theta_min / src.disk_theta;
        x0 = x0 * x0;
        double x1 = 1.0 - x0;
        double rnd = src.disk_theta * sqrt_n (x0 + x1 * uniform (st));
        sincos_any (rnd, &sn, &cs);
        return unit_of<GIVEN> (turn_f (p, normal, cs, sn));
     }
   if ((src.type == MXG_SOURCE_GAUSS) || (src.type == MXG_SOURCE_BETA))
     {
        sincos_turn (uniform (st), sn, cs);
        const vec3 normal = unit_of<GIVEN> (turn_f (p_normal, p, cs, sn));
        double rnd;
        do rnd = uniform (st);
        while (rnd == 0.0);
        if (src.type == MXG_SOURCE_GAUSS)
          rnd = src.gauss_sigma * sqrt_n (-log_n (rnd));
        else
          rnd = src.beta_core * sqrt (pow (rnd, src.beta_xpon) - 1.0);
        sincos_any (rnd, &sn, &cs);
        return unit_of<GIVEN> (turn_f (p, normal, cs, sn));
     }
   if (src.type == MXG_SOURCE_IMAGE)
     {
        const unsigned int ofs = search_f ((float) uniform (st), fa + src.image_off, src.image_n);
        double y = (double) (ofs / src.image_nx);
        double x = (double) (ofs % src.image_nx);
        y += -0.5 * src.image_ny + (uniform (st) - 0.5);
        x += -0.5 * src.image_nx + (uniform (st) - 0.5);
        y = y * src.image_yscale;
        x = x * src.image_xscale;
        double sx, cx, sy, cy;
        sincos_any (x, &sx, &cx);
        sincos_any (y, &sy, &cy);
        sincos_r (line_alpha, sn, cs);
        return unit_of<GIVEN> (turn_f (v3 (-cy * cx, cy * sx, -sy), line_normal, cs, sn));
     }
   if (src.type == MXG_SOURCE_LINE)
     {
        double theta = src.line_theta * (-1.0 + 2.0 * uniform (st));
        sincos_any (theta, &sn, &cs);
        const double sin_theta = -sn;
        vec3 q = v3 (-cs, sin_theta * src.line_cos_phi, sin_theta * src.line_sin_phi);
        sincos_r (line_alpha, sn, cs);
        return unit_of<GIVEN> (turn_f (q, line_normal, cs, sn));
     }
   return p;
}

// the angle and unit axis that rotate a onto b (jdmath/src/vector.c:289-331)
__device__ __forceinline__ double rotation_axis (vec3 a, vec3 b, vec3 &c)
{
   double theta = dot (a, b);
   if (theta > 1.0) theta = 1.0;
   else if (theta < -1.0) theta = -1.0;
   theta = acos (theta);
   vec3 cc = cross (a, b);
   double len = length (cc);
   if (len > 0.0)
     {
        c = v3 (cc.x / len, cc.y / len, cc.z / len);
        return theta;
     }
   c = ((a.x != 0.0) || (a.y != 0.0)) ? v3 (-a.y, -a.x, 0.0) : v3 (-a.z, 0.0, 0.0);
   normalize (c);
   return theta;
}

// sine and cosine of the turn by the nominal roll, internal_dither's when the
// roll does not vary (roll_amp = 0)
__device__ __forceinline__ void roll_turn (const mxg_source_cfg &src, double *roll)
{
   sincos_any (-(double) (float) src.nominal_roll, &roll[0], &roll[1]);
}

// INTERNAL dither (dither.c:167-182, 551-581, 609-658) of the photon with
// tag `tag`, direction p and arrival time t: the Lissajous pointing offset
// at that time, returned in d as float (as the reference stores the dither
// state), Gaussian aspect blur, and the rotation of the direction, which is
// returned; GIVEN: p is a direction that the library did not make, of any
// length (the result's is 1).  roll, non-null only where the roll does not vary: sine and
// cosine of roll_turn.
template <bool GIVEN>
__device__ __forceinline__ vec3 internal_dither (const mxg_source_cfg &src, vec3 p, uint32_t tag, double t,
                                                 double start_time, unsigned long long seed,
                                                 uint32_t source_id, float d[3], const double *roll = nullptr)
{
   Stream st;
   stream_init (st, seed, tag, MXG_STAGE_DITHER, source_id);
   // the angles as the reference rounds them: the state is kept as float; the
   // phases grow with the time since the start over the period, without limit
   const double tt = (2.0 * MXG_PI) * (start_time + t);
   float fra = (float) (src.ra_amp * sin_any (div_x (tt, src.ra_period) + src.ra_phase));
   float fdec = (float) (src.dec_amp * sin_any (div_x (tt, src.dec_period) + src.dec_phase));
   float froll = (float) src.nominal_roll;
   if (src.roll_amp != 0.0)
     froll = (float) (src.nominal_roll + src.roll_amp * sin_any (div_x (tt, src.roll_period) + src.roll_phase));
   d[0] = fra; d[1] = fdec; d[2] = froll;
   double delta_ra = src.aspect_blur * gaussian (st);
   double delta_dec = src.aspect_blur * gaussian (st);
   const double ra = (double) fra + delta_ra, dec = (double) fdec + delta_dec;

   double sr, cr;
   if (roll)
     {
        sr = roll[0];
        cr = roll[1];
     }
   else
     sincos_small (-(double) froll, &sr, &cr);
   p = unit_of<GIVEN> (turn_x_f (p, cr, sr));
   double sin_ra, cos_ra, sin_dec, cos_dec;
   sincos_small (ra, &sin_ra, &cos_ra);
   sincos_small (dec, &sin_dec, &cos_dec);
   // the pointing's axis (0, a, b) / sin(theta)
   const double a = sin_dec, b = -cos_dec * sin_ra;
   const double s2 = fma (a, a, b * b);
   if (s2 > 1e-40)
     {
        double inv;
        const double sin_theta = sqrt_rsqrt_n (s2, inv);
        p = reunit_f (turn_f (p, v3 (0.0, a * inv, b * inv), cos_dec * cos_ra, sin_theta));
     }
   return p;
}

// internal_dither applied in place to photon i of the store at time t
__device__ __forceinline__ void apply_internal_dither (const mxg_source_cfg &src, Soa s, uint32_t i,
                                                       double t, double start_time,
                                                       unsigned long long seed, uint32_t source_id)
{
   float d[3];
   vec3 p = internal_dither<true> (src, v3 (at (s.p0, i), at (s.p1, i), at (s.p2, i)), at (s.tag, i), t, start_time, seed, source_id, d);
   store_dith (s, i, d);
   at (s.p0, i) = p.x; at (s.p1, i) = p.y; at (s.p2, i) = p.z;
}

// ---- one source ------------------------------------------------------------------

constexpr int kTile = 2048;          // photons per scan tile
constexpr int kPer = kTile / kBlock; // photons per thread

__device__ __forceinline__ uint64_t gap_ticks (double e)
{
   return (uint64_t) (e * 4294967296.0 + 0.5);
}

// The source stream of photon `tag` (source.c:268-384): its energy, its
// direction and, for Poisson arrivals, the gap to the photon before in
// 2^-32 units of the mean gap (else its uniform arrival time t).  Both
// passes over the photons draw through this, so they see the same values.
// POINT: compiled for a point source only (its direction is the source's,
// with no draw); GAP: only the gap is wanted (the energy draw, one uniform
// for either spectrum, is skipped over without its table search).
template <bool POINT, bool GAP = false>
__device__ __forceinline__ void source_draws (const mxg_source_cfg &src, const float *__restrict__ fa,
                                              const double *__restrict__ da, uint32_t tag,
                                              unsigned long long seed, uint32_t source_id, bool poisson,
                                              double &energy, vec3 &p, uint64_t &gap, double &t)
{
   Stream st;
   stream_init (st, seed, tag, MXG_STAGE_SOURCE, source_id);
   if (GAP)
     {
        (void) uniform (st);
        energy = 0.0;
     }
   else
     energy = draw_energy (src, da, st);
   if (POINT)
     p = ld3 (src.p);
   else
     p = extended_direction<false> (src, fa, ld3 (src.p), ld3 (src.p_normal), ld3 (src.line_normal), src.line_alpha, st);
   gap = 0;
   t = 0.0;
   if (poisson)
     gap = gap_ticks (expn (st));
   else
     t = src.uniform_tmax * uniform (st);
}

// A photon as the source makes it: energy, time, direction (dithered when
// configured, with the offsets d) and whether it is active.
struct NewPhoton
{
   double energy, t;
   vec3 p;
   float d[3];
   bool dithered, active;
};

// Photon i: its draws; with Poisson arrivals its time from the first pass's
// scan and its tile's offset tile_off (null: a single tile), whether it is active (the first
// photon, or its predecessor arrives before the exposure) and, for the first
// photon at or past the exposure, *first_over (unique: the times do not
// decrease); the INTERNAL dither.  POINT: as in source_draws.
template <bool POINT>
__device__ __forceinline__ NewPhoton source_photon (const mxg_source_cfg &src, const float *__restrict__ fa,
                                                    const double *__restrict__ da, uint32_t i, uint32_t tag,
                                                    double exposure_time, double start_time,
                                                    unsigned long long seed, uint32_t source_id,
                                                    const uint64_t *__restrict__ ticks,
                                                    const uint64_t *__restrict__ tile_off,
                                                    uint32_t *__restrict__ first_over,
                                                    const double *roll = nullptr)
{
   NewPhoton ph;
   const bool poisson = (src.time_mode == MXG_TIME_POISSON);
   uint64_t k;
   source_draws<POINT> (src, fa, da, tag, seed, source_id, poisson, ph.energy, ph.p, k, ph.t);
   ph.active = true;
   if (poisson)
     {
        const uint64_t toff = tile_off ? tile_off[i / kTile] : 0ull;
        const double mt = src.mean_time;
        ph.t = mt * ((double) (ticks[i] + toff) * (1.0 / 4294967296.0));
        if ((exposure_time > 0.0) && (i > 0))
          {
             const uint64_t Sp = ((i % kTile) == 0) ? toff : ticks[i - 1] + toff;
             const double tp = mt * ((double) Sp * (1.0 / 4294967296.0));
             ph.active = !(exposure_time <= tp);
          }
        if (ph.active && (exposure_time > 0.0) && (exposure_time <= ph.t))
          __hip_atomic_store (first_over, i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
     }
   ph.dithered = (src.dither_mode == MXG_DITHER_INTERNAL);
   if (ph.dithered)
     ph.p = internal_dither<false> (src, ph.p, tag, ph.t, start_time, seed, source_id, ph.d, roll);
   return ph;
}

// ---- batched point sources ------------------------------------------------------
//
// Photon i (0 <= i < n) of a batch belongs to the source k with
// off[k] <= i < off[k + 1]: direction dir[3k..3k+2] (unit vector of travel),
// tag *tag_start + i, arrival time uniform over [0, exposure), energy from
// the configured spectrum, INTERNAL dither when configured.  The tag alone
// keys the photon's random streams, so tracing a source alone with
// tag_start = off[k] gives the same photons.  tag_start is read from device
// memory so that a captured launch sequence can be replayed for new tags.
// The kernel also writes the identity active list and its length.

__device__ __forceinline__ uint32_t source_of (const uint32_t *__restrict__ off, uint32_t nsrc, uint32_t i)
{
   uint32_t lo = 0, hi = nsrc;         // off[lo] <= i < off[hi]
   while (hi > lo + 1)
     {
        uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= i) lo = mid;
        else hi = mid;
     }
   return lo;
}

// source_of for the photons first, first + 1, ... of a wave's lanes, by all
// of its lanes: the wave looks for the first photon's source with a probe a
// lane, a step for each factor of 64 sources, and each lane goes on from
// there.
__device__ __forceinline__ uint32_t source_of_wave (const uint32_t *__restrict__ off, uint32_t nsrc, uint32_t first,
                                                    uint32_t i)
{
   const uint32_t lane = __lane_id ();
   uint32_t lo = 0, hi = nsrc;         // off[lo] <= first < off[hi]
   while (hi - lo > 1)
     {
        const uint32_t step = (hi - lo + 63u) / 64u, at = lo + lane * step;
        const uint32_t c = (uint32_t) __popcll (__ballot ((at < hi) && (off[at] <= first)));
        lo += (c - 1u) * step;
        hi = (hi - lo < step) ? hi : lo + step;
     }
   // the sources are mostly longer than a wave
   for (int k = 0; k < 4; k++)
     {
        if (i < off[lo + 1]) return lo;
        if (lo + 2 >= nsrc) return nsrc - 1;
        lo++;
     }
   hi = nsrc;
   while (hi > lo + 1)
     {
        const uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= i) lo = mid;
        else hi = mid;
     }
   return lo;
}

// Photon i of the batch, of source k, with tag `tag`.  POINT: compiled for point sources
// only (the extended shapes' code, and its registers, left out).
template <bool POINT>
__device__ __forceinline__ NewPhoton batch_photon (const mxg_source_cfg &src, const double *__restrict__ da, uint32_t k,
                                                   uint32_t tag, const double *__restrict__ dir, double exposure,
                                                   double start_time, unsigned long long seed,
                                                   const double *roll = nullptr)
{
   NewPhoton ph;
   Stream st;
   stream_init (st, seed, tag, MXG_STAGE_SOURCE, 0u);
   ph.energy = draw_energy (src, da, st);
   ph.p = v3 (dir[3 * k], dir[3 * k + 1], dir[3 * k + 2]);
   if (!POINT && (src.type != MXG_SOURCE_POINT))
     {
        // the shape about this source's direction: its normal as the
        // source set-up makes it, and the rotation of -x onto it
        vec3 nrm = v3 (-ph.p.y / ph.p.x, 1.0, 0.0);
        normalize (nrm);
        vec3 ln = v3 (0.0, 0.0, 0.0);
        double la = 0.0;
        if (src.type == MXG_SOURCE_LINE) la = rotation_axis (v3 (-1.0, 0.0, 0.0), ph.p, ln);
        ph.p = extended_direction<true> (src, nullptr, ph.p, nrm, ln, la, st);
     }
   ph.t = exposure * uniform (st);
   ph.active = true;
   ph.dithered = (src.dither_mode == MXG_DITHER_INTERNAL);
   if (ph.dithered) ph.p = internal_dither<true> (src, ph.p, tag, ph.t, start_time, seed, 0u, ph.d, roll);
   return ph;
}

// Photon i of the batch (tag t0 + i) written to the store: k_batch_source's
// work for one photon.  ENTRY: the mirror's entry follows with the photon as
// fresh (see init_photon), so its position, shell and flags are left to it.
template <bool POINT, bool ENTRY = false>
__device__ __forceinline__ void batch_source_one (const mxg_source_cfg &src, const double *__restrict__ da, Soa s,
                                                  uint32_t i, const uint32_t *__restrict__ off, uint32_t nsrc,
                                                  const double *__restrict__ dir, uint32_t t0, double exposure,
                                                  double start_time, unsigned long long seed)
{
   const NewPhoton ph = batch_photon<POINT> (src, da, source_of (off, nsrc, i), t0 + i, dir, exposure, start_time, seed);
   init_photon (s, i, ph.energy, ph.p, ph.t, t0 + i, true, true, !ph.dithered, !ENTRY);
   if (ph.dithered) store_dith (s, i, ph.d);
}

} // namespace mxg
