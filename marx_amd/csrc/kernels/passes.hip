// passes.hip -- the device-created trace as two or three kernels over the
// whole chunk, for chunks that fill the chip.
//
//   k_create:   source and dither, the mirror's entry up to the paraboloid
//   k_mirror:   both reflections, then in the same lanes what cheaply decides
//               most survivors: without a grating the detector, with one the
//               Rowland torus and the order draw
//   k_diffract: the photons with an order: diffraction, then the detector
//
// Kernels that do one stage each are bound by the columns they exchange: a
// stage alive on a third of the photons still touches nearly every line of
// each column it reads and writes.  Here a photon's path leaves the chip when
// it is made (every line written whole), when the mirror drops or finishes
// it, and for the few that are diffracted once more; the hand-over to
// k_diffract is dense rows (Relay).  The list from k_create carries the
// photon's shell, strut shadow and stream position beside its id, so
// k_mirror reads position, direction and energy only.
//
// A wave of the second kernel loses the lanes of the photons the mirror drops
// (38 percent) through the short part that follows; that costs less than
// writing, listing and reading the survivors.
//
// k_mirror's wave stores what it dropped and what it finished in one go: as
// two stores, each of which wrote part of the lines, it took 0.58 ms (batch
// of 6e7: 3.90, now 3.41).  Waves with ranges of their own, without the
// block's barrier, took longer (0.55): a block's waves share lines.
//
// Paths of large chunks go past the caches from k_create and k_mirror
// (chunk_path): the lines are nearly whole and nobody reads them before the
// kernel ends.  With plain stores k_create took 0.525 ms; k_diffract's few
// photons a line are merged in the cache (0.150 ms, 0.168 past it).
//
// What bounds them now (MI355X, HETG + ACIS-S, 1e7 photons): k_create 0.39 ms,
// 1.30 GB written (126 bytes a photon: once each), the ALUs busy 73 percent;
// k_mirror 0.54 ms, 1.16 GB, the ALUs busy 60 percent at four waves a SIMD;
// k_diffract 0.15 ms, 0.26 GB.  As kernels a stage: source 0.41,
// entry 0.25, reflection 0.68, grating 0.36, detector 0.17 ms.  One launch of
// independent waves that queue photons for each stage in LDS measured 1.62 ms
// in all against 1.37: its three waves a SIMD wait for memory at every stage.
#include "source_stage.h"
#include "hrma_stage.h"
#include "grating_stage.h"
#include "detect_stage.h"
#include "passes.h"

namespace mxg {

// An entry of the list from k_create: the photon's id (below 2^28), shell,
// whether a strut shadows it, and whether its mirror stream is elsewhere than
// after the draws that every photon makes (then rng_pos holds where).
constexpr uint32_t kIdBits = 28, kIdMask = (1u << kIdBits) - 1u;
constexpr uint32_t kBlocked = 1u << 30, kOddStream = 1u << 31;

// the stream position after the entry's draws (vignetting unless ideal,
// shell, radius, azimuth) when none was repeated
__device__ __forceinline__ uint32_t usual_stream (const mxg_hrma_cfg &h)
{
   return h.ideal ? 3u : 4u;
}

// Cycles that wave 0 of the first 64 blocks spends in each of the two parts
// of a kernel: they share the kernel's time between the stages.
struct PartClock
{
   uint64_t last, part[2];
   __device__ __forceinline__ PartClock () : last (__builtin_readcyclecounter ()), part {0, 0} {}
   __device__ __forceinline__ void spent (int k)
   {
      const uint64_t now = __builtin_readcyclecounter ();
      part[k] += now - last;
      last = now;
   }
   __device__ __forceinline__ void finish (TraceReport *sums, int first)
   {
      if ((blockIdx.x < 64) && (threadIdx.x == 0))
        for (int k = 0; k < 2; k++)
          atomicAdd ((unsigned long long *) &sums->busy[first + k], (unsigned long long) part[k]);
   }
};

// POINT: compiled for a point source; BATCH: photons of a batch of point
// sources.
template <bool POINT, bool BATCH>
__global__ __launch_bounds__ (kBlock)
void k_create (TraceArgs first, ListIO io, uint32_t tilted)
{
   __shared__ __align__ (16) unsigned char lds[kHrmaLayOff];
   __shared__ uint32_t seg_wc[2 * (kBlock / 64)];
   __shared__ double roll_lds[2];
   if ((blockIdx.x == 0) && (threadIdx.x == 0))
     {
        first.sums->create = wall_clock64 ();
        *first.n_dev = first.n;
     }
   stage_image (first.mirror.img, kHrmaLayOff / 16, lds);
   if (threadIdx.x == 0) roll_turn (first.cfg->src, roll_lds);
   const double *roll = (first.cfg->src.roll_amp == 0.0) ? roll_lds : nullptr;
   __syncthreads ();
   const mxg_hrma_cfg &h = *(const mxg_hrma_cfg *) lds;
   const uint32_t usual = usual_stream (h);
   const uint32_t t0 = BATCH ? *first.batch_tag : first.tag_start;
   const BlockRange range = block_range (first.n, blockIdx.x, gridDim.x);
   SegWriter hits (io, range, seg_wc);
   PartClock clock;

   for (uint32_t base = range.lo; base < range.hi; base += kBlock)
     {
        const uint32_t i = base + threadIdx.x;
        const uint32_t tag = t0 + i;
        bool keep = false;
        uint32_t entry = 0;
        const TraceArgs a = kernel_args<TraceArgs> ();
        const mxg_source_cfg &src = a.cfg->src;
        NewPhoton ph;
        ph.active = false;
        uint32_t k = 0;
        if (BATCH)
          {
             const uint32_t wave0 = __builtin_amdgcn_readfirstlane (base + (threadIdx.x & ~63u));
             if (wave0 < range.hi) k = source_of_wave (a.off, a.nsrc, wave0, i);
          }
        if (i < range.hi)
          {
             if (BATCH) ph = batch_photon<POINT> (src, a.da, k, tag, a.dir, a.exposure, a.start_time, a.seed, roll);
             else ph = source_photon<POINT> (src, a.fa, a.da, i, tag, a.exposure, a.start_time, a.seed, 0u, a.ticks,
                                             a.tile_off, a.first_over, roll);
             // a photon past the exposure cut is not among those created
             init_photon (a.s, i, ph.energy, ph.p, ph.t, tag, true, !ph.active, !ph.dithered, false);
             if (ph.dithered) store_dith (a.s, i, ph.d);
          }
        clock.spent (0);
        if (ph.active)
          {
             vec3 x = v3 (0.0, 0.0, 0.0), p = ph.p;
             int si = 0;
             uint32_t flags = 0, rng = usual;
             if (hrma_enter_core (h, tilted, tag, src.distance, a.seed, 0u, x, p, si, flags, keep, rng))
               {
                  if (keep && (rng != usual)) a.rng_pos[i] = rng;
               }
             else
               {
                  // vignetted: as the source made it
                  x = v3 (0.0, 0.0, 0.0);
                  p = ph.p;
                  si = 0;
                  flags = PHOTON_MIRROR_VBLOCKED;
               }
             chunk_path (a.s, a.n, i, x, p, flags);
             at (a.s.shell, i) = (uint8_t) si;
             entry = i | ((uint32_t) si << kIdBits) | (flags ? kBlocked : 0u) | ((rng != usual) ? kOddStream : 0u);
          }
        hits.add (keep, entry);
        clock.spent (1);
     }
   hits.finish (io);
   clock.finish (first.sums, 0);
}

// per-wave counts summed over the block into out[0..1] (thread 0)
__device__ __forceinline__ void block_counts (uint32_t c0, uint32_t c1, uint32_t *lds, uint32_t *out)
{
   const uint32_t wave = threadIdx.x >> 6;
   __syncthreads ();
   if ((threadIdx.x & 63u) == 0)
     {
        lds[2 * wave] = c0;
        lds[2 * wave + 1] = c1;
     }
   __syncthreads ();
   if (threadIdx.x < 2)
     {
        uint32_t s = 0;
        for (int w = 0; w < kBlock / 64; w++) s += lds[2 * w + threadIdx.x];
        out[threadIdx.x] = s;
     }
}

// G: with a grating, HETG or LETG (the same code: the support gratings come
// later); KIND: without one the detector family, -1 none.
// counts[2 b], [2 b + 1]: photons of block b out of the mirror, and detected.
template <bool G, int KIND>
__global__ __launch_bounds__ (kBlock, 4)
void k_mirror (TraceArgs a, ListIO io, Relay out, uint32_t *__restrict__ counts)
{
   extern __shared__ __align__ (16) unsigned char lds[];
   __shared__ uint32_t seg_wc[2 * (kBlock / 64)];
   __shared__ uint32_t rings[kBlock / 64][kRing][64];
   if ((blockIdx.x == 0) && (threadIdx.x == 0)) a.sums->mirror = wall_clock64 ();
   float *ltab = (float *) (lds + kHrmaTabOff);
   stage_image (a.mirror.img, a.mirror.n16, lds);
   __syncthreads ();
   uint32_t *ring = &rings[threadIdx.x >> 6][0][threadIdx.x & 63u];
   const mxg_hrma_cfg &h = *(const mxg_hrma_cfg *) lds;
   const HrmaLds &L = *(const HrmaLds *) (lds + kHrmaLayOff);
   const uint32_t usual = usual_stream (h);
   const uint32_t t0 = a.batch_tag ? *a.batch_tag : a.tag_start;
   const BlockRange range = block_range (*io.n_in, blockIdx.x, gridDim.x);
   SegWriter ordered (io, range, seg_wc);
   // a lane's list entry is read a photon ahead
   uint32_t next = (range.lo + threadIdx.x < range.hi) ? io.idx_in[range.lo + threadIdx.x] : 0u;
   uint32_t mirrored = 0, detected = 0;
   PartClock clock;

   for (uint32_t base = range.lo; base < range.hi; base += kBlock)
     {
        const uint32_t i = base + threadIdx.x, entry = next;
        if (i + kBlock < range.hi) next = io.idx_in[i + kBlock];
        bool keep = false;
        uint32_t id = 0, flags = PHOTON_UNREFLECTED;
        int si = 0;
        double energy = 0.0;
        vec3 x, p;
        if (i < range.hi)
          {
             id = entry & kIdMask;
             si = (int) ((entry >> kIdBits) & 3u);
             flags = (entry & kBlocked) ? PHOTON_MIRROR_VBLOCKED : 0u;
             x = v3 (at (a.s.x0, id), at (a.s.x1, id), at (a.s.x2, id));
             p = v3 (at (a.s.p0, id), at (a.s.p1, id), at (a.s.p2, id));
             energy = at (a.s.energy, id);
             const uint32_t rng = (entry & kOddStream) ? a.rng_pos[id] : usual;
             keep = hrma_reflect_core (h, ltab, L, a.fa, a.da, ring, t0 + id, si, energy, rng, a.seed, 0u, x, p, flags);
          }
        clock.spent (0);
        mirrored += (uint32_t) __popcll (__ballot (keep));
        if constexpr (G)
          {
             int8_t order = 0;
             if (keep)
               {
                  Stream st;
                  stream_init (st, a.seed, t0 + id, MXG_STAGE_GRATING, 0u);
                  keep = GRATING_DIFFRACTS == grating_enter_core<false> (a.cfg->grating, a.fa, a.da, nullptr, nullptr, si,
                                                                         energy, x, p, flags, order, st);
               }
             // dropped by either stage: one store for both
             if ((i < range.hi) && !keep) chunk_path (a.s, a.n, id, x, p, flags);
             const uint32_t q = ordered.add (keep, id);
             if (keep)
               {
                  // the row's tag column holds the order: the tag follows from the id
                  PhotonOut o;
                  o.x0 = x.x; o.x1 = x.y; o.x2 = x.z;
                  o.p0 = p.x; o.p1 = p.y; o.p2 = p.z;
                  o.energy = energy;
                  o.tag = (uint32_t) (int) order;
                  o.flags = flags;
                  o.shell = si;
                  relay_put (out, q, o);
               }
          }
        else if constexpr (KIND >= 0)
          {
             if (keep)
               keep = detect_core<false, KIND> (a.cfg->det, a.fa, a.da, a.s, id, t0 + id, energy, x, p, flags, a.tstart,
                                                a.seed, 0u);
             detected += (uint32_t) __popcll (__ballot (keep));
          }
        // the mirror's and the detector's photons in one store
        if (!G && (i < range.hi)) chunk_path (a.s, a.n, id, x, p, flags);
        clock.spent (1);
     }
   if (G) ordered.finish (io);
   block_counts (mirrored, detected, seg_wc, counts + 2 * blockIdx.x);
   clock.finish (a.sums, 2);
}

// The photons with an order, from k_mirror's rows; counts[2 b], [2 b + 1]:
// photons of block b out of the grating, and detected.
template <bool LETG, int KIND>
__global__ __launch_bounds__ (kBlock)
void k_diffract (TraceArgs a, const uint32_t *__restrict__ idx, const uint32_t *__restrict__ n_idx, Relay in,
                 uint32_t *__restrict__ counts)
{
   extern __shared__ __align__ (16) unsigned char lds[];
   __shared__ uint32_t wave_counts[2 * (kBlock / 64)];
   if ((blockIdx.x == 0) && (threadIdx.x == 0)) a.sums->diffract = wall_clock64 ();
   float *gtab = (float *) (lds + kGratingTabOff);
   stage_image (a.grating.img, a.grating.n16, lds);
   __syncthreads ();
   const uint32_t t0 = a.batch_tag ? *a.batch_tag : a.tag_start;
   const BlockRange range = block_range (*n_idx, blockIdx.x, gridDim.x);
   uint32_t diffracted = 0, detected = 0;
   PartClock clock;

   for (uint32_t base = range.lo; base < range.hi; base += kBlock)
     {
        const uint32_t i = base + threadIdx.x;
        bool keep = false;
        uint32_t id = 0, flags = 0;
        double energy = 0.0;
        vec3 x, p;
        if (i < range.hi)
          {
             id = idx[i];
             const uint32_t q = in.pos[i];
             x = v3 (at (in.x0, q), at (in.x1, q), at (in.x2, q));
             p = v3 (at (in.p0, q), at (in.p1, q), at (in.p2, q));
             energy = at (in.energy, q);
             flags = at (in.flags, q);
             const int8_t order = (int8_t) (int) at (in.tag, q);
             at (a.s.order, id) = order;
             Stream st;
             resume_diffraction (st, a.seed, t0 + id, 0u);
             keep = grating_leave_core<LETG, true> (a.cfg->grating, a.fa, a.da, (const GratingLds *) lds, gtab,
                                                    (int) at (in.shell, q), energy, order, x, p, flags, a.s.sup, id, st);
          }
        diffracted += (uint32_t) __popcll (__ballot (keep));
        clock.spent (0);
        if constexpr (KIND >= 0)
          {
             if (keep)
               keep = detect_core<false, KIND> (a.cfg->det, a.fa, a.da, a.s, id, t0 + id, energy, x, p, flags, a.tstart,
                                                a.seed, 0u);
             detected += (uint32_t) __popcll (__ballot (keep));
          }
        if (i < range.hi) store_path (a.s, id, x, p, flags);
        clock.spent (1);
     }
   block_counts (diffracted, detected, wave_counts, counts + 2 * blockIdx.x);
   clock.finish (a.sums, 4);
}

// The launch's report, by one block: the counts of b2 blocks of k_mirror and
// b3 of k_diffract summed, the clocks (cleared for the next launch) and the
// exposure cut.
__global__ __launch_bounds__ (kBlock)
void k_report (TraceArgs a, const uint32_t *__restrict__ n_mid, const uint32_t *__restrict__ counts2, uint32_t b2,
               const uint32_t *__restrict__ n_ordered, const uint32_t *__restrict__ counts3, uint32_t b3)
{
   __shared__ uint32_t sum[4];
   if (threadIdx.x < 4) sum[threadIdx.x] = 0;
   __syncthreads ();
   uint32_t c[4] = {0, 0, 0, 0};
   for (uint32_t b = threadIdx.x; b < b2; b += kBlock)
     {
        c[0] += counts2[2 * b];
        c[1] += counts2[2 * b + 1];
     }
   for (uint32_t b = threadIdx.x; b < b3; b += kBlock)
     {
        c[2] += counts3[2 * b];
        c[3] += counts3[2 * b + 1];
     }
   for (int k = 0; k < 4; k++)
     {
        for (int off = 32; off > 0; off >>= 1) c[k] += __shfl_xor (c[k], off);
        if ((threadIdx.x & 63u) == 0) atomicAdd (&sum[k], c[k]);
     }
   __syncthreads ();
   if (threadIdx.x != 0) return;
   TraceReport *t = a.sums, *r = a.report;
   const uint32_t first = a.first_over ? *a.first_over : 0xFFFFFFFFu;
   r->first_over = first;
   r->in[0] = (first < a.n) ? first + 1 : a.n;
   r->in[1] = *n_mid;
   r->in[2] = sum[0];
   r->in[3] = b3 ? *n_ordered : 0u;
   r->in[4] = b3 ? sum[2] : sum[0];
   r->in[5] = b3 ? sum[3] : sum[1];
   for (int k = 0; k < 6; k++)
     {
        r->busy[k] = t->busy[k];
        t->busy[k] = 0;
     }
   r->scan = t->scan;
   r->create = t->create;
   r->mirror = t->mirror;
   r->diffract = t->diffract;
   r->end = wall_clock64 ();
}

template <bool LETG>
static void (*diffract_kernel (int kind)) (TraceArgs, const uint32_t *, const uint32_t *, Relay, uint32_t *)
{
   switch (kind)
     {
      case MXG_DET_ACIS: return k_diffract<LETG, MXG_DET_ACIS>;
      case MXG_DET_HRC_S: return k_diffract<LETG, MXG_DET_HRC_S>;
      case MXG_DET_HRC_I: return k_diffract<LETG, MXG_DET_HRC_I>;
      default: return k_diffract<LETG, -1>;
     }
}

hipError_t launch_passes (const TraceArgs &a, const mxg_config *hcfg, const PassLists &l, hipStream_t st)
{
   const bool batch = a.off != nullptr, point = hcfg->src.type == MXG_SOURCE_POINT;
   const bool grating = hcfg->grating.type > 0, letg = hcfg->grating.type == MARX_GRATING_LETG;
   const int kind = (hcfg->det.type > 0) ? detector_kind (*hcfg) : -1;
   // the order draw after the mirror searches its tables in the arenas: with
   // them in LDS too a CU would hold two blocks of that kernel, not four
   const size_t lds2 = (size_t) a.mirror.n16 * 16, lds3 = (size_t) a.grating.n16 * 16;
   void (*create) (TraceArgs, ListIO, uint32_t)
     = batch ? (point ? k_create<true, true> : k_create<false, true>)
             : (point ? k_create<true, false> : k_create<false, false>);
   ListIO io = l.create;
   hipLaunchKernelGGL (create, dim3 (io.grid), dim3 (kBlock), 0, st, a, io, hrma_tilted (hcfg->hrma));
   hipError_t e = launch_compact (io, st);
   if (e != hipSuccess) return e;

   void (*mirror) (TraceArgs, ListIO, Relay, uint32_t *)
     = grating ? k_mirror<true, -1>
     : (kind == MXG_DET_ACIS) ? k_mirror<false, MXG_DET_ACIS>
     : (kind == MXG_DET_HRC_S) ? k_mirror<false, MXG_DET_HRC_S>
     : (kind == MXG_DET_HRC_I) ? k_mirror<false, MXG_DET_HRC_I> : k_mirror<false, -1>;
   e = hipFuncSetAttribute ((const void *) mirror, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds2);
   if (e != hipSuccess) return e;
   io = l.mirror;
   hipLaunchKernelGGL (mirror, dim3 (io.grid), dim3 (kBlock), lds2, st, a, io, l.relay, l.counts);
   if (grating)
     {
        e = launch_compact (io, st, l.relay.pos);
        if (e != hipSuccess) return e;
        auto *diffract = letg ? diffract_kernel<true> (kind) : diffract_kernel<false> (kind);
        e = hipFuncSetAttribute ((const void *) diffract, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds3);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL (diffract, dim3 (l.diffract_grid), dim3 (kBlock), lds3, st, a, io.idx_out, io.n_out, l.relay,
                            l.counts + 2 * kMaxSegments);
     }
   hipLaunchKernelGGL (k_report, dim3 (1), dim3 (kBlock), 0, st, a, l.mirror.n_in, l.counts, l.mirror.grid, io.n_out,
                       l.counts + 2 * kMaxSegments, grating ? l.diffract_grid : 0u);
   return hipGetLastError ();
}

} // namespace mxg
