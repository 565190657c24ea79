// passes.h -- the device-created trace as kernels over the whole chunk
// (passes.hip).
#pragma once

#include "dev_store.h"

namespace mxg {

// What a launch leaves for the host, in pinned memory, and the device's own
// running sums and clocks (cleared again when they are reported).
struct TraceReport
{
   uint32_t in[6];              // photons created, into the reflection, out of the mirror, with an order,
                                // into the detector, detected
   uint32_t first_over;         // first photon at or past the exposure (0xFFFFFFFF: none)
   uint32_t pad;
   uint64_t busy[6];            // sampled cycles in source, entry; reflection, what follows it in the
                                // same kernel; diffraction, detector
   uint64_t scan;               // wall clock at the start of the arrival-time scan,
   uint64_t create, mirror, diffract;   // of the kernels,
   uint64_t end;                // and at the end
};

struct TraceArgs
{
   const mxg_config *cfg;
   const float *fa;
   const double *da;
   Soa s;
   uint32_t n;                  // photons created
   uint32_t *n_dev;             // ... for the kernels that read list lengths from HBM (written by k_create)
   unsigned long long seed;
   double exposure, start_time, tstart;
   uint32_t *rng_pos;
   // one source: its first tag, and for Poisson arrivals the scanned gaps
   // (tile_off null: of a single tile)
   uint32_t tag_start;
   const uint64_t *ticks, *tile_off;
   uint32_t *first_over;
   // a batch of sources (off non-null): n photons over nsrc sources
   const uint32_t *off;
   uint32_t nsrc;
   const double *dir;
   const uint32_t *batch_tag;
   LdsImage mirror, grating;    // the tables staged in LDS
   TraceReport *sums, *report;  // device sums, pinned report
};

// Lists and scratch.
struct PassLists
{
   ListIO create, mirror;       // create's output list is mirror's input
   Relay relay;                 // rows for k_diffract
   uint32_t *counts;            // 4 * kMaxSegments block counts
   uint32_t diffract_grid;
};
hipError_t launch_passes (const TraceArgs &a, const mxg_config *hcfg, const PassLists &l, hipStream_t st);

} // namespace mxg
