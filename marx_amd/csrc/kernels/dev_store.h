// dev_store.h -- the structure-of-arrays photon store in HBM and the launch
// helpers shared by the stage kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "marx_gpu.h"
#include "marx_gpu_cfg.h"
#include "dev_math.h"

namespace mxg {

// Column pointers of the resident photon store (one element per photon).
struct Soa
{
   double *energy;
   double *x0, *x1, *x2;
   double *p0, *p1, *p2;
   double *t;
   uint32_t *flags;
   float *ypix, *zpix, *upix, *vpix;
   float *dith[6];
   float *pi;
   int16_t *pha;
   uint8_t *shell;
   int8_t *ccd, *region, *order;
   int8_t *sup[4];
   uint32_t *tag;
};

// The stages' search tables as the host lays them out for LDS (hrma_image,
// grating_image), in HBM: 16-byte words at img, n16 of them.
struct LdsImage
{
   const uint4 *img;
   uint32_t n16;
};

// Copies n16 16-byte words of a host-made LDS image into LDS.  Every thread
// has several loads in flight: the staging is one round of memory latency,
// where copying table by table it was a dozen.
__device__ __forceinline__ void stage_image (const uint4 *__restrict__ img, uint32_t n16, unsigned char *lds)
{
   uint4 *dst = (uint4 *) lds;
#pragma unroll 4
   for (uint32_t w = threadIdx.x; w < n16; w += blockDim.x) dst[w] = img[w];
}

// Per-stage launch arguments: the active index list in, the survivors out.
//
// Survivors are collected without global atomics: block b of a stage kernel
// (grid = `grid` blocks of kBlock lanes) owns the input positions
// [lo_b, hi_b) of block_range() and writes the ids of its survivors, in input
// order, to seg[lo_b ...] and their number to seg_count[b].  k_compact then
// concatenates the segments into idx_out / n_out.  An input list sorted by id
// therefore yields an output list sorted by id.
struct ListIO
{
   const uint32_t *idx_in;
   const uint32_t *n_in;
   uint32_t *idx_out;      // compacted survivors (written by k_compact)
   uint32_t *n_out;
   uint32_t *seg;          // per-block survivor segments, capacity entries
   uint32_t *seg_count;    // grid entries
   uint32_t grid;          // blocks of the stage kernel (<= kMaxSegments)
   uint32_t *n_copy = nullptr;  // when non-null, k_compact also writes the length here
};

constexpr int kBlock = 256;
constexpr uint32_t kMaxSegments = 8192;

// A kernel's survivors handed densely to the next one: the columns the
// grating and the detector read of a photon (x, p, energy, tag, flags,
// shell), written by the producing kernel at the survivor's segment slot (its
// position in seg), and pos, written by k_compact: the slot of each entry of
// the compacted list.  k_mirror hands the photons with an order to k_diffract
// this way, and in traces and batches with a FEF file the reflection its
// survivors to an LETG and either grating its own to the detector.  After the
// mirror about one photon id in three is alive, after the grating one in
// sixteen, so reading the double columns at the ids costs a cache line per
// column for a few photons; the relay's rows are contiguous.
struct Relay
{
   double *x0, *x1, *x2, *p0, *p1, *p2, *energy;
   uint32_t *tag, *flags;
   uint8_t *shell;
   uint32_t *pos;
};

// A photon leaving a stage: the columns of its relay row.
struct PhotonOut
{
   double x0, x1, x2, p0, p1, p2, energy;
   uint32_t tag, flags;
   int shell;
};

// Entry i of a column.  Columns are at most 2^32 bytes, so the byte offset is
// formed in 32 bits and added to the column's address, a scalar, by the memory
// instruction itself.  (Created chunks and batches hold at most 2^28 photons; a
// host list as many as the store takes, whose capacity is a power of two and
// at 292 bytes a photon, with its lists and relays, ends at 2^29 on a card of
// 288 GB.)
template <class T>
__device__ __forceinline__ T &at (T *col, uint32_t i)
{
   return *(T *) ((char *) col + (uint32_t) (i * (uint32_t) sizeof (T)));
}

// a column entry that the kernel writes and no kernel reads soon
template <class T>
__device__ __forceinline__ void put_once (T *p, T v)
{
   __builtin_nontemporal_store (v, p);
}

// the path columns of photon id
__device__ __forceinline__ void store_path (const Soa &s, uint32_t id, vec3 x, vec3 p, uint32_t flags)
{
   at (s.x0, id) = x.x; at (s.x1, id) = x.y; at (s.x2, id) = x.z;
   at (s.p0, id) = p.x; at (s.p1, id) = p.y; at (s.p2, id) = p.z;
   at (s.flags, id) = flags;
}

// Chunks of more photons than this store their paths past the caches in the
// kernels whose waves fill nearly every line: the columns of so many (126
// bytes a photon) do not stay in the 256 MB cache until they are read, and
// keeping them costs its bandwidth.  MI355X, trace of n photons with the
// paths kept and past it: ACIS-S n = 1e6 149 and 151 us, 3e6 318 and 337,
// 4e6 464 and 419, 6e6 714 and 590; HETG + ACIS-S 2e6 253 and 264, 3e6 379
// and 366, 6e6 780 and 651.
constexpr uint32_t kCachedPhotons = 3u << 20;

// store_path in a chunk of n photons
__device__ __forceinline__ void chunk_path (const Soa &s, uint32_t n, uint32_t id, vec3 x, vec3 p, uint32_t flags)
{
   if (n <= kCachedPhotons) store_path (s, id, x, p, flags);
   else
     {
        // (the compiler would make one of the two alternatives, the first)
        asm volatile ("; past the caches");
        put_once (&at (s.x0, id), x.x); put_once (&at (s.x1, id), x.y); put_once (&at (s.x2, id), x.z);
        put_once (&at (s.p0, id), p.x); put_once (&at (s.p1, id), p.y); put_once (&at (s.p2, id), p.z);
        put_once (&at (s.flags, id), flags);
        asm volatile ("; to here");
     }
}

// a survivor's row of a relay
__device__ __forceinline__ void relay_put (const Relay &r, uint32_t q, const PhotonOut &o)
{
   at (r.x0, q) = o.x0; at (r.x1, q) = o.x1; at (r.x2, q) = o.x2;
   at (r.p0, q) = o.p0; at (r.p1, q) = o.p1; at (r.p2, q) = o.p2;
   at (r.energy, q) = o.energy;
   at (r.tag, q) = o.tag;
   at (r.flags, q) = o.flags;
   at (r.shell, q) = (uint8_t) o.shell;
}


// A kernel's first argument, read again from its argument segment.  A loop
// that uses some thirty columns loads their addresses where it needs them;
// the compiler would otherwise load them all before the loop, more than the
// scalar registers hold, and keep the rest in lanes of vector registers, an
// instruction and a wait for each use.
template <class T>
__device__ __forceinline__ T kernel_args ()
{
   typedef const __attribute__ ((address_space (4))) T *Segment;
   Segment p = (Segment) __builtin_amdgcn_kernarg_segment_ptr ();
   asm volatile ("" : "+s" (p));
   return *(const T *) p;
}

struct BlockRange { uint32_t lo, hi; };

// The input positions owned by block b of nblocks: equal chunks rounded up
// to whole blocks of lanes.
__device__ __forceinline__ BlockRange block_range (uint32_t n, uint32_t b, uint32_t nblocks)
{
   uint64_t per = ((uint64_t) n + nblocks - 1) / nblocks;
   uint64_t chunk = (per + kBlock - 1) / kBlock * kBlock;
   uint64_t lo = (uint64_t) b * chunk;
   uint64_t hi = lo + chunk;
   BlockRange r;
   r.lo = (uint32_t) (lo < n ? lo : n);
   r.hi = (uint32_t) (hi < n ? hi : n);
   return r;
}

// Order-preserving survivor output of one block (see ListIO).  add() is
// called by every lane of the block once per pass of kBlock inputs; it
// holds one barrier.  wc is a 2 x (kBlock / 64) LDS array.
struct SegWriter
{
   uint32_t *out;
   uint32_t *wc;
   uint32_t lo;
   uint32_t count;
   uint32_t parity;

   __device__ __forceinline__ SegWriter (const ListIO &io, const BlockRange &r, uint32_t *lds_wc)
      : out (io.seg + r.lo), wc (lds_wc), lo (r.lo), count (0), parity (0) {}

   // returns the slot (position in seg) of a kept id
   __device__ __forceinline__ uint32_t add (bool keep, uint32_t id)
   {
      constexpr int kWaves = kBlock / 64;
      unsigned long long mask = __ballot (keep);
      const int wave = threadIdx.x >> 6, lane = __lane_id ();
      uint32_t *w = wc + parity * kWaves;
      if (lane == 0) w[wave] = (uint32_t) __popcll (mask);
      __syncthreads ();
      uint32_t before = 0, total = 0;
#pragma unroll
      for (int k = 0; k < kWaves; k++)
        {
           uint32_t c = w[k];
           before += (k < wave) ? c : 0u;
           total += c;
        }
      const uint32_t q = count + before + (uint32_t) __popcll (mask & ((1ull << lane) - 1ull));
      if (keep) out[q] = id;
      count += total;
      parity ^= 1u;
      return lo + q;
   }

   __device__ __forceinline__ void finish (const ListIO &io)
   {
      if (threadIdx.x == 0) io.seg_count[blockIdx.x] = count;
   }
};

// Launches k_compact over the segments a stage kernel of io.grid blocks
// wrote; pos_out, when non-null, receives the slot of each list entry.
hipError_t launch_compact (const ListIO &io, hipStream_t st, uint32_t *pos_out = nullptr);

// Output files (output.hip): the photons not flagged bad, in order, then the
// requested columns of them packed big-endian, column k at out + offset[k].
constexpr int kMaxPackCols = 32;
struct PackArgs
{
   int32_t ncols;
   int32_t col[kMaxPackCols];
   uint64_t offset[kMaxPackCols];
   double total_time;
};
hipError_t launch_keep_list (const uint32_t *flags, uint32_t n, const ListIO &io, hipStream_t st);

// Event coordinates (events.hip): row q of each column for photon idx[q].
struct EventOut
{
   uint32_t *tag;
   int32_t *ccd, *tdetx, *tdety;
   double *detx, *dety, *x, *y;
   int16_t *fltgrade;
};
// The frame heads (first row of each row's frame, for the held dither
// state) take head[m], chunk_max[ceil(m / kBlock)] and chunk_pre[same].
hipError_t launch_event_coords (const mxg_config *cfg, const mxg_event_params *params, const float *subtab,
                                const Soa &s, const uint32_t *idx, uint32_t m, double total_time, double time_del,
                                unsigned long long seed, uint32_t *head, uint32_t *chunk_max, uint32_t *chunk_pre,
                                const EventOut &out, hipStream_t st);
hipError_t launch_pack_columns (const Soa &s, const uint32_t *idx, const uint32_t *n_kept, uint32_t m,
                                const PackArgs &a, uint8_t *out, hipStream_t st);

// Minimum waves per SIMD of the mirror's reflection kernel unless the
// launch schedule says otherwise (256 lanes per block = one wave per SIMD
// per block).  At 109 to 113 VGPRs, without spills, it holds four waves
// whichever instance is launched; the instances differ in scheduling only.
#define MXG_REFLECT_WAVES_DEFAULT 4
// waves per SIMD that the compiler must leave room for (0: unbounded).
// The source kernels (50 to 70 VGPRs), the grating passes (75 to 89) and the
// ACIS detector (94) need fewer than the 128 of four waves without
// being told.
#ifndef MXG_SOURCE_WAVES
#define MXG_SOURCE_WAVES 4
#endif
#ifndef MXG_BATCH_SOURCE_WAVES
#define MXG_BATCH_SOURCE_WAVES 4
#endif
// waves of the reflection kernel of the schedule's largest setting, and of
// the aperture kernel (unbounded, 52 VGPRs)
#ifndef MXG_REFLECT_WAVES_TOP
#define MXG_REFLECT_WAVES_TOP 4
#endif
#ifndef MXG_ENTER_WAVES
#define MXG_ENTER_WAVES 0
#endif
#ifndef MXG_LETG_GRATING_WAVES
#define MXG_LETG_GRATING_WAVES 4
#endif
#ifndef MXG_GRATING_WAVES
#define MXG_GRATING_WAVES 3
#endif
#ifndef MXG_DETECT_WAVES
#define MXG_DETECT_WAVES 0
#endif
// the ACIS instance of the detector kernel (without FEF): waves per SIMD
#ifndef MXG_ACIS_DETECT_WAVES
#define MXG_ACIS_DETECT_WAVES 0
#endif

// Device buffers and launch shape of the mirror stage's second kernel.
struct HrmaScratch
{
   uint32_t *idx_mid;      // photons that hit the paraboloid (capacity entries)
   uint32_t *n_mid;        // its length (written by k_compact)
   uint32_t *rng_pos;      // per photon: random-stream word at the split
   uint32_t reflect_grid;  // blocks of k_hrma_reflect
   int reflect_waves;      // 2, 3 or 4: the instance of k_hrma_reflect launched
   LdsImage image;         // the mirror's tables
   uint32_t *n_mid_copy = nullptr;  // when non-null, also receives the middle list's length
};

// Stage launchers (defined in the stage .hip files).
// cfg: device copy; hcfg: host copy of the same configuration (launch
// geometry and LDS layout are computed from it).  ev, when non-null, holds
// four events recorded around k_hrma_enter (0, 1) and k_hrma_reflect (2, 3).
// relay_out, when non-null: the mirror's survivors go to it for the grating,
// which stores their x, p and flags (the reflection kernel stores those of
// the photons it drops only)
// fresh: the input photons come straight from launch_source with
// entry_follows (unread flags, all zero; the entry writes every photon's
// position, shell and flags)
hipError_t launch_hrma (const mxg_config *cfg, const mxg_config *hcfg, const float *fa,
                        const double *da, Soa s, ListIO io, HrmaScratch hs, uint32_t n_upper,
                        double source_distance, unsigned long long seed, uint32_t source_id,
                        const Relay *relay_out, bool fresh, hipStream_t st, hipEvent_t *ev);
// k_hrma_reflect alone, from io.idx_in (photons that hit the paraboloid,
// stream positions in rng_pos) to io's survivor segments (io.grid blocks;
// the caller compacts them); waves: the instance launched (2, 3 or 4)
hipError_t launch_hrma_reflect (const mxg_config *cfg, const mxg_config *hcfg, const float *fa,
                                const double *da, Soa s, ListIO io, const uint32_t *rng_pos, LdsImage image, int waves,
                                unsigned long long seed, uint32_t source_id, const Relay *relay_out,
                                hipStream_t st);
// The blocks of k_grating that one CU holds at once for configuration hcfg
// (its waves per SIMD, fewer if its LDS tables do not fit that many), 8 if
// the runtime cannot say.  A grid of whole rounds of them measured fastest
// (HETG + ACIS-S: 3 blocks per CU 0.36 ms, 4 0.47 ms, 8 0.40 ms).
uint32_t grating_blocks_per_cu (const mxg_config *hcfg);
// hcfg: the host copy of cfg; image: the tables the kernel stages in LDS;
// letg: the instance compiled for the LETG pass; relay_in, when non-null (with
// letg and relay_out only): the input list is the mirror's with this relay,
// whose rows the kernel reads instead of the store's; relay_out, when
// non-null (without letg or with relay_in): the survivors go to it for
// launch_detect, which stores their x, p and flags (the kernel stores those
// of the photons it drops only)
hipError_t launch_grating (const mxg_config *cfg, const mxg_config *hcfg, const float *fa, const double *da, Soa s,
                           ListIO io, LdsImage image, uint32_t n_upper, unsigned long long seed,
                           uint32_t source_id, bool letg, const Relay *relay_in, const Relay *relay_out,
                           hipStream_t st);
// fef: run the variant with the ACIS FEF step (the configuration read a FEF
// file); kind: the detector family (detector_kind of the configuration)
enum { MXG_DET_ACIS = 0, MXG_DET_HRC_S = 1, MXG_DET_HRC_I = 2 };
inline int detector_kind (const mxg_config &c)
{
   return (c.det.type == MARX_DETECTOR_HRC_S) ? MXG_DET_HRC_S
     : (c.det.type == MARX_DETECTOR_HRC_I) ? MXG_DET_HRC_I : MXG_DET_ACIS;
}
// relay, when non-null (ACIS with the FEF step only): the input list is the
// one the grating left with this relay, whose rows the kernel reads instead
// of the store's
hipError_t launch_detect (const mxg_config *cfg, const float *fa, const double *da, Soa s,
                          ListIO io, uint32_t n_upper, double tstart,
                          unsigned long long seed, uint32_t source_id, bool fef, int kind,
                          const Relay *relay, hipStream_t st);

hipError_t launch_dither_store (const mxg_config *cfg, Soa s, uint32_t n, double start_time,
                                unsigned long long seed, hipStream_t st);
// Photon creation (source.hip): photons 0..n-1 of the store from tag
// tag_start, the exposure cut in *first_over, the active list idx and its
// length *count (and *count_copy when non-null); ticks (n entries) and
// tile_tot (ceil(n / 2048) entries) are scratch; point: the configured
// shape is a point (the instance without the extended shapes);
// entry_follows: launch_hrma with fresh set follows on the created photons
// (the source leaves their position, shell and flags to it).
hipError_t launch_source (const mxg_config *cfg, const float *fa, const double *da, Soa s, uint32_t n,
                          uint32_t tag_start, double exposure_time, double start_time,
                          unsigned long long seed, uint32_t source_id, uint64_t *ticks, uint64_t *tile_tot,
                          uint32_t *first_over, uint32_t *count, uint32_t *count_copy, uint32_t *idx, bool point,
                          bool entry_follows, hipStream_t st);

// The arrival-time scan alone (launch_source's first pass, n > 0): ticks and
// tile_tot filled, *first_over set to 0xFFFFFFFF, and the wall clock at its
// start in *begin when non-null; *tile_off: the tiles' offsets for
// source_photon (null for a single tile, whose offset is 0).
hipError_t launch_source_scan (const mxg_config *cfg, const float *fa, const double *da, uint32_t n,
                               uint32_t tag_start, unsigned long long seed, uint32_t source_id, uint64_t *ticks,
                               uint64_t *tile_tot, uint32_t *first_over, uint64_t *begin, bool point,
                               const uint64_t **tile_off, hipStream_t st);

// Batched point sources (see source.hip): n photons over nsrc sources with
// prefix offsets off[nsrc + 1] and unit directions dir[3 nsrc]; point: the
// configured shape is a point (the instance without the extended shapes);
// entry_follows: launch_hrma with fresh set follows (as for launch_source).
hipError_t launch_batch_source (const mxg_config *cfg, const double *da, Soa s, uint32_t n,
                                const uint32_t *off, uint32_t nsrc, const double *dir,
                                const uint32_t *tag_start, double exposure, double start_time,
                                unsigned long long seed, uint32_t *idx, uint32_t *count,
                                uint32_t grid, bool point, bool entry_follows,
                                hipStream_t st);

// largest persistent tile that a schedule may name
constexpr uint32_t kMaxPersistTile = 4096;

// The differentiable mirror (diff.hip).
struct DiffOut
{
   // a row for each photon that reached the paraboloid, in the list's order
   double *w, *y, *z;           // n values each, of which the rows
   double *dw, *dy, *dz;        // MXG_DIFF_NPAR x n derivatives each
   uint8_t *row_shell;
   uint8_t *shell;              // by photon
   double *block_w;             // per-block summed weight
};
hipError_t launch_diff_forward (const mxg_config *cfg, const float *fa, const double *da,
                                const mxg_diff_cfg *dcfg, uint32_t n, uint32_t tag_start,
                                unsigned long long seed, const mxg_image_spec *spec, float *image,
                                float *win_partial, float *slice_sum, DiffOut out, const ListIO &enter,
                                uint32_t grid, double *wsum_dev, int tangents, hipStream_t st,
                                hipEvent_t *ev);
hipError_t launch_diff_adjoint (uint32_t n, const uint32_t *n_rows, DiffOut in, int tangents, const mxg_image_spec *spec, const float *g,
                                double *partial, uint32_t grid, double *grad_dev, hipStream_t st,
                                hipEvent_t *ev);

// The energy order of the store's first n photons (sort.hip): stable
// radix sort of (energy, index) pairs.  With tmp == nullptr only
// *tmp_bytes (rocPRIM's temporary storage) is set.
hipError_t sort_energies (const double *energy, uint32_t n, double *keys_in, uint32_t *vals_in,
                          double *keys_out, uint32_t *vals_out, void *tmp, size_t *tmp_bytes,
                          hipStream_t st);
// out[i] = energy[idx[i]] for i < *n_dev (n_upper an upper bound of *n_dev)
hipError_t gather_energies (const double *energy, const uint32_t *idx, const uint32_t *n_dev, uint32_t n_upper,
                            double *out, hipStream_t st);

} // namespace mxg
