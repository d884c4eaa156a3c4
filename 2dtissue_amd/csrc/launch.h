// Host-side launchers for the kernels in kernels.hip and resident.hip (plain C++ signatures,
// callable from the C-ABI layer).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "device.h"

namespace tissue {

// Held while a graph is captured and around every use of the legacy stream (synchronous copies): the runtime
// refuses such a use while a stream of any thread is being captured, and ends the capture
inline std::mutex g_capture_mu;

// fixed-point scale of the order-parameter sums: cos and sin of the headings are summed as
// integers llrint(value * 2^40), which is exact and associative, so the sums do not depend on the
// order of the particles or on how they are grouped; each term is rounded by at most 2^-41, and
// up to 2^22 particles per replica stay inside int64
constexpr double kPhiScale = 1099511627776.0;  // 2^40

// what a system may have: particle and vertex numbers that the kernels' 32-bit byte offsets (load_at) and the
// whole-wave walk's list (kOwnerShift) can hold. Null, or what is too large
constexpr long kMaxParticlesTotal = 0x7fffffffl / 16;
constexpr long kMaxVertices = 1l << tdev::kOwnerShift;
inline const char* size_error(long particles, long vertices) {
  if (particles > kMaxParticlesTotal) return "too many particles";
  if (vertices >= kMaxVertices) return "too many UV vertices (at most 2^26 - 1)";
  return nullptr;
}

struct OrderPartial {
  long long cs, sn;  // sums of cos / sin of the new headings, fixed point (kPhiScale)
  int sgn, pad;      // sum of sign(x vy - y vx)
};

// one replica: particles [off, off + n) of the concatenated arrays
struct ReplicaDesc {
  int off, n;
  tdev::StepParams prm;
};

// one workgroup of the tiled step kernel: particles [first, first + block / lanes) of replica r
struct TileDesc {
  int r;        // replica; -1 marks an idle workgroup (padding of the XCD-balanced order)
  int first;    // first particle of the tile, counted within the replica
  int q;        // tile index within the replica
  int logical;  // the tile's order-parameter partials start at logical * partials_per_tile(block)
                // (tiles of a replica are consecutive)
  int clr_lo, clr_hi;  // the tile clears these vertices of its replica's oldest bucket set (clear_end)
};
// where the share of tile q of nq ends and the next one's begins: whole words of the occupancy mask
__host__ __device__ inline int clear_end(int nv, long q, long nq) {
  const long share = ((nv + nq - 1) / nq + 31) & ~31l, end = (q + 1) * share;
  return (int)(end < nv ? end : nv);
}

// one vertex-bucket set of all replicas: replica r owns count[r*nv ..], slot[r*nv*kSlots ..],
// the occupancy mask occ[r*occ_words(nv) ..], the counters ovf_n[r], big_n[r] and
// the entries ovf, multi and big at [off_r .. off_r + n_r). As the set a step fills, multi may be
// null: no finalize pass follows, so the step lists no bucket for sorting.
struct BucketSet {
  unsigned* occ;
  int* count;
  int* slot;
  int* ovf_n;
  int2* ovf;
  int* multi;
  int* big_n;
  int* big;
  int sorted;  // 1: readers see it after k_bucket_finalize; 0: raw (readers order each bucket)
};

// buckets of replica r (particles [off, ...)) within a set, as the step's readers see them
__device__ __forceinline__ tdev::BucketsIn replica_in(const BucketSet& s, int r, int nv, int off) {
  return {s.count + (size_t)r * nv, s.slot + (size_t)r * nv * tdev::kSlots, s.big + off, s.ovf + off, s.ovf_n + r,
          s.sorted};
}

// everything one step of the tiled kernel reads and writes besides the mesh and the buckets
struct TiledIO {
  const float4* xycs_in;  // (x, y, cos theta, sin theta)
  const float* th_in;
  const int* vid_in;
  float4* xycs_out;
  float* th_out;
  int* vid_out;
  float* vx;
  float* vy;
  float* r3x;
  float* r3y;
  float* r3z;
  int* face;
  int* nbr;
  const float* noise;       // eta of this step, [ntot] (may be null: zero noise), shifted by
  const int* noise_row0;    //   noise_row0[0] rows of noise_stride (null: no shift); lets one
  size_t noise_stride;      //   captured graph serve any first noise row
  OrderPartial* partial;    // [logical tiles][partials_per_tile] of this step
  const unsigned* halt_in;  // [R] flags raised before this step (a flagged replica passes through)
  unsigned* halt_out;       // [R] flags raised up to and including this step
  unsigned* halt_clr;       // [R] the third flag row, cleared for the next step
  int* first_bad;           // [R] first step of the run that raised a flag
  int step;                 // step index within the run
  int areas;                // waves of a workgroup that can hold particles (step_areas)
  float4* tape_fs;          // adjoint tape of this step, [ntot] (Fx, Fy, Sx, Sy); used by the TAPE variant
  int* tape_q;              // [ntot] quarter turns of the seam wrap
  int2* visit;              // [ntot] (na, vh) of StepOut: the neighbour set the step's own walk
                            //   visited (-1, 0 for a replica passed through); null: not recorded
};

// What a run's last kernel does for every replica r besides its own work: halt = the run's last flags,
// also to tail[r] and the first failing step to tail[R + r] (the run's read-back words), and for the
// next run its first step's output row cleared and no failure yet. halt null: not the last kernel.
struct RunEnd {
  const unsigned* last_row;  // [R] the run's last flag row (the persistent kernel has them at hand)
  unsigned* halt;
  int* first_bad;
  unsigned* tail;
  unsigned* next_out_row;
};

__device__ __forceinline__ void end_run(const RunEnd& e, int R, int r, unsigned flags, int first_bad) {
  e.halt[r] = flags;
  e.tail[r] = flags;
  e.tail[R + r] = (unsigned)first_bad;
  e.next_out_row[r] = 0u;
  e.first_bad[r] = 0x7fffffff;
}

struct ResidentIO {
  float4* xycs;           // batch state, read at launch start and written back at the end
  float* th;
  int* vid;
  float4* stage_xycs;     // per-step staging of the new state (same layout as the state)
  float* stage_th;
  int* stage_vid;
  float* vx;              // outputs of the launch's last step
  float* vy;
  float* r3x;
  float* r3y;
  float* r3z;
  int* face;
  int* nbr;
  const float* noise;     // eta of the launch's first step; step s at noise + s * noise_stride,
  size_t noise_stride;    // shifted by noise_row0[0] rows (null: no shift)
  const int* noise_row0;
  double* phi;            // (phi_ref, phi_polar) of replica r, run step t at phi[2 * (r * phi_stride + t)]
  int phi_stride;
  int t_base;             // run step index of the launch's first step
  const unsigned* flags_in;  // [R] flags before the launch
  unsigned* flags_out;       // [R] flags after the launch
  int* first_bad;            // [R]
  RunEnd end;
};

// largest workgroup of the tiled step kernel and of the persistent kernel (register budget of
// two waves per SIMD)
constexpr int kStepMaxBlock = 512;

// Whether the tiled step kernel stages the replica's vertex-occupancy mask in LDS: each workgroup
// loads the whole mask (one word per 32 vertices) before its first particle, which pays when the
// workgroup holds enough particles per word (measured on MI355X: 256 replicas, 64 particles per
// workgroup and 324 words, 7 % faster; 2,000 particles at 8 per workgroup, 6 % slower; 100,000
// particles at 64 per workgroup and 3,134 words, 1 % slower). Results are the same either way. Only
// such launches keep the mask up to date: for the others it would be one more memory-side atomic per
// occupied vertex (63,000 of them in a step of 100,000 particles).
constexpr int kOccWordsPerParticle = 8;
// Waves of a workgroup that can hold particles: of replicas of at most nmax particles, the first so many lanes.
// Only they have a walk area: areas for the waves past the last particle too, which end at once, kept other
// workgroups out of the CU's LDS (4,000 replicas of 30 particles in workgroups of 256 99 -> 76 us per step)
inline int step_areas(int nmax, int block, int phys) {
  return (int)((std::min<long>(nmax, block / phys) * phys + 63) / 64);
}
// LDS of one workgroup of the tiled step kernel: the waves' walk areas and the staged mask
inline size_t step_lds_bytes(int nv, int areas, int lanes, int phys, bool crowded, bool occ) {
  return (tdev::wave_area(lanes, phys, crowded) ? (size_t)areas * sizeof(tdev::WaveWalk) : 0) +
         (occ ? sizeof(unsigned) * (size_t)tdev::occ_words(nv) : 0);
}
constexpr size_t kStepMaxLds = 64 * 1024;  // what a launch may ask for without raising the limit
static_assert(kStepMaxBlock / 64 * sizeof(tdev::WaveWalk) <= kStepMaxLds, "the areas of the largest workgroup");
inline bool stage_occupancy(int nv, int block, int lanes, int phys) {
  return phys <= lanes && tdev::occ_words(nv) <= kOccWordsPerParticle * (block / phys) &&
         step_lds_bytes(nv, block / 64, lanes, phys, false, true) <= kStepMaxLds;
}
// Physical lanes per particle for sums laid out over `lanes` lanes (the results are the same for any).
// As many as the layout where the chip is full; more where it is not and a step's longest chain counts
// (MI355X, us per step): 4 -> 8 at 9,001 particles 23.0 / 18.8, 20,000 32.3 / 26.2, 30,000 in 30 replicas
// 21.4 / 21.0, but 40,000 33.5 / 37.0 and 100,000 72.6 / 78.2; 8 -> 16 at 5,000 particles 16.7 / 14.1, 8,000
// 17.9 / 14.6; 2 -> 4 for replicas sparse on a mesh too large for the occupancy mask, 64 x 2,000
// 57.4 / 55.1, but with the mask 80,000 particles 36.6 / 36.6, 250,000 85.5 / 85.5 and 525,000 159 / 164. Replicas
// of at most 64 particles keep 4 earlier, as their tiles at 8 are many and half empty: 909 replicas of 33 particles
// 25.5 / 29.6, 600 of 50 23.1 / 26.7, but 449 of 55 20.4 / 19.9.
// Fewer lanes than the layout were slower throughout (525,000 particles, 2 -> 1: 163 / 192, before the
// figures above).
inline int phys_lanes(int lanes, int ntot, int nmax, int nv, int block) {
  if (lanes == 8 && ntot <= 16384) return 16;
  if (lanes == 4 && ntot <= (nmax <= 64 ? 24576 : 32768)) return 8;
  if (lanes == 2 && ntot <= 163840 && !stage_occupancy(nv, block, 2, 2)) return 4;
  return lanes;
}
constexpr int kResidentMaxBlock = 512;  // of the persistent kernel's shapes; see kFullBlock in resident.hip

// lanes per particle for the persistent kernel when not tuned: wider groups for smaller replicas
inline int resident_default_lanes(int nmax) { return nmax <= 256 ? 8 : (nmax <= 1024 ? 4 : (nmax <= 2048 ? 2 : 1)); }

// Default launch shape of the tiled step kernel (lanes per particle, threads per workgroup) for
// R replicas of ntot particles in all, the largest of nmax, on nv vertices. Measured on MI355X: a single system
// of a few thousand particles fills few CUs, so more lanes per particle shorten its critical path, and one-wave
// workgroups let every wave start its walk without waiting for another at the staging barrier
// (2,000 particles: 32 lanes in 64 threads 10.08 us, 16 in 64 10.48 us, 16 in 128 10.54 us, 64 in 64
// 10.19 us, 8 in 64 10.83 us); beyond, workgroups of 128 leave a shorter last round than 256 (525,000
// particles in 256 replicas 34.1 -> 33.2 ms per 200 steps; 100,000 particles 68.5 -> 67.3 us per step, 64
// threads 66.6, but slower in the batch), but replicas that fit in one workgroup of 256 and not in one of 128
// take that (1,000 replicas of 100 particles 41.7 us against 45.1 in twos of 128, 1,538 of 65 54.5 against 61.8);
// a single 100,000-particle system is fastest with 4 (2 lanes 82.6 us), a large batch with 2 (autotuned).
inline void tiled_default_shape(int R, int ntot, int nmax, int nv, int* lanes, int* block) {
  const int big_lanes = R == 1 ? 4 : 2;
  *lanes = ntot <= 4096 ? 32 : (ntot <= 8192 ? 8 : (ntot <= 65536 ? 4 : big_lanes));
  *block = ntot <= 4096 ? 64 : 128;
  if (*block == 128 && R > 1 && nmax > 128 / phys_lanes(*lanes, ntot, nmax, nv, 128) &&
      nmax <= 256 / phys_lanes(*lanes, ntot, nmax, nv, 256))
    *block = 256;
}

// Replicas of a few thousand particles, at most one per two vertices, leave their vertex buckets
// raw: the finalize pass would cost a kernel boundary per step, and the readers order the few
// particles of each bucket themselves (the same visiting order, so the same results). Denser or
// larger systems pile particles onto vertices (the exit snapping), and a crowded raw bucket costs
// each reader a scan of the overflow list.
constexpr int kRawBucketsMax = 8192;
inline bool raw_buckets_for(int nmax, int nv) { return nmax <= kRawBucketsMax && 2L * nmax <= nv; }

// LDS bytes of one workgroup of the persistent kernel for a mesh with nv vertices and replicas of
// at most nmax particles; resident_max_particles is the largest nmax that fits one CU
size_t resident_lds_bytes(int nv, int nmax);
int resident_max_particles(int nv);
// allow the persistent kernels the LDS of replicas up to nmax particles (call outside capture)
hipError_t resident_prepare(int nv, int nmax);
hipError_t launch_resident(int lanes, int block, const tdev::MeshDev& mesh, const ReplicaDesc* reps, int R, int nmax,
                           int steps, const ResidentIO& io, hipStream_t st);

// one step of every replica: n_tiles workgroups of `block` threads, `phys` lanes per particle, its
// sums laid out over `lanes` lanes (phys: phys_lanes);
// reads bucket set bin, writes bout, clears bclr; tape selects the variant that records the
// adjoint tape; wave the seam-wrap loop of crowded systems (same results, see seam_wrap_group)
hipError_t launch_step_tiled(int lanes, int phys, int block, bool tape, bool wave, const tdev::MeshDev& mesh, const ReplicaDesc* reps,
                             const TileDesc* tiles, int n_tiles, const BucketSet& bin, const BucketSet& bout,
                             const BucketSet& bclr, const TiledIO& io, hipStream_t st);
// sort the buckets of set bs that hold two or more particles (over the same tiles as the step);
// crowded buckets (more than kSlots) move, sorted, into the big area. single_n: the particle
// count when there is one replica (its tiles are then not read), else 0
hipError_t launch_bucket_finalize(int block, const ReplicaDesc* reps, const TileDesc* tiles, int n_tiles, int nv,
                                  int single_n, const BucketSet& bs, hipStream_t st);
// order parameters of `steps` steps of every replica from the step kernel's partials, one per
// wave: per_tile = waves per workgroup, partial[(s * n_logical + tile) * per_tile + wave];
// replica r's tiles are tile_begin[r] .. tile_begin[r+1]
hipError_t launch_phi_tiles(int R, int steps, const int* tile_begin, int n_logical, int per_tile,
                            const OrderPartial* partial, const ReplicaDesc* reps, double* phi, int phi_stride,
                            int t_base, const RunEnd& end, hipStream_t st);
// order-parameter partials the tiled step kernel writes per tile (one per wave)
inline int partials_per_tile(int block) { return block / 64; }
// run start: rows[0] = halt, rows[1] = 0, first_bad = INT_MAX
hipError_t launch_flags_begin(int R, const unsigned* halt, unsigned* rows, int* first_bad, hipStream_t st);
// the state of n particles from x, y, theta (device or mapped host memory; x, y may be vx, vy), velocities,
// neighbour counts and the R replicas' halt flags zeroed
hipError_t launch_adopt(int n, const float* x, const float* y, const float* th, float4* xycs, float* th_out, float* vx,
                        float* vy, int* nbr, int R, unsigned* halt, hipStream_t st);
// particles [first, first + n) as consecutive arrays at out (mapped host memory), those that are asked for:
// array k (x, y, theta, vid) at out + at[k] n unless at[k] < 0
struct PackAt { int at[5]; };
hipError_t launch_pack_state(int first, int n, const float4* xycs, const float* th, const int* vid, const PackAt& where,
                             float* out, hipStream_t st);
// the same of vx, vy, r3d ([n][3], so three words of n), face, nbr
hipError_t launch_pack_outputs(int first, int n, const float* vx, const float* vy, const float* r3x, const float* r3y,
                               const float* r3z, const int* face, const int* nbr, const PackAt& where, float* out,
                               hipStream_t st);
// n words of mapped host memory into device memory
hipError_t launch_fetch(size_t n, const float* from, float* to, hipStream_t st);
// counts, masks and list lengths of n_sets (1 to 3) bucket sets of R replicas zeroed
hipError_t launch_clear_sets(int R, int nv, const BucketSet* sets, int n_sets, hipStream_t st);
hipError_t launch_locate(const tdev::MeshDev& mesh, int n, const float4* xycs, int* vid, int* face, float* r3x,
                         float* r3y, float* r3z, hipStream_t st);
// copy step t's outputs into the per-step output ring (when its global step number, ctl[1] + t + 1,
// is a multiple of every): ring [depth][5][ntot] = x, y, X, Y, Z; ring_nbr [depth][ntot]
hipError_t launch_record(int ntot, const int* ctl, int t, int every, int depth, const float4* xycs, const float* r3x,
                         const float* r3y, const float* r3z, const int* nbr, float* ring, int* ring_nbr, hipStream_t st);
// area-uniform initial positions and headings of every replica (replica r from seeds[r])
hipError_t launch_init_random(int ntot, const int* rid, const ReplicaDesc* reps, const uint64_t* seeds,
                              const double* cdf, const tdev::MeshDev& mesh, float* x, float* y, float* th, hipStream_t st);
// seam wrap of n moves start -> end (end overwritten), lanes = 1, 2, 4, 8, 16, 32 or 64 per move;
// wave: a wave's last flight is finished by all of its lanes (seam_wrap_group)
hipError_t launch_seam_wrap(int lanes, int n, const double2* start, double2* end, double* dtheta, int* quarter, int* ok,
                            int max_crossings, int wave, hipStream_t st);
// clears a bucket set that holds the state with vertex ids vid where that state is
hipError_t launch_clear_held(int ntot, const int* vid, const int* rid, int R, int nv, const BucketSet& bs, hipStream_t st);
// bucket every particle of every replica (rid[g] = replica of particle g) into set `bs`
hipError_t launch_insert(int ntot, const int* vid, const int* rid, const ReplicaDesc* reps, int nv,
                         const BucketSet& bs, hipStream_t st);
// neighbour sets {j : d_ij < 2 sigma} of the current state (ids counted within the replica)
hipError_t launch_neighbor_lists(const tdev::MeshDev& mesh, const ReplicaDesc* reps, const int* rid, int ntot,
                                 const BucketSet& bs, const int* vid, int cap, int* counts, int* cols,
                                 hipStream_t st);

}  // namespace tissue
