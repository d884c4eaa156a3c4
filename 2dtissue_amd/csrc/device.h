// Device-side building blocks of the per-step update (gfx950, wave64). Shared by the per-step
// kernel, the batched persistent kernel and the adjoint.
//
// Precision plan: state and pair arithmetic in FP32; the decisive or ill-conditioned parts in
// FP64 (seam-wrap geometry, point location, nearest vertex, order-parameter sign, and the
// alignment mean when the neighbour sum nearly cancels). All code is compiled with
// -ffp-contract=off, so every expression rounds as written. Point location ranks candidate faces
// in FP32 and falls back to FP64 (the host oracle's operation order, so the same decisions)
// whenever the FP32 ranking or the nearest-vertex choice is within its error margin.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "geom.h"

namespace tdev {

constexpr int kSlots = 8;                       // particles held per vertex bucket before overflow
constexpr float kPiF = 3.14159274f;             // pi rounded to float
constexpr float kTwoPiF = 6.28318548f;

// per-simulation constants (FP32 values of the FP64 parameters; thresholds reproduce the FP64
// comparisons d < 2 sigma and d <= 2.4 sigma exactly for FP32 d)
struct StepParams {
  float t_near;    // largest float f with (double)f < 2 sigma
  float t_count;   // largest float f with (double)f <= 2.4 sigma
  float two_sigma, k, v0, mu, dt, rate;  // rate = dt / tau
  int32_t max_crossings, pad;
  double two_sigma64, k64, v064, mu64, dt64, rate64;  // the same parameters for the FP64 paths
  double kc64;  // k64 / two_sigma64: Fij / d = kc (d - 2 sigma) / d, to a few ulps
};

// displacement (UV units) above which the force, speed and Euler update are redone in FP64:
// an FP32 speed carries ~1e-7 relative error, which a displacement D turns into ~1e-7 D absolute
constexpr float kBigStep = 2.0f;

// Vertex buckets of one step: count[v] particles. Sorted (after k_bucket_finalize): up to kSlots
// of them in slot[v*kSlots ..] in ascending id order; a bucket with more holds its ids, ascending,
// in big[slot[v*kSlots] ..] instead. Raw (no finalize pass): the first kSlots arrivals in
// slot[v*kSlots ..] in arrival order, later ones in the (vertex, id) overflow list ovf[0 .. *ovf_n);
// readers order them themselves. Either way a bucket is visited in ascending id order.
struct BucketsIn {
  const int* count;
  const int* slot;
  const int* big;
  const int2* ovf;
  const int* ovf_n;
  int sorted;
};
// The same buckets while the step fills them: the first kSlots arrivals of a vertex take its
// slots, later ones go to the (vertex, id) overflow list; the second arrival at a vertex also
// leaves the vertex in its particle's entry of multi (the buckets the finalize pass must sort, -1 in
// the entries of the other particles; null when no finalize pass
// follows); where the step's kernels read the occupancy mask occ, the first arrival sets the vertex's
// bit in it (bit v % 32 of word v / 32).
struct BucketsOut { int* count; int* slot; int* ovf_n; int2* ovf; int* multi; unsigned* occ; };

// words of a vertex-occupancy mask over nv vertices
__host__ __device__ constexpr int occ_words(int nv) { return (nv + 31) >> 5; }

// base[i] for a uniform base and 0 <= i * sizeof(T) < 2^32: the address is the scalar base plus a
// 32-bit lane offset, two or three instructions fewer than a 64-bit one (arrays by particle or by vertex
// of one replica, below 4 GiB each: 2^27 particles, 2^26 vertices; the geodesic table may be larger and
// goes through table_entry)
template <class T>
__device__ __forceinline__ T load_at(const T* base, int i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (uint32_t)i * (uint32_t)sizeof(T));
}

// ------------------------------------------------------------------ neighbour traversal

// visit the particles of bucket w in ascending id order (fixed order => reproducible sums)
template <class B, class F>
__device__ __forceinline__ void for_bucket(const B& b, int w, F&& f) {
  const int c = b.count[w];
  if (c == 0) return;
  const int* s = b.slot + (size_t)w * kSlots;
  if (b.sorted) {
    if (c <= kSlots) {
      for (int q = 0; q < c; ++q) f(s[q]);
      return;
    }
    const int* g = b.big + s[0];
    for (int q = 0; q < c; ++q) f(g[q]);
    return;
  }
  if (c <= kSlots) {  // raw: the slots in registers, sorted by the network (8 slots are in bounds)
    const int4 s0 = reinterpret_cast<const int4*>(s)[0], s1 = reinterpret_cast<const int4*>(s)[1];
    int a[kSlots] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int q = 0; q < kSlots; ++q) a[q] = q < c ? a[q] : 0x7fffffff;
    sort8(a);
    for (int q = 0; q < c; ++q) f(a[q]);
    return;
  }
  // raw and crowded (rare for the systems that skip the finalize pass): the next id each time is
  // the least one above the previous among the slots and the bucket's overflow entries
  const int n_ovf = *b.ovf_n;
  int prev = -1;
  for (int k = 0; k < c; ++k) {
    int best = 0x7fffffff;
    for (int q = 0; q < kSlots; ++q) {
      const int id = s[q];
      best = (id > prev && id < best) ? id : best;
    }
    for (int o = 0; o < n_ovf; ++o) {
      const int2 e = b.ovf[o];
      best = (e.x == w && e.y > prev && e.y < best) ? e.y : best;
    }
    f(best);
    prev = best;
  }
}

// force coefficient Fij / d for a pair at table distance d < 2 sigma
// (ForceHelper.cpp:55-70, 84-104: d == 0 becomes 0.001; the adhesion branch is unreachable)
__device__ __forceinline__ float pair_coef(float d, const StepParams& p) {
  const float dd = (d == 0.0f) ? 0.001f : d;
  const float fij = (-p.k * (p.two_sigma - dd)) / p.two_sigma;
  return fij / dd;
}

// sum over the group, in the order of a butterfly from LANES / 2 down; every lane gets it
template <int LANES, int OFF = LANES / 2, class T>
__device__ __forceinline__ T group_sum(T v) {
  if constexpr (OFF >= 1) {
    T a, b;
    butterfly<OFF, LANES>(v, a, b);
    return group_sum<LANES, OFF / 2>(a + b);
  } else {
    return v;
  }
}

constexpr unsigned kFlagLost = 1u, kFlagNonfinite = 2u, kFlagTiling = 4u;

// result of one particle's step
struct StepOut {
  float xo, yo, to, co, so;  // new position, heading and its cos / sin
  float vx, vy;              // r_dot (unrotated, as the reference outputs it)
  Located L;                 // remap of (xo, yo)
  int nb;                    // neighbour count
  unsigned fl;               // validation flags
  int sgn;                   // sign of x vy - y vx (order parameter)
  // what the adjoint replays and the visit check records (dead, and removed by the compiler, in
  // kernels that do not record them)
  int na;                    // particles visited within 2 sigma (the neighbour set, self included)
  unsigned vh;               // sum of visit_mix(j) over them (mod 2^32): the set, order-free
  float Fx, Fy;              // force sum
  float Sx, Sy;              // alignment sums (cos, sin) over the neighbour set incl. self
  int q;                     // seam wrap: counter-clockwise quarter turns of the composed map
};

// table entries per lane loaded together in the neighbour walk (scan phase, and the FP64 redo)
constexpr int kRowChunk = 4;
constexpr int kScanChunk = 8;  // measured on MI355X: 4 and 16 are slower
// lanes per particle from which the walk loads bucket heads in its scan (measured on MI355X: 1.7 %
// faster at 16 lanes, 1 % slower at 4 lanes with chunks of 4), and its chunk of entries per lane
constexpr int kHeadScanLanes = 8;

// 32-bit mixing of a particle index (the MurmurHash3 finaliser): summed over a neighbour set it
// names the set independently of the visiting order
__host__ __device__ inline unsigned visit_mix(unsigned h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}
constexpr int kHeadChunk = 2;
static_assert(32 % kScanChunk == 0, "scan chunks must tile the 32-entry window");

// Global-memory neighbour source: the previous step's SoA state and vertex buckets. With OCC the
// buckets' occupancy mask is staged in LDS by the workgroup: the table walk tests occupancy there
// and touches a bucket in global memory only when its vertex holds particles; without it the walk
// reads each entry's bucket count. Both visit the same buckets in the same order.
// SORTED: the buckets are known to be sorted (the kernels of crowded systems).
template <bool OCC, bool SORTED = false>
struct GlobalSource {
  static constexpr bool kOcc = OCC;
  static constexpr bool kCoop = true;
  BucketsIn b;
  const float4* xycs;
  const float* th;
  const unsigned* occ;  // LDS copy of the replica's occupancy mask of b (OCC only)
  __device__ __forceinline__ bool occupied(int w) const { return (occ[w >> 5] >> (w & 31)) & 1u; }
  struct Head { int c = 0, s0 = 0, s1 = 0; };
  // bucket head: count and the first two slots, loaded together (the slots are in bounds
  // whatever the count)
  __device__ __forceinline__ Head head(int w) const {
    Head h;
    h.c = load_at(b.count, w);
    const int2 s = load_at(reinterpret_cast<const int2*>(b.slot), w * (kSlots / 2));
    h.s0 = s.x;
    h.s1 = s.y;
    return h;
  }
  __device__ __forceinline__ int count(int w) const { return load_at(b.count, w); }
  __device__ __forceinline__ void slots(int w, int (&a)[kSlots]) const {
    const int4 s0 = load_at(reinterpret_cast<const int4*>(b.slot), 2 * w),
               s1 = load_at(reinterpret_cast<const int4*>(b.slot), 2 * w + 1);
    a[0] = s0.x; a[1] = s0.y; a[2] = s0.z; a[3] = s0.w;
    a[4] = s1.x; a[5] = s1.y; a[6] = s1.z; a[7] = s1.w;
  }
  // the particles of bucket w in ascending id order, without (each) and with (each_pos) their state
  template <class F>
  __device__ __forceinline__ void each(int w, const Head& h, F&& f) const {
    if (h.c == 0) return;
    if (h.c == 1) { f(h.s0); return; }
    if (h.c == 2) {  // in order when sorted by the finalize pass; else ordered here
      const int lo = b.sorted ? h.s0 : min(h.s0, h.s1), hi = b.sorted ? h.s1 : max(h.s0, h.s1);
      f(lo);
      f(hi);
      return;
    }
    for_bucket(b, w, f);
  }
  template <class F>
  __device__ __forceinline__ void each_pos(int w, const Head& h, F&& f) const {
    const int c = h.c;
    if (c == 0) return;
    if (c <= 2) {  // ids in the head
      const bool swap = !SORTED && !b.sorted && c == 2 && h.s1 < h.s0;
      const int j0 = swap ? h.s1 : h.s0, j1 = c == 2 ? (swap ? h.s0 : h.s1) : h.s0;
      const float4 q0 = pos(j0), q1 = pos(j1);
      f(j0, q0);
      if (c == 2) f(j1, q1);
      return;
    }
    if constexpr (!SORTED) {
      if (c > kSlots) {
        for_bucket(b, w, [&](int j) { f(j, pos(j)); });
        return;
      }
      // the slots in order, then the states of four at a time in flight together: one at a time, the few
      // particles piled on a vertex made their reader's wave the step's longest (2,000 particles 10.64 -> 10.25 us
      // per step)
      int a[kSlots];
      slots(w, a);
#pragma unroll
      for (int q = 0; q < kSlots; ++q) a[q] = q < c ? a[q] : 0x7fffffff;
      if (!b.sorted) sort8(a);
#pragma unroll
      for (int q0 = 0; q0 < kSlots; q0 += 4) {
        if (q0 >= c) break;
        float4 p[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = pos(q0 + k < c ? a[q0 + k] : a[0]);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (q0 + k < c) f(a[q0 + k], p[k]);
      }
    } else {
      // kBatch particles at a time: the next ids and all of a batch's states are in flight together.
      // One at a time, two dependent loads per particle, a lane with a few crowded vertices (up to
      // 60 particles each) walked 100 us by itself and bounded the 100,000-particle step.
      constexpr int kBatch = 4;
      const int* ids = c <= kSlots ? b.slot + (size_t)w * kSlots : b.big + h.s0;
      int id[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) id[k] = ids[k < c ? k : c - 1];
      for (int q0 = 0; q0 < c; q0 += kBatch) {
        float4 q[kBatch];
        int nx[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) q[k] = pos(id[k]);
        if (q0 + kBatch < c) {
#pragma unroll
          for (int k = 0; k < kBatch; ++k) nx[k] = ids[q0 + kBatch + k < c ? q0 + kBatch + k : c - 1];
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
          if (q0 + k < c) f(id[k], q[k]);
#pragma unroll
        for (int k = 0; k < kBatch; ++k) id[k] = nx[k];
      }
    }
  }
  __device__ __forceinline__ float4 pos(int j) const { return load_at(xycs, j); }
  __device__ __forceinline__ float theta(int j) const { return load_at(th, j); }
};

// LDS-resident neighbour source of the persistent kernel: vertex buckets as a CSR over the
// particles counting-sorted by vertex (begin[v] .. begin[v+1]), visited in ascending id order like
// the global buckets, so both paths add neighbours in the same order.
struct LdsSource {
  const uint32_t* begin;   // [V+1]
  const uint16_t* sorted;  // [n]
  const float4* xycs;
  const float* th;
  struct Head { int b = 0, c = 0; };
  __device__ __forceinline__ Head head(int w) const {
    Head h;
    h.b = (int)begin[w];
    h.c = (int)begin[w + 1] - h.b;
    return h;
  }
  static constexpr bool kOcc = false;  // counts are LDS reads already
  static constexpr bool kCoop = false;
  __device__ __forceinline__ int count(int w) const { return (int)begin[w + 1] - (int)begin[w]; }
  __device__ __forceinline__ bool occupied(int w) const { return begin[w + 1] != begin[w]; }
  template <class F>
  __device__ __forceinline__ void each(int, const Head& h, F&& f) const {
    const int b = h.b, c = h.c;
    if (c == 0) return;
    if (c == 1) { f((int)sorted[b]); return; }
    if (c == 2) {
      const int a = sorted[b], d = sorted[b + 1];
      if (a < d) { f(a); f(d); } else { f(d); f(a); }
      return;
    }
    int prev = -1;
    for (int r = 0; r < c; ++r) {
      int best = 0x7fffffff;
      for (int q = 0; q < c; ++q) {
        const int id = sorted[b + q];
        if (id > prev && id < best) best = id;
      }
      f(best);
      prev = best;
    }
  }
  template <class F>
  __device__ __forceinline__ void each_pos(int w, const Head& h, F&& f) const {
    each(w, h, [&](int j) { f(j, pos(j)); });
  }
  __device__ __forceinline__ float4 pos(int j) const { return xycs[j]; }
  __device__ __forceinline__ float theta(int j) const { return th[j]; }
};

// orders the LDS / global accesses of one wave (its lanes exchange data through memory)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// inclusive sum over the lanes of a wave (all active)
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// ---- neighbour walk of a whole wave (narrow groups)
//
// With one to four lanes per particle a lane owns several table entries, few of which are occupied,
// by one particle or by several: walked lane by lane, a wave pays for its unluckiest lane in every
// loop, and each visit is a chain of three dependent loads. Here the wave's occupied entries are
// compacted into LDS, its 64 lanes take one entry each (bucket head, pair coefficient) and then the
// entries' particles, leaving each pair's terms in LDS, and every lane adds the terms of its own
// entries in its own order: the sums are those of the lane-by-lane walk, bit for bit. Particles of a
// crowded bucket (more than kSlots) are added by the owner lane itself, in their place. Lanes without
// work load a fixed address instead of branching around the load: a load under a branch is waited
// for before the next is issued. Area per wave:
constexpr int kWaveEntries = 256;  // entries compacted at a time (more: entry by entry of the lanes)
constexpr int kWavePairs = 184;    // pairs of a round (a round takes as many entries as fit)
// whether P physical lanes per particle walk this way for sums laid out over LANES lanes (crowded:
// sorted buckets; with as many lanes as the layout the lane-by-lane walk is 2-3 % faster there, 65,000
// and 100,000 particles)
constexpr bool coop_walk(int lanes, int p, bool crowded) { return p != lanes || (lanes <= 4 && !crowded); }
// whether a wave has an area: for the walk, and for the FP64 headings of wave_heading_sum
constexpr bool wave_area(int lanes, int p, bool crowded) { return lanes <= 8 || coop_walk(lanes, p, crowded); }
// table entries per lane taken together, by physical lanes
constexpr int coop_chunk(int p) { return p >= 16 ? 2 : (p == 8 ? 4 : 8); }
struct WaveWalk {
  double2 F[kWavePairs];        // force terms
  float2 S[kWavePairs];         // alignment terms
  int2 ent[kWaveEntries + 64];  // (vertex | owner lane << 26, float bits of the distance); then a slot
                                //   per lane for what is not kept
  int pp[64 + 4];               // before each entry of the round: pairs, and << 16 particles counted
  unsigned vh[kWavePairs];      // visit_mix of the pair's particle (visit check only)
};
// what particle_step calls with the new vertex id, as soon as that is known
struct NoPlaced {
  __device__ void operator()(int) const {}
};
constexpr int kOwnerShift = 26;  // vertex ids below 2^26 (size_error)

// The alignment sum of one particle over the FP64 cosines and sines of its neighbours' headings, by the
// whole wave (all lanes present): rs .. re its row. A lane takes one entry and its bucket, then one
// neighbour and its sine; then every lane adds the terms of strand lane % LANES in the strand's order.
// The redo of a nearly cancelling sum is rare per particle but not per wave, and walked by the
// particle's own lanes it was the step's longest chain (up to 18,000 cycles of 38,000 at 9,001 particles,
// 54,000 of 107,000 at 100,000): four entries a lane at a time, each neighbour's heading and sine behind
// the one before. 9,001 particles 20.7 -> 18.8 us per step, 100,000 84.1 -> 72.9, 525,000 in 256 replicas
// 150.4 -> 148.5.
template <int LANES, class Src>
__device__ __forceinline__ void wave_heading_sum(const MeshDev& mesh, float t_near, const Src& src, WaveWalk* ww,
                                                 int rs, int re, double& sx, double& sy) {
  static_assert(kWavePairs >= 64 && (kWaveEntries + 64) * 2 >= 64 * kSlots, "terms of a round, ids of 64 buckets");
  const int wl = (int)__lane_id();
  int* ids = reinterpret_cast<int*>(ww->ent);
  for (int base = rs; base < re; base += 64) {  // a multiple of LANES: entry base + l is of strand l % LANES
    int2 ent = table_entry(mesh.nbr, min(base + wl, re - 1));
    if (base + wl >= re) ent.y = 0x7f800000;
    const bool near = __int_as_float(ent.y) <= t_near && (!Src::kOcc || src.occupied(ent.x));
    const int count = src.count(near ? ent.x : 0);
    int a[kSlots];
    src.slots(near ? ent.x : 0, a);
    const int c = near ? count : 0;
    if (!src.b.sorted && __builtin_amdgcn_ballot_w64(c > kSlots) != 0) {  // raw and crowded: rare
      for (int t = wl & (LANES - 1); t < 64 && base + t < re; t += LANES) {
        const int2 e = table_entry(mesh.nbr, base + t);
        if (__int_as_float(e.y) > t_near) break;
        src.each(e.x, src.head(e.x), [&](int j) {
          double sj, cj;
          sincos((double)src.theta(j), &sj, &cj);
          sx += cj;
          sy += sj;
        });
      }
    } else {
      if (!src.b.sorted && __builtin_amdgcn_ballot_w64(c > 1) != 0) {  // ids ascending
#pragma unroll
        for (int q = 0; q < kSlots; ++q) a[q] = q < c ? a[q] : 0x7fffffff;
        sort8(a);
      }
      const int upto = wave_scan(c), total = __builtin_amdgcn_readlane(upto, 63);
      ww->pp[wl] = upto - c;
      if (wl == 63) ww->pp[64] = upto;
      reinterpret_cast<int4*>(ids)[2 * wl] = make_int4(a[0], a[1], a[2], a[3]);
      reinterpret_cast<int4*>(ids)[2 * wl + 1] = make_int4(a[4], a[5], a[6], a[7]);
      constexpr uint64_t kEvery = LANES == 1 ? ~0ull : (LANES == 2 ? 0x5555555555555555ull :
                                  (LANES == 4 ? 0x1111111111111111ull : 0x0101010101010101ull));
      static_assert(LANES == 1 || LANES == 2 || LANES == 4 || LANES == 8, "strand mask");
      const uint64_t strand = __builtin_amdgcn_ballot_w64(c > 0) & (kEvery << (wl & (LANES - 1)));
      wave_sync();
      for (int k0 = 0; k0 < total; k0 += 64) {
        const int k = min(k0 + wl, total - 1);
        int t = 0;  // the entry that holds neighbour k
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) t += ww->pp[t + s] <= k ? s : 0;
        const int first = ww->pp[t], held = ww->pp[t + 1] - first;
        int j = ids[t * kSlots + (held > kSlots ? 0 : k - first)];
        if (held > kSlots) j = src.b.big[j + k - first];
        double sj, cj;
        sincos((double)src.theta(j), &sj, &cj);
        ww->F[wl] = make_double2(cj, sj);
        wave_sync();
        for (uint64_t m = strand; m != 0; m &= m - 1) {
          const int e = __builtin_ctzll(m), hi = min(ww->pp[e + 1], k0 + 64);
          for (int p = max(ww->pp[e], k0); p < hi; ++p) {
            const double2 f = ww->F[p - k0];
            sx += f.x;
            sy += f.y;
          }
        }
        wave_sync();
      }
    }
    if (__int_as_float(__builtin_amdgcn_readlane(ent.y, 63)) > t_near) break;  // rows ascend in distance
  }
}

// One particle's update (U1-U6 of the reference step) by a group of P lanes. The sums over the
// neighbours are laid out over LANES lanes: lane l of LANES adds the entries l, l + LANES, .. of the
// particle's table row in order, and a butterfly adds the lanes. That layout fixes the results to the
// bit; P, the lanes that do the work, is free: more than LANES where waves are few and the longest chain
// counts (the whole-wave walk, phys_lanes), half of 8 where that halves the passes of a workgroup (the
// persistent kernel).
//   me = (x, y, cos theta, sin theta) of particle i, th its heading, v its vertex id.
// Neighbours: particles bucketed on the vertices w of row v of the geodesic table; pair
// distance d = D[v, w]. Force and alignment for d < 2 sigma (ForceHelper.cpp:34-73,
// OrientationHelper.cpp:29-74, self included in the mean), count for 0 < d <= 2.4 sigma
// (2DTissue.cpp:254-268). The force is summed in FP64 (its FP32 rounding feeds the FP32 speed
// and Euler step; the FP64 value the large-displacement path); the alignment sums are FP32, redone
// in FP64 when they nearly cancel.
// active: false for the lanes past the last particle, which only help the wave (their own result
// is not used); ww: the wave's LDS area (whole-wave walk: all lanes of the wave present; else
// null). WAVE selects the seam-wrap loop of crowded systems (seam_wrap_group). Always inlined: as an
// out-of-line call (which the inliner picks once two kernels share an instantiation) its result
// and live state go through scratch memory.
template <int LANES, int P, bool WAVE = false, bool VISITS = false, class Src, class Placed = NoPlaced>
__device__ __forceinline__ StepOut particle_step(const MeshDev& mesh, const StepParams& prm, const Src& src, int i, float4 me,
                                        float th, int v, float eta, int lane, bool active = true,
                                        WaveWalk* ww = nullptr, const Placed& placed = {}) {
  // a lane's sums: those of strand lane % LANES of the layout (its copies on the lanes above LANES equal it);
  // with P = LANES / 2 those of strands lane and lane + P. The force is summed in FP64 (its FP32 rounding
  // drives the FP32 path).
  static_assert(P >= LANES || 2 * P == LANES, "one or two strands per lane");
  constexpr int NS = P < LANES ? 2 : 1, SUMW = P < LANES ? P : LANES;
  float Sx = 0.f, Sy = 0.f, Sx1 = 0.f, Sy1 = 0.f;  // (the second strand's, unused with one)
  double Fx64 = 0.0, Fy64 = 0.0, Fx1 = 0.0, Fy1 = 0.0;
  const double kc64 = prm.kc64;
  int na = 0, nb = 0, nb_only = 0;  // nb_only: counted without a pair by the whole-wave scan
  unsigned vh = 0u;
  const int rs = load_at(mesh.row_ptr, v), re = active ? load_at(mesh.row_ptr, v + 1) : rs;
  // pair set-up of a near entry (vertex w at distance d, bucket head h) and its particles
  auto visit_into = [&](double& fx, double& fy, float& sx, float& sy, int w, float d,
                        const typename Src::Head& h) __attribute__((always_inline)) {
    const double dd = d == 0.0f ? 0.001 : (double)d;
    const double g64 = (kc64 * (dd - prm.two_sigma64)) / dd;
    const bool counted = d != 0.0f;
    src.each_pos(w, h, [&](int j, const float4& q) __attribute__((always_inline)) {
      if (j != i) {
        fx += g64 * ((double)me.x - (double)q.x);
        fy += g64 * ((double)me.y - (double)q.y);
      }
      sx += q.z;
      sy += q.w;
      ++na;
      vh += visit_mix((unsigned)j);
      if (counted) ++nb;
    });
  };
  auto visit = [&](int w, float d, const typename Src::Head& h) __attribute__((always_inline)) {
    visit_into(Fx64, Fy64, Sx, Sy, w, d, h);
  };
  // Each lane walks its entries rs + lane + m * LANES, m = 0, 1, .., in order.
  if constexpr (LANES >= kHeadScanLanes && P <= LANES) {
    // At most a few entries per lane: the scan loads each near entry's bucket head (count and
    // first slots) together with the entries' counts, and the lane visits its occupied entries
    // from registers: table entry -> bucket head -> particles, no reload of marked entries.
    constexpr int kChunk = kHeadChunk * NS;
    for (int base = rs + lane; base < re; base += kChunk * P) {
      int2 ent[kChunk];
      typename Src::Head hd[kChunk];
#pragma unroll
      for (int k = 0; k < kChunk; ++k) {
        const int e = base + k * P;
        ent[k] = table_entry(mesh.nbr, min(e, re - 1));
        if (e >= re) ent[k].y = 0x7f800000;  // +inf ends the walk
      }
      bool oc[kChunk];
#pragma unroll
      for (int k = 0; k < kChunk; ++k)
        oc[k] = __int_as_float(ent[k].y) <= prm.t_count && (!Src::kOcc || src.occupied(ent[k].x));
#pragma unroll
      for (int k = 0; k < kChunk; ++k) {
        hd[k] = src.head(oc[k] ? ent[k].x : 0);
        if (!oc[k]) hd[k].c = 0;
      }
      bool stop = false;
#pragma unroll
      for (int k = 0; k < kChunk; ++k) {
        const float d = __int_as_float(ent[k].y);
        if (d > prm.t_count) {  // rows ascend in distance
          stop = true;
          break;
        }
        if (d > prm.t_near) nb += hd[k].c;  // counted only
        else if (hd[k].c > 0) {
          if (k % NS == 0) visit(ent[k].x, d, hd[k]);
          else visit_into(Fx1, Fy1, Sx1, Sy1, ent[k].x, d, hd[k]);
        }
      }
      if (stop) break;
    }
  } else if constexpr (Src::kCoop && coop_walk(LANES, P, WAVE)) {
    constexpr int kChunk = coop_chunk(P);
    const int wl = (int)__lane_id();
    bool done = false;
    for (int wbase = rs + lane;; wbase += kChunk * P) {
      const bool more = !done && wbase < re;
      if (__builtin_amdgcn_ballot_w64(more) == 0) break;
      // the lane's next kChunk entries, the occupied ones marked (with the mask in LDS: counted-only
      // entries too, their count comes with the head; else their count is added here)
      int2 ent[kChunk];
      unsigned mark = 0u;
#pragma unroll
      for (int k = 0; k < kChunk; ++k) {
        const int e = wbase + k * P;
        ent[k] = table_entry(mesh.nbr, max(min(e, re - 1), 0));
        if (!more || e >= re) ent[k].y = 0x7f800000;
      }
      if constexpr (Src::kOcc) {
#pragma unroll
        for (int k = 0; k < kChunk; ++k)
          mark |= __int_as_float(ent[k].y) <= prm.t_count && src.occupied(ent[k].x) ? 1u << k : 0u;
      } else {
        int cnt[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) cnt[k] = src.count(__int_as_float(ent[k].y) <= prm.t_count ? ent[k].x : 0);
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          const float d = __int_as_float(ent[k].y);
          nb_only += d > prm.t_near && d <= prm.t_count ? cnt[k] : 0;
          mark |= d <= prm.t_near && cnt[k] > 0 ? 1u << k : 0u;
        }
      }
      done = __int_as_float(ent[kChunk - 1].y) > prm.t_count;  // rows ascend in distance
      // (hardly ever more marks than the list holds: then one entry of each lane at a time)
      const bool split = 64 * kChunk > kWaveEntries &&
                         __builtin_amdgcn_readlane(wave_scan(__builtin_popcount(mark)), 63) > kWaveEntries;
      for (unsigned all = split ? 1u : ~0u; all != 0u; all = split ? (all << 1) & ((1u << kChunk) - 1u) : 0u) {
        // places in the list: by particle, then by strand, then in the row's order; [first, last) of
        // the lane's strand
        int first, last, at[kChunk], total = 0;
        const unsigned kept = mark & all;
        if constexpr (P == LANES) {
          const int mine = __builtin_popcount(kept), upto = wave_scan(mine);
          total = __builtin_amdgcn_readlane(upto, 63);
          last = first = upto - mine;
#pragma unroll
          for (int k = 0; k < kChunk; ++k) {
            at[k] = last;
            last += (kept >> k) & 1u;
          }
        } else {
          // lanes v, v + LANES, .. of the group share strand v = lane % LANES
          constexpr unsigned kEvery = LANES == 1 ? ~0u : (LANES == 2 ? 0x55555555u : (LANES == 4 ? 0x11111111u : 0x01010101u));
          constexpr unsigned kGroup = P >= 32 ? ~0u : (1u << P) - 1u;
          const int v = lane & (LANES - 1), gbase = wl & ~(P - 1);
          const unsigned same = kEvery << v & kGroup;                // the strand's lanes
          const unsigned less = kEvery * ((1u << v) - 1u) & kGroup;  // the lanes of the strands before
          const unsigned below = same & ((1u << lane) - 1u);
          int p = 0, in_strand = 0;
#pragma unroll
          for (int k = 0; k < kChunk; ++k) {
            const uint64_t b = __builtin_amdgcn_ballot_w64(((kept >> k) & 1u) != 0u);
            const unsigned g = (unsigned)(b >> gbase) & kGroup;
            p += __builtin_popcountll(b & ((1ull << gbase) - 1ull)) + __builtin_popcount(g & less);
            at[k] = in_strand + __builtin_popcount(g & below);
            in_strand += __builtin_popcount(g & same);
            total += __builtin_popcountll(b);
          }
#pragma unroll
          for (int k = 0; k < kChunk; ++k) at[k] += p;
          first = p;
          last = p + in_strand;
        }
        if (total == 0) continue;
#pragma unroll
        for (int k = 0; k < kChunk; ++k)
          ww->ent[(kept >> k) & 1u ? at[k] : kWaveEntries + wl] =
              make_int2((int)((unsigned)ent[k].x | ((unsigned)wl << kOwnerShift)), ent[k].y);
        wave_sync();
        for (int r0 = 0; r0 < total;) {
          // one entry per lane: its bucket and pair coefficient
          const bool has = r0 + wl < total;
          const int2 en = ww->ent[has ? r0 + wl : r0];
          const int w = en.x & ((1 << kOwnerShift) - 1), owner = (int)((unsigned)en.x >> kOwnerShift);
          const float d = __int_as_float(en.y);
          const int count = src.count(has ? w : 0);
          int a[kSlots];  // the slots are in bounds whatever the count
          src.slots(has ? w : 0, a);
          const float ox = __shfl(me.x, owner, 64), oy = __shfl(me.y, owner, 64);
          const int oi = __shfl(i, owner, 64);
          const double dd = d == 0.0f ? 0.001 : (double)d;
          const double g64 = (kc64 * (dd - prm.two_sigma64)) / dd;
          const int c = has ? count : 0;
          const bool is_near = !Src::kOcc || d <= prm.t_near;
          const int np = c > kSlots || !is_near ? 0 : c;  // pairs left in LDS
          const int pk = c > kSlots ? 0 : (np | (d != 0.0f ? c << 16 : 0));
          const int sum = wave_scan(pk), before = sum - pk;
          const uint64_t fits = __builtin_amdgcn_ballot_w64((sum & 0xffff) <= kWavePairs);
          const int taken = min(fits == ~0ull ? 64 : __builtin_ctzll(~fits), total - r0);  // entries of this round
          const bool crowded = __builtin_amdgcn_ballot_w64(c > kSlots && wl < taken) != 0;
          const int at = before & 0xffff;
          auto term = [&](int q, int j, const float4& p) __attribute__((always_inline)) {
            const double fx = g64 * ((double)ox - (double)p.x), fy = g64 * ((double)oy - (double)p.y);
            ww->F[at + q] = j != oi ? make_double2(fx, fy) : make_double2(0.0, 0.0);
            ww->S[at + q] = make_float2(p.z, p.w);
            if constexpr (VISITS) ww->vh[at + q] = visit_mix((unsigned)j);
          };
          const int mine_np = wl < taken ? np : 0;
          const bool more2 = __builtin_amdgcn_ballot_w64(mine_np > 2) != 0;
          if (!src.b.sorted) {  // ids ascending
            if (more2) {
#pragma unroll
              for (int q = 0; q < kSlots; ++q) a[q] = q < np ? a[q] : 0x7fffffff;
              sort8(a);
            } else if (np == 2) {
              const int j0 = min(a[0], a[1]);
              a[1] = max(a[0], a[1]);
              a[0] = j0;
            }
          }
          {
            const float4 p0 = src.pos(mine_np > 0 ? a[0] : 0), p1 = src.pos(mine_np > 1 ? a[1] : 0);
            if (!more2) {
              if (mine_np > 0) term(0, a[0], p0);
              if (mine_np > 1) term(1, a[1], p1);
            } else {
              const float4 p2 = src.pos(mine_np > 2 ? a[2] : 0), p3 = src.pos(mine_np > 3 ? a[3] : 0);
              if (mine_np > 0) term(0, a[0], p0);
              if (mine_np > 1) term(1, a[1], p1);
              if (mine_np > 2) term(2, a[2], p2);
              if (mine_np > 3) term(3, a[3], p3);
              if (__builtin_amdgcn_ballot_w64(mine_np > 4) != 0) {
                float4 p[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) p[q] = src.pos(mine_np > 4 + q ? a[4 + q] : 0);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                  if (mine_np > 4 + q) term(4 + q, a[4 + q], p[q]);
              }
            }
          }
          ww->pp[wl] = before;
          if (wl == 63) ww->pp[64] = sum;
          wave_sync();
          // the strand's entries of the round
          const int lo = min(max(first - r0, 0), taken), hi = min(max(last - r0, 0), taken);
          const int s0 = ww->pp[lo], s1 = ww->pp[hi];
          auto add = [&](int p) __attribute__((always_inline)) {
            const double2 f = ww->F[p];
            const float2 q = ww->S[p];
            Fx64 += f.x;
            Fy64 += f.y;
            Sx += q.x;
            Sy += q.y;
            if constexpr (VISITS) vh += ww->vh[p];
          };
          if (!crowded) {
            for (int p = s0 & 0xffff; p < (s1 & 0xffff); ++p) add(p);
          } else {
            for (int t = lo; t < hi; ++t) {
              const int p1 = ww->pp[t + 1] & 0xffff;
              int p = ww->pp[t] & 0xffff;
              if (p == p1) {  // crowded, or counted only
                const int2 e = ww->ent[r0 + t];
                const int we = e.x & ((1 << kOwnerShift) - 1);
                const typename Src::Head he = src.head(we);
                if (he.c > kSlots) {
                  if (__int_as_float(e.y) <= prm.t_near) visit(we, __int_as_float(e.y), he);
                  else nb += he.c;
                }
              }
              for (; p < p1; ++p) add(p);
            }
          }
          na += (s1 - s0) & 0xffff;
          nb += (s1 >> 16) - (s0 >> 16);
          wave_sync();
          r0 += taken;
        }
      }
    }
  } else {
    // Windows of 32 entries per lane:
    //  (1) scan: the window's table entries are loaded kScanChunk at a time (one load latency per
    //      chunk) and their occupancy found (from the LDS mask, or from the bucket counts);
    //      occupied counted-only entries (2 sigma <= d <= 2.4 sigma) add their bucket count to nb,
    //      and occupied near entries are marked;
    //  (2) visit: only the marked entries, in order, set up their pair coefficient and add their
    //      particles. Most table entries have empty buckets, so the lanes of a wave loop over a
    //      few occupied entries instead of paying the pair set-up for every entry; the order, and
    //      so every sum, is that of a walk over all entries.
    bool done = false;
    for (int wbase = rs + lane; !done && wbase < re; wbase += 32 * LANES) {
      unsigned mark = 0u;
      for (int m0 = 0; m0 < 32 && !done; m0 += kScanChunk) {
        int2 ent[kScanChunk];
        int cnt[kScanChunk];
#pragma unroll
        for (int k = 0; k < kScanChunk; ++k) {
          const int e = wbase + (m0 + k) * LANES;
          ent[k] = table_entry(mesh.nbr, min(e, re - 1));
          if (e >= re) ent[k].y = 0x7f800000;  // +inf ends the walk
        }
        bool oc[kScanChunk];
        if constexpr (Src::kOcc) {
          // occupancy from LDS; bucket counts only for the occupied entries counted without a
          // pair (2 sigma <= d <= 2.4 sigma)
#pragma unroll
          for (int k = 0; k < kScanChunk; ++k) oc[k] = __int_as_float(ent[k].y) <= prm.t_count && src.occupied(ent[k].x);
#pragma unroll
          for (int k = 0; k < kScanChunk; ++k) {
            const bool want = oc[k] && __int_as_float(ent[k].y) > prm.t_near;
            cnt[k] = src.count(want ? ent[k].x : 0);
            if (!want) cnt[k] = 0;
          }
        } else {
#pragma unroll
          for (int k = 0; k < kScanChunk; ++k) {
            const bool want = __int_as_float(ent[k].y) <= prm.t_count;
            cnt[k] = src.count(want ? ent[k].x : 0);
            if (!want) cnt[k] = 0;
          }
#pragma unroll
          for (int k = 0; k < kScanChunk; ++k) oc[k] = cnt[k] > 0;
        }
#pragma unroll
        for (int k = 0; k < kScanChunk; ++k) {
          const float d = __int_as_float(ent[k].y);
          if (d > prm.t_count) {  // rows ascend in distance
            done = true;
            break;
          }
          if (d > prm.t_near) nb += cnt[k];  // counted only
          else if (oc[k]) mark |= 1u << (m0 + k);
        }
      }
      while (mark) {
        const int m = __builtin_ctz(mark);
        mark &= mark - 1u;
        const int2 en = table_entry(mesh.nbr, wbase + m * LANES);
        visit(en.x, __int_as_float(en.y), src.head(en.x));
      }
    }
  }
  if constexpr (NS == 2) {  // the butterfly's first level
    Fx64 += Fx1;
    Fy64 += Fy1;
    Sx += Sx1;
    Sy += Sy1;
  }
  Fx64 = group_sum<SUMW>(Fx64);
  Fy64 = group_sum<SUMW>(Fy64);
  float Fx = (float)Fx64, Fy = (float)Fy64;
  Sx = group_sum<SUMW>(Sx);
  Sy = group_sum<SUMW>(Sy);
  na = group_sum<SUMW>(na);
  vh = group_sum<SUMW>(vh);
  nb = group_sum<SUMW>(nb);
  if constexpr (Src::kCoop && coop_walk(LANES, P, WAVE)) nb += group_sum<P>(nb_only);

  // speed, velocity, Euler step (Locomotion.cpp:71-84)
  const float Fm = sqrtf(Fx * Fx + Fy * Fy);
  const float spd = prm.v0 + prm.mu * Fm;
  float vx = me.z * spd, vy = me.w * spd;
  double xn = (double)(me.x + vx * prm.dt), yn = (double)(me.y + vy * prm.dt);

  // The FP32 mean heading has error ~ na * 6e-8 / |S|, scaled by dt/tau in the update; the FP32
  // displacement has error ~ 1e-7 * |D|. Either beyond ~1e-7 => redo that part in FP64.
  const float Sm = sqrtf(Sx * Sx + Sy * Sy);
  const bool weak = !(Sm >= 0.6f * prm.rate * (float)na);
  const bool big = !(spd * prm.dt <= kBigStep);
  double thn;
  if (big) {  // uniform over the particle's lanes: the sums were reduced over the group
    double st, ct;
    sincos((double)th, &st, &ct);
    const double spd64 = prm.v064 + prm.mu64 * sqrt(Fx64 * Fx64 + Fy64 * Fy64);
    const double vx64 = ct * spd64, vy64 = st * spd64;
    xn = (double)me.x + vx64 * prm.dt64;
    yn = (double)me.y + vy64 * prm.dt64;
    vx = (float)vx64;
    vy = (float)vy64;
  }
  double Sx64 = 0.0, Sy64 = 0.0;
  constexpr bool kWaveHeadings = Src::kCoop && wave_area(LANES, P, WAVE) && LANES <= 8;
  if constexpr (kWaveHeadings) {
    for (uint64_t m = __builtin_amdgcn_ballot_w64(weak && active && lane == 0); m != 0; m &= m - 1) {
      const int first = __builtin_ctzll(m);
      double sx = 0.0, sy = 0.0;
      wave_heading_sum<LANES>(mesh, prm.t_near, src, ww, __builtin_amdgcn_readlane(rs, first),
                              __builtin_amdgcn_readlane(re, first), sx, sy);
      if (((int)__lane_id() & ~(P - 1)) == first) {
        Sx64 = sx;
        Sy64 = sy;
      }
    }
  }
  if (weak) {
    // the alignment sum again, over the neighbours' headings in FP64
    auto strand = [&](int first, double& sx, double& sy) __attribute__((always_inline)) {
      for (int base = rs + first; base < re; base += kRowChunk * LANES) {
        int2 ent[kRowChunk];
        typename Src::Head head[kRowChunk];
#pragma unroll
        for (int k = 0; k < kRowChunk; ++k) {
          const int e = base + k * LANES;
          ent[k] = table_entry(mesh.nbr, min(e, re - 1));
          if (e >= re) ent[k].y = 0x7f800000;
        }
#pragma unroll
        for (int k = 0; k < kRowChunk; ++k) {
          const bool oc = __int_as_float(ent[k].y) <= prm.t_near && (!Src::kOcc || src.occupied(ent[k].x));
          head[k] = src.head(oc ? ent[k].x : 0);
          if (!oc) head[k].c = 0;
        }
        bool stop = false;
#pragma unroll
        for (int k = 0; k < kRowChunk; ++k) {
          const float d = __int_as_float(ent[k].y);
          if (d > prm.t_near) { stop = true; break; }
          src.each(ent[k].x, head[k], [&](int j) {
            double sj, cj;
            sincos((double)src.theta(j), &sj, &cj);
            sx += cj;
            sy += sj;
          });
        }
        if (stop) break;
      }
    };
    if constexpr (kWaveHeadings) {
    } else if constexpr (NS == 1) {
      strand(lane & (LANES - 1), Sx64, Sy64);
    } else {
      double sx[2] = {0.0, 0.0}, sy[2] = {0.0, 0.0};
      strand(lane, sx[0], sy[0]);
      strand(lane + P, sx[1], sy[1]);
      Sx64 = sx[0] + sx[1];
      Sy64 = sy[0] + sy[1];
    }
    {
      Sx64 = group_sum<SUMW>(Sx64);
      Sy64 = group_sum<SUMW>(Sy64);
      const double mean = atan2(Sy64, Sx64);
      double delta = mean - (double)th;
      if (delta > kPi) delta -= 2.0 * kPi;
      else if (delta <= -kPi) delta += 2.0 * kPi;
      thn = (double)th + prm.rate64 * delta + (double)eta;
      Sx = (float)Sx64;
      Sy = (float)Sy64;
    }
  }
  if (!weak) {
    const float mean = atan2f(Sy, Sx);
    float delta = mean - th;
    if (delta > kPiF) delta -= kTwoPiF;
    else if (delta <= -kPiF) delta += kTwoPiF;
    thn = (double)(th + prm.rate * delta + eta);
  }

  // seam wrap (EuclideanTiling.cpp:31-69) and validation (Validation.cpp:40-72)
  StepOut o;
  o.fl = 0;
  o.q = 0;
  o.Fx = Fx;
  o.Fy = Fy;
  o.Sx = Sx;
  o.Sy = Sy;
  double px = xn, py = yn;
  const bool finite = isfinite(xn) && isfinite(yn) && isfinite(thn);
  if (!finite) o.fl |= kFlagNonfinite;
  const bool leaves = finite && !inside_unit(px, py);
  bool folded = false;
  if (leaves) folded = seam_fold(me.x, me.y, px, py, thn, prm.max_crossings, &o.q);
  const bool loop = leaves && !folded;  // rare: the closed form does not settle the move
  double dth = 0.0;
  if constexpr (WAVE) {  // every lane of the wave goes along, so that all 64 can take the last flight
    if (__builtin_amdgcn_ballot_w64(loop) != 0) {
      double lx = loop ? px : 0.5, ly = loop ? py : 0.5;
      int q = 0;
      const bool good = seam_wrap_group<P, true>(me.x, me.y, lx, ly, dth, prm.max_crossings, lane, &q);
      if (loop) {
        px = lx;
        py = ly;
        o.q = q;
        if (!good) o.fl |= kFlagTiling;
      }
    }
  } else if (loop) {
    if (!seam_wrap_group<P, false>(me.x, me.y, px, py, dth, prm.max_crossings, lane, &o.q)) o.fl |= kFlagTiling;
  }
  if (finite && !folded) thn = wrap_heading(thn + dth);
  if (finite && !inside_unit(px, py)) o.fl |= kFlagLost;
  o.xo = (float)px;
  o.yo = (float)py;
  o.to = (float)thn;
  o.vx = vx;
  o.vy = vy;
  o.nb = nb;
  o.na = na;
  o.vh = vh;
  // UV -> 3D remap of the stored FP32 position (CellHelper.cpp:71-85)
  o.L = locate<P>(mesh, (double)o.xo, (double)o.yo, lane);
  placed(o.L.vid);
  sincosf(o.to, &o.so, &o.co);
  // order parameter (LinearAlgebra.cpp:90-105, z = 0): sign of the cross product's z component
  const double cz = (double)o.xo * (double)vy - (double)o.yo * (double)vx;
  o.sgn = cz > 0.0 ? 1 : (cz < 0.0 ? -1 : 0);
  return o;
}

}  // namespace tdev
