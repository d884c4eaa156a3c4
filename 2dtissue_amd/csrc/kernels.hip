// gfx950 kernels around the tiled step (step_kernel.h): bucket finalize, order parameters, flags, initial
// states, output stream, neighbour lists; and the dispatch of the step's launch shapes.
#include <hip/hip_runtime.h>

#include <climits>

#include "launch.h"
#include "rng.h"
#include "step_kernel.h"

using namespace tdev;

namespace tissue {

namespace {

// crowded buckets up to this many particles are sorted in LDS (larger ones in global memory)
constexpr int kSortCap = 512;

// Sort every bucket of set bs that holds two or more particles. One thread per particle: the
// bucket's second arrival (the insertion left the vertex in its entry of multi, -1 in the others)
// sorts it, up to kSlots ids in place with the register network. (A compact list of such buckets
// needs a counter, and a returning atomic on one address is served every 12 ns: with 25,000 shared
// vertices it cost the bucketing of 100,000 particles 300 us by itself.)
// A crowded bucket (more than kSlots) is then taken by its whole wave: its slots and its entries
// of the overflow list are gathered (ballot compaction), ranked, and written in ascending order to
// a fresh range of the replica's big area, whose offset replaces the bucket's first slot.
// The kernel is a chain of dependent loads, so independent ones are issued together: the overflow
// count and the particle's entry, then a bucket's count and all of its slots, and for a crowded
// bucket the big-area reservation with the overflow scan. single_n > 0: one replica of single_n
// particles, whose tiles need not be read (block b covers particles b * blockDim.x ...).
__global__ void __launch_bounds__(kStepMaxBlock) k_bucket_finalize(const ReplicaDesc* reps, const TileDesc* tiles,
                                                                   int nv, int single_n, BucketSet bs) {
  __shared__ __align__(16) int lds[kStepMaxBlock / 64][kSortCap];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int r = 0, off = 0, k = blockIdx.x * (int)blockDim.x + tid, cap = single_n;
  if (single_n <= 0) {
    const TileDesc tile = tiles[blockIdx.x];
    if (tile.r < 0) return;
    r = tile.r;
    off = reps[r].off;
    cap = reps[r].n;
    k = tile.q * (int)blockDim.x + tid;
  }
  const int novf = bs.ovf_n[r];
  const int v = k < cap ? bs.multi[off + k] : -1;
  int* slot = bs.slot + (size_t)r * nv * kSlots;
  int c = 0;
  int4 s0 = make_int4(0, 0, 0, 0), s1 = s0;
  if (v >= 0) {
    int* sl = slot + (size_t)v * kSlots;
    s0 = reinterpret_cast<const int4*>(sl)[0];
    s1 = reinterpret_cast<const int4*>(sl)[1];
    c = bs.count[(size_t)r * nv + v];
    if (c <= kSlots) {
      int a[kSlots] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
      for (int q = 0; q < kSlots; ++q) a[q] = q < c ? a[q] : 0x7fffffff;
      sort8(a);
#pragma unroll
      for (int q = 0; q < kSlots; ++q)
        if (q < c) sl[q] = a[q];
    }
  }
  unsigned long long crowded = __ballot(c > kSlots);
  if (crowded == 0ull) return;  // uniform over the wave
  const int2* ovf = bs.ovf + off;
  int* big = bs.big + off;
  // the ranges of all the wave's crowded buckets reserved with one atomic, in lane order (a
  // returning device-scope atomic is a memory-side round trip; one per bucket serialised them)
  int pre = c > kSlots ? c : 0;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(pre, d, 64);
    if (lane >= d) pre += o;
  }
  const int total = __shfl(pre, 63, 64);
  int base0 = 0;
  if (lane == 0) base0 = atomicAdd(&bs.big_n[r], total);
  base0 = __shfl(base0, 0, 64);
  const int my_start = base0 + pre - (c > kSlots ? c : 0);
  // the overflow list's first 256 entries, loaded once for all the wave's crowded buckets
  int2 e0[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int q = 64 * u + lane;
    e0[u] = q < novf ? ovf[q] : make_int2(-1, 0);
  }
  while (crowded) {
    const int src = __ffsll((long long)crowded) - 1;
    crowded &= crowded - 1ull;
    const int w = __shfl(v, src, 64);
    const int cw = __shfl(c, src, 64);
    const int reserved = __shfl(my_start, src, 64);
    int* sl = slot + (size_t)w * kSlots;
    const bool in_lds = cw <= kSortCap - 4;  // room for the padding below
    if (in_lds) {
      int* buf = lds[wave];
      // the bucket's slots as its lane loaded them above
      const int f0 = __builtin_amdgcn_readlane(s0.x, src), f1 = __builtin_amdgcn_readlane(s0.y, src);
      const int f2 = __builtin_amdgcn_readlane(s0.z, src), f3 = __builtin_amdgcn_readlane(s0.w, src);
      const int f4 = __builtin_amdgcn_readlane(s1.x, src), f5 = __builtin_amdgcn_readlane(s1.y, src);
      const int f6 = __builtin_amdgcn_readlane(s1.z, src), f7 = __builtin_amdgcn_readlane(s1.w, src);
      if (lane < kSlots)
        buf[lane] = lane < 4 ? (lane < 2 ? (lane == 0 ? f0 : f1) : (lane == 2 ? f2 : f3))
                             : (lane < 6 ? (lane == 4 ? f4 : f5) : (lane == 6 ? f6 : f7));
      int fill = kSlots;
      // the overflow entries in chunks of 256 (four loads per lane in flight together; the first
      // chunk loaded before the loop), compacted in order
      for (int q0 = 0; q0 < novf; q0 += 256) {
        int2 e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int q = q0 + 64 * u + lane;
          e[u] = q0 == 0 ? e0[u] : (q < novf ? ovf[q] : make_int2(-1, 0));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bool m = e[u].x == w;
          const unsigned long long bm = __ballot(m);
          if (m) buf[fill + __popcll(bm & ((1ull << lane) - 1ull))] = e[u].y;
          fill += __popcll(bm);
        }
      }
      if (lane < 4) buf[cw + lane] = 0x7fffffff;  // pad to a multiple of four (never below an id)
      wave_sync();
      int* dst = big + reserved;
      // rank of each id among the bucket's (distinct) ids = its position in ascending order; the
      // ids are read four at a time, several reads in flight
      const int cw4 = (cw + 3) & ~3;
      for (int q = lane; q < cw; q += 64) {
        const int val = buf[q];
        int rank = 0;
#pragma unroll 4
        for (int j = 0; j < cw4; j += 4) {
          const int4 b4 = *reinterpret_cast<const int4*>(buf + j);
          rank += (int)(b4.x < val) + (int)(b4.y < val) + (int)(b4.z < val) + (int)(b4.w < val);
        }
        dst[rank] = val;
      }
    } else {
      // rare: gathered and sorted in place in global memory
      int* dst = big + reserved;
      if (lane < kSlots) dst[lane] = sl[lane];
      int fill = kSlots;
      for (int q0 = 0; q0 < novf; q0 += 64) {
        const int q = q0 + lane;
        const int2 e = q < novf ? ovf[q] : make_int2(-1, 0);
        const bool m = e.x == w;
        const unsigned long long bm = __ballot(m);
        if (m) dst[fill + __popcll(bm & ((1ull << lane) - 1ull))] = e.y;
        fill += __popcll(bm);
      }
      wave_sync();
      if (lane == 0) {
        for (int a = 1; a < cw; ++a) {
          const int val = dst[a];
          int b = a - 1;
          while (b >= 0 && dst[b] > val) { dst[b + 1] = dst[b]; --b; }
          dst[b + 1] = val;
        }
      }
    }
    wave_sync();
    if (lane == 0) sl[0] = reserved;
  }
}

// order parameters of replica r at step s, one workgroup per (r, s)
__global__ void __launch_bounds__(kPhiBlock) k_phi_tiles(int steps, const int* tile_begin, int n_logical, int per_tile,
                                                         const OrderPartial* partial, const ReplicaDesc* reps,
                                                         double* phi, int phi_stride, int t_base, int R, RunEnd end) {
  // the run's last reduction also ends the run, one thread per replica in its first workgroups
  if (end.halt) {
    const int e = blockIdx.x * kPhiBlock + (int)threadIdx.x;
    if (e < R) end_run(end, R, e, end.last_row[e], end.first_bad[e]);
  }
  const int r = blockIdx.x / steps, s = blockIdx.x % steps;
  block_phi(partial + (size_t)s * n_logical * per_tile, tile_begin[r] * per_tile, tile_begin[r + 1] * per_tile, reps[r].n,
            phi + 2 * ((size_t)r * phi_stride + t_base + s));
}

__global__ void k_flags_begin(int R, const unsigned* halt, unsigned* rows, int* first_bad) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  rows[r] = halt[r];
  rows[R + r] = 0u;
  first_bad[r] = INT_MAX;
}

// the state from x, y, theta (device memory, or mapped host memory: each value is read once), with no
// velocity, neighbour count or flag yet; x, y and theta may be vx, vy and a buffer written later
__global__ void k_adopt(int n, const float* x, const float* y, const float* th, float4* xycs, float* th_out, float* vx,
                        float* vy, int* nbr, int R, unsigned* halt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < R) halt[i] = 0u;  // R <= n: a replica holds a particle at least
  if (i >= n) return;
  const float xi = x[i], yi = y[i], ti = th[i];
  float s, c;
  sincosf(ti, &s, &c);
  xycs[i] = make_float4(xi, yi, c, s);
  th_out[i] = ti;
  vx[i] = 0.f;
  vy[i] = 0.f;
  nbr[i] = 0;
}

// particles [first, first + n) of the state and of the outputs, what is asked for of them (PackAt), laid out as
// the caller's arrays are, into mapped host memory (consecutive lanes write consecutive words). The writes pass
// over the host link and bound the call: all arrays for a caller who wants one were 75 us instead of 29
// (neighbour counts of 100,000 particles). ALL: every array (no choices to load)
template <bool ALL>
__global__ void k_pack_state(int first, int n, const float4* xycs, const float* th, const int* vid, PackAt w, float* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const auto at = [&](int k) __attribute__((always_inline)) { return out + (ALL ? k : w.at[k]) * (size_t)n + i; };
  if (ALL || w.at[0] >= 0 || w.at[1] >= 0) {
    const float4 q = xycs[first + i];
    if (ALL || w.at[0] >= 0) *at(0) = q.x;
    if (ALL || w.at[1] >= 0) *at(1) = q.y;
  }
  if (ALL || w.at[2] >= 0) *at(2) = th[first + i];
  if (ALL || w.at[3] >= 0) *reinterpret_cast<int*>(at(3)) = vid[first + i];
}

template <bool ALL>
__global__ void k_pack_outputs(int first, int n, const float* vx, const float* vy, const float* r3x, const float* r3y,
                               const float* r3z, const int* face, const int* nbr, PackAt w, float* out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;  // a word of r3d [n][3]; the first n also one of each other
  if (t >= 3 * n) return;
  const auto at = [&](int k, int all) __attribute__((always_inline)) { return out + (ALL ? all : w.at[k]) * (size_t)n + t; };
  if (ALL || w.at[2] >= 0) {
    const int i = t / 3, c = t - 3 * i;
    *at(2, 2) = (c == 0 ? r3x : (c == 1 ? r3y : r3z))[first + i];
  }
  if (t >= n) return;
  if (ALL || w.at[0] >= 0) *at(0, 0) = vx[first + t];
  if (ALL || w.at[1] >= 0) *at(1, 1) = vy[first + t];
  if (ALL || w.at[3] >= 0) *reinterpret_cast<int*>(at(3, 5)) = face[first + t];
  if (ALL || w.at[4] >= 0) *reinterpret_cast<int*>(at(4, 6)) = nbr[first + t];
}

// words of mapped host memory into device memory
__global__ void k_fetch(size_t n, const float* from, float* to) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) to[i] = from[i];
}

// the counts, masks and list lengths of three bucket sets
__global__ void k_clear_sets(size_t cells, size_t words, int R, BucketSet a, BucketSet b, BucketSet c, int sets) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const BucketSet& s = k == 0 ? a : (k == 1 ? b : c);
    if (k >= sets) break;
    if (i < cells) s.count[i] = 0;
    if (i < words) s.occ[i] = 0u;
    if (i < (size_t)R) {
      s.ovf_n[i] = 0;
      s.big_n[i] = 0;
    }
  }
}

// seam wrap of n moves, LANES lanes per move (the step kernel's lane groups); whole groups only
template <int LANES, bool WAVE>
__global__ void __launch_bounds__(256) k_seam_wrap(int n, const double2* start, double2* end, double* dtheta,
                                                   int* quarter, int* ok, int max_crossings) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = t / LANES, lane = t & (LANES - 1);
  if (i >= n) return;  // uniform over the group
  const double2 a = start[i];
  double px = end[i].x, py = end[i].y, dth = 0.0;
  int q = 0;
  const bool good = seam_wrap_group<LANES, WAVE>(a.x, a.y, px, py, dth, max_crossings, lane, &q);
  if (lane == 0) {
    end[i] = make_double2(px, py);
    dtheta[i] = dth;
    quarter[i] = q;
    ok[i] = good ? 1 : 0;
  }
}

// area-uniform initial state of every replica (replica r from seeds[r]); the draws are those of
// the host initialisation (rng.h), so the state equals it bit for bit
__global__ void k_init_random(int ntot, const int* rid, const ReplicaDesc* reps, const uint64_t* seeds,
                              const double* cdf, MeshDev mesh, float* x, float* y, float* th) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntot) return;
  const int r = rid[g];
  const tissue::InitDraw d = tissue::area_uniform_draw(seeds[r], g - reps[r].off, cdf, mesh.nf);
  const float2 a = mesh.uv[mesh.faces[3 * d.face]], b = mesh.uv[mesh.faces[3 * d.face + 1]],
               c = mesh.uv[mesh.faces[3 * d.face + 2]];
  tissue::barycentric_uv(a.x, a.y, b.x, b.y, c.x, c.y, d.r1, d.r2, &x[g], &y[g]);
  th[g] = d.th;
}

// per-step output stream: copies step t's UV position, 3-D position and neighbour count into the
// ring slot of its global step number g = ctl[1] + t + 1 when g is a multiple of `every`
__global__ void k_record(int ntot, const int* ctl, int t, int every, int depth, const float4* xycs, const float* r3x,
                         const float* r3y, const float* r3z, const int* nbr, float* ring, int* ring_nbr) {
  const long g = (long)ctl[1] + t + 1;
  if (g % every != 0) return;  // uniform over the grid
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ntot) return;
  const size_t slot = (size_t)((g / every) % depth);
  float* f = ring + slot * 5 * (size_t)ntot;
  const float4 q = xycs[i];
  f[i] = q.x;
  f[(size_t)ntot + i] = q.y;
  f[2 * (size_t)ntot + i] = r3x[i];
  f[3 * (size_t)ntot + i] = r3y[i];
  f[4 * (size_t)ntot + i] = r3z[i];
  ring_nbr[slot * (size_t)ntot + i] = nbr[i];
}

// the counts, mask words and list lengths of a set that holds the state with vertex ids vid
__global__ void k_clear_held(int ntot, const int* vid, const int* rid, int R, int nv, BucketSet bs) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntot) return;
  const int v = vid[g];
  const size_t r = rid[g];
  bs.count[r * nv + v] = 0;
  bs.occ[r * occ_words(nv) + (v >> 5)] = 0u;
  if (g < R) {
    bs.ovf_n[g] = 0;
    bs.big_n[g] = 0;
  }
}

__global__ void k_locate(MeshDev mesh, int n, const float4* xycs, int* vid, int* face, float* r3x, float* r3y,
                         float* r3z) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4 p = xycs[i];
  const Located L = locate<1>(mesh, (double)p.x, (double)p.y, 0);
  vid[i] = L.vid;
  if (face) face[i] = L.face;
  if (r3x) { r3x[i] = (float)L.X; r3y[i] = (float)L.Y; r3z[i] = (float)L.Z; }
}

__global__ void k_insert(int ntot, const int* vid, const int* rid, const ReplicaDesc* reps, int nv, BucketSet bs) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntot) return;
  const int r = rid[g];
  bucket_insert<true>(replica_out(bs, r, nv, reps[r].off), vid[g], g);
}

__global__ void k_neighbor_lists(MeshDev mesh, const ReplicaDesc* reps, const int* rid, int ntot, BucketSet bs,
                                 const int* vid, int cap, int* counts, int* cols) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntot) return;
  const int r = rid[g];
  const int off = reps[r].off;
  const float t_near = reps[r].prm.t_near;
  const BucketsIn b = replica_in(bs, r, mesh.nv, off);
  const int v = vid[g];
  int k = 0;
  for (int e = mesh.row_ptr[v]; e < mesh.row_ptr[v + 1]; ++e) {
    const int2 ent = mesh.nbr[e];
    if (__int_as_float(ent.y) > t_near) break;
    for_bucket(b, ent.x, [&](int j) {
      if (k < cap) cols[(size_t)g * cap + k] = j - off;
      ++k;
    });
  }
  counts[g] = k;
}

inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

}  // namespace

// one translation unit per layout of the sums and physical lanes (step_lanes.hip)
#define TISSUE_STEP_SHAPES(X) X(1, 1) X(2, 2) X(2, 4) X(4, 4) X(4, 8) X(8, 8) X(8, 16) X(16, 16) X(32, 32) X(64, 64)
#define X(L, P)                                                                                              \
  hipError_t launch_step_l##L##_p##P(int block, bool tape, bool wave, const MeshDev& mesh,                    \
                                     const ReplicaDesc* reps, const TileDesc* tiles, int n_tiles,             \
                                     const BucketSet& bin, const BucketSet& bout, const BucketSet& bclr,      \
                                     const TiledIO& io, hipStream_t st);
TISSUE_STEP_SHAPES(X)
#undef X

hipError_t launch_step_tiled(int lanes, int phys, int block, bool tape, bool wave, const MeshDev& mesh,
                             const ReplicaDesc* reps, const TileDesc* tiles, int n_tiles, const BucketSet& bin,
                             const BucketSet& bout, const BucketSet& bclr, const TiledIO& io, hipStream_t st) {
  if (block < 64 || block > kStepMaxBlock || block % 64 || n_tiles < 1 || mesh.nv >= kMaxVertices)
    return hipErrorInvalidValue;
#define X(L, P)                \
  if (lanes == L && phys == P) \
    return launch_step_l##L##_p##P(block, tape, wave, mesh, reps, tiles, n_tiles, bin, bout, bclr, io, st);
  TISSUE_STEP_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_bucket_finalize(int block, const ReplicaDesc* reps, const TileDesc* tiles, int n_tiles, int nv,
                                  int single_n, const BucketSet& bs, hipStream_t st) {
  if (single_n > 0) n_tiles = cdiv(single_n, block);
  hipLaunchKernelGGL(k_bucket_finalize, dim3(n_tiles), dim3(block), 0, st, reps, tiles, nv, single_n, bs);
  return hipGetLastError();
}

hipError_t launch_phi_tiles(int R, int steps, const int* tile_begin, int n_logical, int per_tile,
                            const OrderPartial* partial, const ReplicaDesc* reps, double* phi, int phi_stride,
                            int t_base, const RunEnd& end, hipStream_t st) {
  hipLaunchKernelGGL(k_phi_tiles, dim3(R * steps), dim3(kPhiBlock), 0, st, steps, tile_begin, n_logical, per_tile,
                     partial, reps, phi, phi_stride, t_base, R, end);
  return hipGetLastError();
}

hipError_t launch_flags_begin(int R, const unsigned* halt, unsigned* rows, int* first_bad, hipStream_t st) {
  hipLaunchKernelGGL(k_flags_begin, dim3(cdiv(R, 64)), dim3(64), 0, st, R, halt, rows, first_bad);
  return hipGetLastError();
}

hipError_t launch_adopt(int n, const float* x, const float* y, const float* th, float4* xycs, float* th_out, float* vx,
                        float* vy, int* nbr, int R, unsigned* halt, hipStream_t st) {
  hipLaunchKernelGGL(k_adopt, dim3(cdiv(n, 256)), dim3(256), 0, st, n, x, y, th, xycs, th_out, vx, vy, nbr, R, halt);
  return hipGetLastError();
}

hipError_t launch_pack_state(int first, int n, const float4* xycs, const float* th, const int* vid, const PackAt& where,
                             float* out, hipStream_t st) {
  const bool all = where.at[0] >= 0 && where.at[1] >= 0 && where.at[2] >= 0 && where.at[3] >= 0;
  hipLaunchKernelGGL(all ? k_pack_state<true> : k_pack_state<false>, dim3(cdiv(n, 256)), dim3(256), 0, st, first, n, xycs,
                     th, vid, where, out);
  return hipGetLastError();
}

hipError_t launch_pack_outputs(int first, int n, const float* vx, const float* vy, const float* r3x, const float* r3y,
                               const float* r3z, const int* face, const int* nbr, const PackAt& where, float* out,
                               hipStream_t st) {
  const bool all = where.at[0] >= 0 && where.at[1] >= 0 && where.at[2] >= 0 && where.at[3] >= 0 && where.at[4] >= 0;
  hipLaunchKernelGGL(all ? k_pack_outputs<true> : k_pack_outputs<false>, dim3(cdiv(where.at[2] >= 0 ? 3l * n : n, 256)),
                     dim3(256), 0, st, first, n, vx, vy, r3x, r3y, r3z, face, nbr, where, out);
  return hipGetLastError();
}

hipError_t launch_fetch(size_t n, const float* from, float* to, hipStream_t st) {
  hipLaunchKernelGGL(k_fetch, dim3(cdiv((long)n, 256)), dim3(256), 0, st, n, from, to);
  return hipGetLastError();
}

hipError_t launch_clear_sets(int R, int nv, const BucketSet* sets, int n_sets, hipStream_t st) {
  const BucketSet &a = sets[0], &b = sets[n_sets > 1 ? 1 : 0], &c = sets[n_sets > 2 ? 2 : 0];
  hipLaunchKernelGGL(k_clear_sets, dim3(cdiv((long)R * nv, 256)), dim3(256), 0, st, (size_t)R * nv, (size_t)R * occ_words(nv),
                     R, a, b, c,
                     n_sets);
  return hipGetLastError();
}

hipError_t launch_locate(const MeshDev& mesh, int n, const float4* xycs, int* vid, int* face, float* r3x, float* r3y,
                         float* r3z, hipStream_t st) {
  hipLaunchKernelGGL(k_locate, dim3(cdiv(n, 256)), dim3(256), 0, st, mesh, n, xycs, vid, face, r3x, r3y, r3z);
  return hipGetLastError();
}

template <bool WAVE>
void launch_seam_wrap_mode(int lanes, dim3 grid, dim3 block, int n, const double2* start, double2* end, double* dtheta,
                           int* quarter, int* ok, int max_crossings, hipStream_t st) {
  switch (lanes) {
    case 1: hipLaunchKernelGGL((k_seam_wrap<1, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    case 2: hipLaunchKernelGGL((k_seam_wrap<2, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    case 4: hipLaunchKernelGGL((k_seam_wrap<4, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    case 8: hipLaunchKernelGGL((k_seam_wrap<8, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    case 16: hipLaunchKernelGGL((k_seam_wrap<16, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    case 32: hipLaunchKernelGGL((k_seam_wrap<32, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    case 64: hipLaunchKernelGGL((k_seam_wrap<64, WAVE>), grid, block, 0, st, n, start, end, dtheta, quarter, ok, max_crossings); break;
    default: break;
  }
}

hipError_t launch_seam_wrap(int lanes, int n, const double2* start, double2* end, double* dtheta, int* quarter, int* ok,
                            int max_crossings, int wave, hipStream_t st) {
  if (lanes < 1 || lanes > 64 || (lanes & (lanes - 1))) return hipErrorInvalidValue;
  const dim3 grid(cdiv(n * lanes, 256)), block(256);
  if (wave)
    launch_seam_wrap_mode<true>(lanes, grid, block, n, start, end, dtheta, quarter, ok, max_crossings, st);
  else
    launch_seam_wrap_mode<false>(lanes, grid, block, n, start, end, dtheta, quarter, ok, max_crossings, st);
  return hipGetLastError();
}

hipError_t launch_init_random(int ntot, const int* rid, const ReplicaDesc* reps, const uint64_t* seeds,
                              const double* cdf, const MeshDev& mesh, float* x, float* y, float* th, hipStream_t st) {
  hipLaunchKernelGGL(k_init_random, dim3(cdiv(ntot, 256)), dim3(256), 0, st, ntot, rid, reps, seeds, cdf, mesh, x, y, th);
  return hipGetLastError();
}

hipError_t launch_record(int ntot, const int* ctl, int t, int every, int depth, const float4* xycs, const float* r3x,
                         const float* r3y, const float* r3z, const int* nbr, float* ring, int* ring_nbr, hipStream_t st) {
  hipLaunchKernelGGL(k_record, dim3(cdiv(ntot, 256)), dim3(256), 0, st, ntot, ctl, t, every, depth, xycs, r3x, r3y,
                     r3z, nbr, ring, ring_nbr);
  return hipGetLastError();
}

hipError_t launch_clear_held(int ntot, const int* vid, const int* rid, int R, int nv, const BucketSet& bs,
                             hipStream_t st) {
  hipLaunchKernelGGL(k_clear_held, dim3(cdiv(ntot, 256)), dim3(256), 0, st, ntot, vid, rid, R, nv, bs);
  return hipGetLastError();
}

hipError_t launch_insert(int ntot, const int* vid, const int* rid, const ReplicaDesc* reps, int nv,
                         const BucketSet& bs, hipStream_t st) {
  hipLaunchKernelGGL(k_insert, dim3(cdiv(ntot, 256)), dim3(256), 0, st, ntot, vid, rid, reps, nv, bs);
  return hipGetLastError();
}

hipError_t launch_neighbor_lists(const MeshDev& mesh, const ReplicaDesc* reps, const int* rid, int ntot,
                                 const BucketSet& bs, const int* vid, int cap, int* counts, int* cols,
                                 hipStream_t st) {
  hipLaunchKernelGGL(k_neighbor_lists, dim3(cdiv(ntot, 256)), dim3(256), 0, st, mesh, reps, rid, ntot, bs, vid, cap,
                     counts, cols);
  return hipGetLastError();
}

}  // namespace tissue
