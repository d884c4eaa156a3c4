// gfx950 kernel of the tiled per-step update (one launch per step, all replicas at once).
//
// k_step_tiled<LANES, P>: each workgroup is a tile of one replica (TileDesc); P lanes of a wave64
// cooperate on one particle, whose sums are laid out over LANES lanes (particle_step). They stride over
// the particle's row of the truncated geodesic table (vertices within 2.4 sigma of its vertex, ascending
// in distance), visit the particles bucketed on those vertices, and reduce force, alignment sum and
// neighbour count with butterfly shuffles.
//
// The kernel is bound by chains of dependent loads (table row, bucket, particles; cell, candidates, face)
// and, where the chip is full, by instruction issue; never by bandwidth (2.9 TB/s at most), but for replicas with
// some 100 vertices per particle and more, where clearing the bucket sets is most of it. 2,000 particles 18.7 -> 10.1 us
// per step, 100,000 274 -> 66 (the first 50 steps of a run), 525,000 in 256 replicas 211 -> 150.
// Every lane then runs the per-particle epilogue (speed, Euler, heading, seam wrap) and the lanes
// split the point-location candidates of the face bucket. Lane 0 writes the SoA outputs, inserts
// the particle into next step's vertex buckets and contributes to the tile's order-parameter
// partials. A single system is the case of one replica.
#pragma once
#include <hip/hip_runtime.h>

#include <climits>

#include "launch.h"

namespace tissue {

using namespace tdev;

namespace {

// particle i into vertex v's bucket as its arrival number old (the value its add to b.count[v] returned)
template <bool OCC>
__device__ __forceinline__ void bucket_place(const BucketsOut& b, int v, int i, int old) {
  if (OCC && old == 0) atomicOr(&b.occ[v >> 5], 1u << (v & 31));
  if (old < kSlots) {
    b.slot[(size_t)v * kSlots + old] = i;
  } else {
    const int o = atomicAdd(b.ovf_n, 1);
    b.ovf[o] = make_int2(v, i);
  }
  if (b.multi) b.multi[i] = old == 1 ? v : -1;  // the second arrival has the bucket sorted
}

template <bool OCC>
__device__ __forceinline__ void bucket_insert(const BucketsOut& b, int v, int i) {
  bucket_place<OCC>(b, v, i, atomicAdd(&b.count[v], 1));
}

__device__ __forceinline__ BucketsOut replica_out(const BucketSet& s, int r, int nv, int off) {
  return {s.count + (size_t)r * nv, s.slot + (size_t)r * nv * kSlots, s.ovf_n + r, s.ovf + off, s.multi,
          s.occ + (size_t)r * occ_words(nv)};
}

// order parameters of one replica and step by one workgroup of kPhiBlock threads: the threads add the wave
// partials row[first .. last) in a strided split, then a wave and a workgroup sum (integer, so the split
// does not matter)
constexpr int kPhiBlock = 256;
__device__ __forceinline__ void block_phi(const OrderPartial* row, int first, int last, int n, double* out) {
  __shared__ long long s_cs[kPhiBlock / 64], s_sn[kPhiBlock / 64];
  __shared__ long s_sg[kPhiBlock / 64];
  long long cs = 0, sn = 0;
  long sg = 0;
  for (int b = first + (int)threadIdx.x; b < last; b += kPhiBlock) {
    const OrderPartial p = row[b];
    cs += p.cs;
    sn += p.sn;
    sg += p.sgn;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    cs += __shfl_xor(cs, off, 64);
    sn += __shfl_xor(sn, off, 64);
    sg += __shfl_xor(sg, off, 64);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { s_cs[wave] = cs; s_sn[wave] = sn; s_sg[wave] = sg; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kPhiBlock / 64; ++w) { cs += s_cs[w]; sn += s_sn[w]; sg += s_sg[w]; }
    const double c = (double)cs / kPhiScale, q = (double)sn / kPhiScale;
    out[0] = (1.0 / n) * fabs((double)sg);
    out[1] = sqrt(c * c + q * q) / n;
  }
}

}  // namespace

#ifdef TISSUE_STEP_KERNEL  // the kernel itself, for the translation units that instantiate it

namespace {

// the sum over the lanes 0, STRIDE, 2 STRIDE, .. of the wave (integers, so the order is free)
template <int STRIDE, int OFF = 32, class T>
__device__ __forceinline__ T strided_wave_sum(T v) {
  if constexpr (OFF >= STRIDE) {
    T a, b;
    butterfly<OFF, 64>(v, a, b);
    return strided_wave_sum<STRIDE, OFF / 2>(a + b);
  } else {
    return v;
  }
}

// the wave's sums of (sgn, cs, sn) in fixed point over the first lane of each group, written by its
// lane 0 to out: each wave keeps its own partial (no workgroup barrier, so a finished wave leaves at
// once); integer sums make the result independent of their order
template <int LANES>
__device__ __forceinline__ void wave_order_partial(int sgn, long long cs, long long sn, OrderPartial* out) {
  sgn = strided_wave_sum<LANES>(sgn);
  cs = strided_wave_sum<LANES>(cs);
  sn = strided_wave_sum<LANES>(sn);
  if ((threadIdx.x & 63) == 0) *out = OrderPartial{cs, sn, sgn, 0};
}

// words [lo, hi) at p zeroed by `width` threads, four at a time
__device__ __forceinline__ void clear_words(unsigned* p, int lo, int hi, int tid, int width) {
  typedef unsigned Four __attribute__((ext_vector_type(4), aligned(4)));
  int w = lo + 4 * tid;
  for (; w + 3 < hi; w += 4 * width) *reinterpret_cast<Four*>(p + w) = Four{0u, 0u, 0u, 0u};
  for (; w < hi; ++w) p[w] = 0u;
}

template <int LANES, int P, bool TAPE, bool OCC, bool VISITS, bool WAVE>
__global__ void __launch_bounds__(kStepMaxBlock) k_step_tiled(MeshDev mesh, const ReplicaDesc* __restrict__ reps,
                                                              const TileDesc* __restrict__ tiles, BucketSet bin, BucketSet bout,
                                                              BucketSet bclr, TiledIO io) {
  // the waves' walk areas (whole-wave walk), then with OCC occ_words(nv) words, the input buckets'
  // occupancy mask
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr bool kArea = wave_area(LANES, P, WAVE);
  WaveWalk* ww = kArea ? reinterpret_cast<WaveWalk*>(smem) + (threadIdx.x >> 6) : nullptr;
  unsigned* s_occ = reinterpret_cast<unsigned*>(smem + (kArea ? io.areas * sizeof(WaveWalk) : 0));
  const TileDesc tile = tiles[blockIdx.x];
  if (tile.r < 0) return;  // idle padding workgroup (whole block)
  const int r = tile.r;
  const ReplicaDesc& rep = reps[r];  // uniform: read through the scalar cache where used
  const int nv = mesh.nv, tid = threadIdx.x, nw = occ_words(nv);
  const int lane = tid & (P - 1);
  const int i = tile.first + tid / P;
  const bool active = i < rep.n;
  const bool wave_holds = __builtin_amdgcn_ballot_w64(active) != 0;  // (by all lanes: not behind a branch on active)
  const int g = rep.off + i;
  // the particle's inputs first: their loads are in flight during the set-up below
  float4 me = make_float4(0.f, 0.f, 0.f, 0.f);
  float th = 0.f, eta = 0.f;
  int v = 0;
  if (active) {
    me = io.xycs_in[g];
    th = io.th_in[g];
    v = io.vid_in[g];
    const size_t shift = io.noise_row0 ? (size_t)io.noise_row0[0] * io.noise_stride : 0;
    eta = io.noise ? io.noise[shift + g] : 0.0f;
  }
  if constexpr (OCC) {  // stage this replica's occupancy mask of the input buckets in LDS
    const unsigned* occ_in = bin.occ + (size_t)r * nw;
    for (int k = tid; k < nw; k += (int)blockDim.x) s_occ[k] = occ_in[k];
    __syncthreads();
  }
  // a replica flagged before this step passes its state through unchanged (the reference stops
  // at the first failure); the flag rows rotate like the bucket sets
  const unsigned halt = io.halt_in[r];
  if (tile.q == 0 && tid == 0) {
    bclr.ovf_n[r] = 0;
    bclr.big_n[r] = 0;
    io.halt_clr[r] = 0u;
    if (halt) atomicOr(&io.halt_out[r], halt);
  }
  const BucketsOut bo = replica_out(bout, r, nv, rep.off);

  int sgn = 0;
  long long pcs = 0, psn = 0;
  // a wave with an area needs all of its lanes where one holds a particle; waves past the last particle have no
  // area (step_areas) and do nothing
  if (active || (kArea && !halt && wave_holds)) {
    if (halt) {
      if (lane == 0) {
        io.xycs_out[g] = me;
        io.th_out[g] = th;
        io.vid_out[g] = v;
        bucket_insert<OCC>(bo, v, g);
        if constexpr (VISITS) io.visit[g] = make_int2(-1, 0);
      }
    } else {
      const GlobalSource<OCC, WAVE> src{replica_in(bin, r, nv, rep.off), io.xycs_in, io.th_in, s_occ};
      // the arrival counter is asked as soon as the new vertex is known: the answer comes while the heading's
      // sine and the outputs are written (asked with the rest of the insertion it was the wave's last wait:
      // 2,000 particles 10.75 -> 10.64 us per step, 525,000 in 256 replicas 151.2 -> 150.0 us)
      int arrival = 0;
      const auto arrive = [&](int vnew) __attribute__((always_inline)) {
        if (active && lane == 0) arrival = atomicAdd(&bo.count[vnew], 1);
      };
      const StepOut o = particle_step<LANES, P, WAVE, VISITS>(mesh, rep.prm, src, g, me, th, v, eta, lane, active, ww, arrive);
      if (active && lane == 0) {
        io.xycs_out[g] = make_float4(o.xo, o.yo, o.co, o.so);
        io.th_out[g] = o.to;
        io.vid_out[g] = o.L.vid;
        io.vx[g] = o.vx;
        io.vy[g] = o.vy;
        io.r3x[g] = (float)o.L.X;
        io.r3y[g] = (float)o.L.Y;
        io.r3z[g] = (float)o.L.Z;
        io.face[g] = o.L.face;
        io.nbr[g] = o.nb;  // count_particle_neighbors (2DTissue.cpp:254-268)
        bucket_place<OCC>(bo, o.L.vid, g, arrival);
        if (o.fl) {
          atomicOr(&io.halt_out[r], o.fl);
          atomicMin(&io.first_bad[r], io.step);
        }
        if constexpr (TAPE) {
          io.tape_fs[g] = make_float4(o.Fx, o.Fy, o.Sx, o.Sy);
          io.tape_q[g] = o.q;
        }
        if constexpr (VISITS) io.visit[g] = make_int2(o.na, (int)o.vh);
        sgn = o.sgn;
        pcs = __double2ll_rn((double)o.co * kPhiScale);
        psn = __double2ll_rn((double)o.so * kPhiScale);
      }
    }
  }
  // clear the tile's share of its replica's bucket set consumed two steps ago (it is next step's output); last, so
  // that no load of the step waits behind these stores, and four words a store: with 100 vertices per particle
  // they are 40 MB of a 40 us step, and word by word at its end cost 5 us of it
  clear_words(reinterpret_cast<unsigned*>(bclr.count) + (size_t)r * nv, tile.clr_lo, tile.clr_hi, tid, (int)blockDim.x);
  if constexpr (OCC) clear_words(bclr.occ + (size_t)r * nw, tile.clr_lo >> 5, occ_words(tile.clr_hi), tid, (int)blockDim.x);
  const int wpb = (int)blockDim.x >> 6;
  wave_order_partial<P>(sgn, pcs, psn, io.partial + (size_t)tile.logical * wpb + (tid >> 6));
}

template <int LANES, int P, bool OCC, bool WAVE>
void launch_tiled_mode(int block, bool tape, const MeshDev& mesh, const ReplicaDesc* reps, const TileDesc* tiles,
                       int n_tiles, const BucketSet& bin, const BucketSet& bout, const BucketSet& bclr,
                       const TiledIO& io, hipStream_t st) {
  const size_t lds = step_lds_bytes(mesh.nv, io.areas, LANES, P, WAVE, OCC);
  if (tape)
    hipLaunchKernelGGL((k_step_tiled<LANES, P, true, OCC, false, WAVE>), dim3(n_tiles), dim3(block), lds, st, mesh, reps,
                       tiles, bin, bout, bclr, io);
  else if (io.visit)  // the visit check: the same step, recording each particle's visited set
    hipLaunchKernelGGL((k_step_tiled<LANES, P, false, OCC, true, WAVE>), dim3(n_tiles), dim3(block), lds, st, mesh, reps,
                       tiles, bin, bout, bclr, io);
  else
    hipLaunchKernelGGL((k_step_tiled<LANES, P, false, OCC, false, WAVE>), dim3(n_tiles), dim3(block), lds, st, mesh, reps,
                       tiles, bin, bout, bclr, io);
}

// wave: crowded systems (sorted buckets, the seam-wrap loop of seam_wrap_group), compiled for up to 8
// lanes of the sums (the shapes such systems run at); wider shapes take the plain kernel (same results)
template <int LANES, int P, bool OCC>
void launch_tiled_variant(int block, bool tape, bool wave, const MeshDev& mesh, const ReplicaDesc* reps,
                          const TileDesc* tiles, int n_tiles, const BucketSet& bin, const BucketSet& bout,
                          const BucketSet& bclr, const TiledIO& io, hipStream_t st) {
  if constexpr (LANES <= 8) {
    if (wave) {
      launch_tiled_mode<LANES, P, OCC, true>(block, tape, mesh, reps, tiles, n_tiles, bin, bout, bclr, io, st);
      return;
    }
  }
  (void)wave;
  launch_tiled_mode<LANES, P, OCC, false>(block, tape, mesh, reps, tiles, n_tiles, bin, bout, bclr, io, st);
}

}  // namespace

#endif

}  // namespace tissue
