// Persistent, LDS-resident kernel: one workgroup runs one replica for many steps.
//
// Per workgroup the replica's state (x, y, cos, sin, theta, vertex id) and the step's vertex
// buckets live in LDS. Each step:
//   1. counting sort of the particles by vertex id into a CSR (LDS atomics + block scan);
//   2. every group of P lanes updates its particles with the shared particle_step (sums laid out over LANES
//      lanes; the geodesic-table rows and the mesh stay in L2). The update is Jacobi, every particle reads
//      the old state: the new one of a group's last particle stays in registers, that of its earlier ones
//      is staged in a global slice;
//   3. barrier, then the new states go to LDS and the last wave adds up the order parameters, which it
//      finishes beside the next step's update.
// Per step only the noise row is read from HBM and the order parameters written; the staged
// state stays in L2; the state goes back to its HBM home once per launch.
#include <hip/hip_runtime.h>

#include "launch.h"

using namespace tdev;

namespace tissue {

namespace {

// A shape's largest block, 512, means a full workgroup: 1,024 threads where their reduction words still fit
// beside the replica in LDS (the capacity is that of 512). A CU holds one such workgroup, and its
// steps are chains of loads and waits: 16 waves instead of 8 hide them better (MI355X, 100 steps: 256 x
// 200 particles 3.06 -> 2.27 ms, of which 0.2 ms is the transfer of states and outputs; 100 particles,
// 50 steps 0.92 -> 0.74 ms). The particles' results do not depend on the number of threads.
constexpr int kFullBlock = 1024;
constexpr size_t kLdsBytes = 160 * 1024;

__host__ __device__ inline size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

struct LdsLayout {
  size_t begin, xycs, th, vid, sorted, scan, red_cs, red_sn, red_sg, total;
  __host__ __device__ LdsLayout(int nv, int nmax, int waves) {
    size_t o = 0;
    begin = o; o = align16(o + 4 * (size_t)(nv + 1));
    xycs = o; o = align16(o + 16 * (size_t)nmax);
    th = o; o = align16(o + 4 * (size_t)nmax);
    vid = o; o = align16(o + 4 * (size_t)nmax);
    sorted = o; o = align16(o + 2 * (size_t)nmax);
    scan = o; o = align16(o + 4 * (size_t)waves);
    red_cs = o; o = align16(o + 8 * (size_t)waves);
    red_sn = o; o = align16(o + 8 * (size_t)waves);
    red_sg = o; o = align16(o + 4 * (size_t)waves);
    total = o;
  }
};

// exclusive sum over the workgroup's threads; every wave adds up the waves' totals for itself (one thread
// doing it was 16 LDS round trips with 15 waves waiting). tmp: a word per wave, free again after the
// caller's next barrier
__device__ uint32_t block_exclusive_scan(uint32_t x, uint32_t* tmp) {
  const int lane = threadIdx.x & 63, nw = (blockDim.x + 63) >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t inc = (uint32_t)wave_scan((int)x);
  if (lane == 63) tmp[wave] = inc;
  __syncthreads();
  const uint32_t mine = lane < nw ? tmp[lane] : 0u;
  const uint32_t before = (uint32_t)wave_scan((int)mine) - mine;
  return (uint32_t)__builtin_amdgcn_readlane((int)before, wave) + inc - x;
}

// a value the compiler does not know to be the same in every step: what is derived from it is computed where
// it is used instead of being kept (spilled) across the update
__device__ __forceinline__ int in_step(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// the counts begin[0 .. nv) to inclusive sums, N consecutive vertices per thread in registers
template <int N>
__device__ __forceinline__ void scan_counts(uint32_t* begin, int nv, int chunk, uint32_t* tmp) {
  const int lo = in_step((int)threadIdx.x) * chunk, len = min(chunk, nv - lo);
  uint32_t c[N];
#pragma unroll
  for (int k = 0; k < N; ++k) c[k] = begin[min(lo + k, nv)];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    sum += k < len ? c[k] : 0u;
    c[k] = sum;
  }
  const uint32_t excl = block_exclusive_scan(sum, tmp);
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (k < len) begin[lo + k] = c[k] + excl;
}

// counting sort of particles by vertex: afterwards begin[v] .. begin[v+1] lists the particles on
// vertex v (begin[nv] = n). begin: zeroed
__device__ void build_buckets(uint32_t* begin, uint16_t* sorted, const int* vid, int n, int nv, uint32_t* tmp) {
  const int tid = threadIdx.x, nthr = blockDim.x;
  for (int i = tid; i < n; i += nthr) atomicAdd(&begin[vid[i]], 1u);
  __syncthreads();
  const int chunk = (nv + nthr - 1) / nthr;
  if (chunk <= 8) {
    scan_counts<8>(begin, nv, chunk, tmp);
  } else if (chunk <= 16) {
    scan_counts<16>(begin, nv, chunk, tmp);
  } else {
    const int lo = min(tid * chunk, nv), hi = min(lo + chunk, nv);
    uint32_t sum = 0;
    for (int v = lo; v < hi; ++v) {
      sum += begin[v];
      begin[v] = sum;
    }
    const uint32_t excl = block_exclusive_scan(sum, tmp);
    for (int v = lo; v < hi; ++v) begin[v] += excl;
  }
  __syncthreads();
  for (int i = tid; i < n; i += nthr) {
    const uint32_t p = atomicSub(&begin[vid[i]], 1u) - 1u;
    sorted[p] = (uint16_t)i;
  }
  if (tid == 0) begin[nv] = (uint32_t)n;
  __syncthreads();
}

__device__ __forceinline__ double lane_double(double v, int l) {
  uint32_t w[2];
  __builtin_memcpy(w, &v, sizeof v);
  w[0] = __builtin_amdgcn_readlane(w[0], l);
  w[1] = __builtin_amdgcn_readlane(w[1], l);
  __builtin_memcpy(&v, w, sizeof v);
  return v;
}

// What bounds a step: one workgroup's chain of barriers and dependent loads, the CU's other resources idle.
// Hence nothing serial stands between two barriers: the new state of a group's last particle stays in
// registers until the old one has been read (only earlier passes go through global memory), begin is
// cleared where the state is copied, and the order parameters are added up by the last wave, with all its
// reads in flight, and finished by it beside the next step's update (100 particles, 50 steps 0.705 -> 0.660 ms;
// 256 x 200 particles, 100 steps 1.97 -> 1.83 ms).
template <int LANES, int P>
__global__ void __launch_bounds__(kFullBlock) k_resident(MeshDev mesh, const ReplicaDesc* __restrict__ reps, int nmax, int steps,
                                                        ResidentIO io) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ unsigned s_flags;
  const LdsLayout L(mesh.nv, nmax, (int)blockDim.x >> 6);
  double* red_cs = (double*)(smem + L.red_cs);
  double* red_sn = (double*)(smem + L.red_sn);
  int* red_sg = (int*)(smem + L.red_sg);
  uint32_t* begin = (uint32_t*)(smem + L.begin);
  float4* xycs = (float4*)(smem + L.xycs);
  float* th = (float*)(smem + L.th);
  int* vid = (int*)(smem + L.vid);
  uint16_t* sorted = (uint16_t*)(smem + L.sorted);
  uint32_t* scan_tmp = (uint32_t*)(smem + L.scan);

  const int r = blockIdx.x;
  const ReplicaDesc& rep = reps[r];
  const int n = rep.n, off = rep.off;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lane = tid & (P - 1), group = tid / P, ngroups = nthr / P;
  float4* nxt_xycs = io.stage_xycs + off;
  float* nxt_th = io.stage_th + off;
  int* nxt_vid = io.stage_vid + off;

  for (int i = tid; i < n; i += nthr) {
    xycs[i] = io.xycs[off + i];
    th[i] = io.th[off + i];
    vid[i] = io.vid[off + i];
  }
  for (int v = tid; v <= mesh.nv; v += nthr) begin[v] = 0u;
  if (tid == 0) s_flags = io.flags_in[r];
  __syncthreads();

  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = (nthr + 63) >> 6;
  // the sums of the step before (in the last wave, one value a wave), and where its order parameters go
  double sum_cs = 0.0, sum_sn = 0.0;
  int sum_sg = 0;
  double* last_phi = nullptr;
  auto finish_phi = [&]() __attribute__((always_inline)) {
    if (last_phi && wave == nw - 1 && (tid & 63) == 0) {
      last_phi[0] = (1.0 / n) * fabs((double)sum_sg);
      last_phi[1] = sqrt(sum_cs * sum_cs + sum_sn * sum_sn) / n;
    }
    last_phi = nullptr;
  };

  const LdsSource src{begin, sorted, xycs, th};
  for (int s = 0; s < steps; ++s) {
    const int t = io.t_base + s;
    double* phi = io.phi + 2 * ((size_t)r * io.phi_stride + t);
    if (s_flags != 0u) {  // a failed step stops the replica (the reference stops at the first failure)
      finish_phi();
      if (tid == 0) { phi[0] = 0.0; phi[1] = 0.0; }
      continue;
    }
    build_buckets(begin, sorted, vid, n, mesh.nv, scan_tmp);
    const size_t row = (size_t)s + (io.noise_row0 ? (size_t)io.noise_row0[0] : 0);
    const float* eta_row = io.noise ? io.noise + row * io.noise_stride + off : nullptr;
    int sgn = 0;
    double cs = 0.0, sn = 0.0;
    unsigned fl = 0;
    finish_phi();
    // the update is Jacobi, every particle must read the old state of its neighbours: the new state of a
    // group's last particle is held in registers, that of its earlier ones staged in global memory (this
    // workgroup's slice, L2-resident)
    float4 held_xycs = make_float4(0.f, 0.f, 0.f, 0.f);
    float held_th = 0.f;
    int held_vid = 0, held = -1;
    for (int i = group; i < n; i += ngroups) {
      if (held >= 0) {
        nxt_xycs[held] = held_xycs;
        nxt_th[held] = held_th;
        nxt_vid[held] = held_vid;
      }
      const float eta = eta_row ? eta_row[i] : 0.0f;
      const StepOut o = particle_step<LANES, P>(mesh, rep.prm, src, i, xycs[i], th[i], vid[i], eta, lane);
      if (lane == 0) {
        held = i;
        held_xycs = make_float4(o.xo, o.yo, o.co, o.so);
        held_th = o.to;
        held_vid = o.L.vid;
        sgn += o.sgn;
        cs += (double)o.co;
        sn += (double)o.so;
        fl |= o.fl;
        if (s == steps - 1) {
          const int g = off + i;
          io.vx[g] = o.vx; io.vy[g] = o.vy;
          io.r3x[g] = (float)o.L.X; io.r3y[g] = (float)o.L.Y; io.r3z[g] = (float)o.L.Z;
          io.face[g] = o.L.face;
          io.nbr[g] = o.nb;
        }
      }
    }
    if (fl) {
      atomicOr(&s_flags, fl);
      atomicMin(&io.first_bad[r], t);
    }
    // order parameters of the step: butterfly per wave, waves summed in order below
    sgn = group_sum<64>(sgn);
    cs = group_sum<64>(cs);
    sn = group_sum<64>(sn);
    if ((tid & 63) == 0) { red_cs[wave] = cs; red_sn[wave] = sn; red_sg[wave] = sgn; }
    __syncthreads();  // all reads of the old state done; the staged state is visible to the workgroup
    if (held >= 0) {
      xycs[held] = held_xycs;
      th[held] = held_th;
      vid[held] = held_vid;
    }
    for (int i = tid; i < n - ngroups; i += nthr) {
      xycs[i] = nxt_xycs[i];
      th[i] = nxt_th[i];
      vid[i] = nxt_vid[i];
    }
    for (int v = tid; v <= mesh.nv; v += nthr) begin[v] = 0u;
    if (wave == nw - 1) {  // the waves' sums in order, the cosines on lane 0 and the sines on lane 1
      static_assert(kFullBlock <= 16 * 64, "waves of a workgroup");
      const int l = in_step(tid) & 63, waves = __builtin_amdgcn_readfirstlane(in_step(nw));
      const double* part = l == 0 ? red_cs : red_sn;
      const int g = l < waves ? red_sg[l] : 0;
      double v[16], sum = 0.0;
#pragma unroll
      for (int w = 0; w < 16; ++w) v[w] = part[w < waves ? w : 0];
#pragma unroll
      for (int w = 0; w < 16; ++w) sum += w < waves ? v[w] : 0.0;
      sum_cs = lane_double(sum, 0);
      sum_sn = lane_double(sum, 1);
      sum_sg = __builtin_amdgcn_readfirstlane(group_sum<64>(g));
    }
    last_phi = phi;
    __syncthreads();
  }
  finish_phi();

  for (int i = tid; i < n; i += nthr) {
    io.xycs[off + i] = xycs[i];
    io.th[off + i] = th[i];
    io.vid[off + i] = vid[i];
  }
  if (tid == 0) {
    io.flags_out[r] = s_flags;
    // (first_bad[r] is this workgroup's alone; atomic, as its other threads' updates were)
    if (io.end.halt) end_run(io.end, (int)gridDim.x, r, s_flags, atomicAdd(&io.first_bad[r], 0));
  }
}

template <int LANES, int P>
hipError_t launch_one(int block, const MeshDev& mesh, const ReplicaDesc* reps, int R, int nmax, int steps,
                      const ResidentIO& io, hipStream_t st) {
  const size_t lds = LdsLayout(mesh.nv, nmax, block / 64).total;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  hipError_t e = hipStreamIsCapturing(st, &cap);
  if (e != hipSuccess) return e;
  if (cap == hipStreamCaptureStatusNone) {  // under capture the attribute was set by resident_prepare
    e = hipFuncSetAttribute((const void*)k_resident<LANES, P>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_resident<LANES, P>), dim3(R), dim3(block), lds, st, mesh, reps, nmax, steps, io);
  return hipGetLastError();
}

}  // namespace

size_t resident_lds_bytes(int nv, int nmax) {
  return LdsLayout(nv, nmax, kResidentMaxBlock / 64).total + 16;
}

// threads of a workgroup for the shape's block
static int resident_threads(int nv, int nmax, int block) {
  return block == kResidentMaxBlock && LdsLayout(nv, nmax, kFullBlock / 64).total + 16 <= kLdsBytes ? kFullBlock : block;
}

int resident_max_particles(int nv) {
  int lo = 0, hi = 65535;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (resident_lds_bytes(nv, mid) <= kLdsBytes) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

hipError_t resident_prepare(int nv, int nmax) {
  const int lds = (int)LdsLayout(nv, nmax, resident_threads(nv, nmax, kResidentMaxBlock) / 64).total;
  const void* fns[] = {(const void*)k_resident<1, 1>, (const void*)k_resident<2, 2>, (const void*)k_resident<4, 4>,
                       (const void*)k_resident<8, 8>, (const void*)k_resident<8, 4>};
  for (const void* f : fns) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_resident(int lanes, int block, const MeshDev& mesh, const ReplicaDesc* reps, int R, int nmax,
                           int steps, const ResidentIO& io, hipStream_t st) {
  if (block < 64 || block > kResidentMaxBlock || block % 64 || nmax > resident_max_particles(mesh.nv)) return hipErrorInvalidValue;
  block = resident_threads(mesh.nv, nmax, block);
  switch (lanes) {
    case 1: return launch_one<1, 1>(block, mesh, reps, R, nmax, steps, io, st);
    case 2: return launch_one<2, 2>(block, mesh, reps, R, nmax, steps, io, st);
    case 4: return launch_one<4, 4>(block, mesh, reps, R, nmax, steps, io, st);
    case 8:
      // four lanes, two strands each, where eight take more than one pass over the replica (256 replicas
      // x 100 steps: 200 particles 2.20 -> 1.96 ms, 256 particles 3.03 -> 2.66 ms); where eight fit in one
      // pass four are slower (100 particles, 100 steps 1.21 -> 1.31 ms, 256 x 100 particles 1.51 -> 1.72 ms)
      if (nmax * 8 > block) return launch_one<8, 4>(block, mesh, reps, R, nmax, steps, io, st);
      return launch_one<8, 8>(block, mesh, reps, R, nmax, steps, io, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tissue
