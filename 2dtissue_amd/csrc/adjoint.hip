// Reverse pass of the step (gfx950), through the forward's frozen decisions.
//
// Step t maps the state (r_i, theta_i) to
//   p_i      = r_i + dt s_i e_i,  e_i = (cos theta_i, sin theta_i),  s_i = v0 + mu |F_i|,
//   F_i      = sum_{j in A_i, j != i} c_ij (r_i - r_j),    c_ij = f(d~_ij) / d~_ij  (frozen d_ij),
//   r_i'     = R_i p_i + b_i                                (seam wrap: rotation by q_i quarter turns),
//   theta_i' = theta_i + rho wrap(atan2(S_i, C_i) - theta_i) + eta_i + const,  rho = dt / tau,
//   S_i, C_i = sum_{j in A_i} (sin, cos) theta_j            (A_i includes i),
// and adds w_v |rdot_i - u(r_i)|^2 to the loss (w_v = w_velocity / (T n)).
// Its adjoint, for incoming (lr_i, lt_i) of the new state:
//   lp = R_i^T lr;  lrdot = dt lp + 2 w_v (rdot - u);  ls = lrdot . e;  lF = mu ls F / |F|;
//   lr_i  = lp - 2 w_v J_u^T (rdot - u) + sum_{j in A_i, j != i} c_ij (lF_i - lF_j);
//   lS_i  = rho lt_i C_i / Q_i,  lC_i = -rho lt_i S_i / Q_i,  Q_i = C_i^2 + S_i^2;
//   lt_i  = (1 - rho) lt_i + s_i lrdot . (-sin, cos) + cos theta_i sum_{j in A_i} lS_j - sin theta_i sum_{j in A_i} lC_j.
// The neighbour relation is symmetric (the geodesic table is min-symmetrised), so the transposed
// sums are gathers over the particle's own neighbour set, along the same geodesic rows and vertex
// buckets as the forward step. A particle's factors of step t (lF, lS, lC, what its neighbours gather)
// follow from its own adjoint of the new state alone, so one kernel does the gather of step t and the
// factors of step t - 1 (k_adj_reverse, kBoth); the first step's factors and the last step's gather
// run by themselves (kFactors, kGather), and so does every step where a segment's tape is recomputed.
// The adjoint state of replica r is held as lambda * 2^-E_r (FP32, E_r >= 0 in sexp[r]): the map
// is linear in lambda, so only the loss sources are scaled by 2^-E_r and the FP64 parameter
// accumulators by 2^E_r. E_r is raised whenever |lambda| outgrows 2^20: the gather records each
// replica's max |lambda| (one atomic per wave), and the next factors are scaled by the matching power
// of two and carry E_r forward (the first ones by the seeds' max). In kBoth the factors follow in the same
// kernel, before that max is complete, so they go by the max of the step before, less the scaling it has
// caused already: |lambda| then reaches 2^21 times the growth of two steps where by kFactors it reaches 2^21
// times that of one, so FP32 holds growths below 2^53 a step instead of 2^106 (and large velocity weights,
// which nothing scales before the first max, times one more step's growth). An adjoint that leaves FP32 stays
// non-finite back to the initial state, where a particle's own terms carry it; the engine then takes the pass
// again by kFactors and kGather alone. The scaling is exact either way, so both give the same gradients (but
// for values 2^-126 below their replica's largest, which underflow in one or the other). (Slots alternate by
// step, so that no kernel reads one that another thread of it writes.)
#include <hip/hip_runtime.h>

#include "adjoint.h"

using namespace tdev;

namespace tissue {

namespace {

// the target field u and its Jacobian at (x, y), by a group of G lanes: each lane evaluates one mode at a
// time, and all add the modes in order
struct Field { float ux, uy, jxx, jxy, jyx, jyy; };

template <int G>
__device__ __forceinline__ Field field_eval(const LossDev& L, float x, float y, int lane) {
  Field f{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int m0 = 0; m0 < L.n_modes; m0 += G) {
    const int m = min(m0 + lane, L.n_modes - 1);
    const float kx = L.kx[m], ky = L.ky[m], amp = L.amp[m];
    float s, c;
    sincosf(kx * x + ky * y + L.phase[m], &s, &c);
    const float v = amp * s, d = amp * c, dx = d * kx, dy = d * ky;
#pragma unroll
    for (int l = 0; l < G; ++l) {
      if (m0 + l >= L.n_modes) break;  // uniform
      const float vl = G == 1 ? v : __shfl(v, l, G), xl = G == 1 ? dx : __shfl(dx, l, G), yl = G == 1 ? dy : __shfl(dy, l, G);
      if (L.comp[m0 + l] == 0) { f.ux += vl; f.jxx += xl; f.jxy += yl; }
      else { f.uy += vl; f.jyx += xl; f.jyy += yl; }
    }
  }
  return f;
}

// R_q^T v for a rotation by q counter-clockwise quarter turns
__device__ __forceinline__ float2 rot_t(int q, float2 v) {
  switch (q & 3) {
    case 1: return make_float2(v.y, -v.x);
    case 2: return make_float2(-v.x, -v.y);
    case 3: return make_float2(-v.y, v.x);
    default: return v;
  }
}

// deterministic FP64 sum over a block (wave butterflies, waves added in order)
__device__ double block_sum(double v, double* tmp) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) tmp[wave] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < nw; ++w) s += tmp[w];
  return s;
}

// one block per replica: polar order of the final state and the seeds of the heading adjoint
// (mx: their largest, float bits)
__global__ void k_adj_seed(const ReplicaDesc* reps, const float4* xycs, LossDev L, const unsigned* halt, float2* lr,
                           float* lt, double* out, unsigned* mx) {
  __shared__ double tmp[kAdjBlock / 64];
  __shared__ unsigned s_mx;
  if (threadIdx.x == 0) s_mx = 0u;
  const int r = blockIdx.x;
  const int off = reps[r].off, n = reps[r].n;
  double cx = 0.0, cy = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float4 q = xycs[off + i];
    cx += (double)q.z;
    cy += (double)q.w;
  }
  const double Px = block_sum(cx, tmp);
  const double Py = block_sum(cy, tmp);
  const double norm = sqrt(Px * Px + Py * Py);
  const double phi = norm / n;
  const bool ok = halt[r] == 0u;
  // d phi / d theta_i = (-Px sin theta_i + Py cos theta_i) / (n |P|)
  const double coef = (ok && norm > 0.0) ? L.w_order * 2.0 * (phi - L.target) / (n * norm) : 0.0;
  float largest = 0.f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float4 q = xycs[off + i];
    const float l = (float)(coef * (-Px * (double)q.w + Py * (double)q.z));
    lr[off + i] = make_float2(0.f, 0.f);
    lt[off + i] = l;
    largest = fmaxf(largest, fabsf(l));
  }
  atomicMax(&s_mx, __float_as_uint(largest));
  __syncthreads();
  if (threadIdx.x == 0) {
    mx[r] = s_mx;
    out[2 * r] = phi;
    out[2 * r + 1] = L.w_order * (phi - L.target) * (phi - L.target);
  }
}

// power-of-two exponent that brings a replica's max |lambda| (float bits of a non-negative value),
// already scaled down by 2^-done, below 2^21; 0 when no rescale is needed or the max is not finite
__device__ __forceinline__ int rescale_exponent(unsigned mx_bits, int done) {
  const float mx = __uint_as_float(mx_bits);
  if (!(mx > 0.f) || !isfinite(mx)) return 0;
  const int s = ilogbf(mx) - done - 20;
  return s > 0 ? s : 0;
}

// particle j's factors of step t's reverse, from its tape entry and its incoming adjoint (scaled
// by 2^-E, then by down = 2^-s_up): the factors its neighbours gather, its own terms of the new
// adjoint, and what the accumulators take.
struct AdjLocal {
  float2 lF, lsc;          // d loss / d F, (d loss / d sum sin, d loss / d sum cos)
  float lrx, lry, lth;     // the particle's own terms of the new adjoint
  float ls, m, ltn, wv, dvx, dvy;
};

__device__ __forceinline__ AdjLocal adj_local(const StepParams& prm, const LossDev& L, const Field& u, int n_r,
                                              float down, float src, float4 me, float4 f, int quarter, float2 lr_s,
                                              float lt_s) {
  AdjLocal o;
  const float2 lp = rot_t(quarter, make_float2(lr_s.x * down, lr_s.y * down));
  o.ltn = lt_s * down;
  o.m = sqrtf(f.x * f.x + f.y * f.y);
  const float s = prm.v0 + prm.mu * o.m;
  const float rdx = me.z * s, rdy = me.w * s;
  o.wv = L.w_velocity / ((float)L.n_steps * (float)n_r);
  o.dvx = rdx - u.ux;
  o.dvy = rdy - u.uy;
  const float sw = 2.f * o.wv * src;
  const float lrdx = prm.dt * lp.x + sw * o.dvx, lrdy = prm.dt * lp.y + sw * o.dvy;
  o.lrx = lp.x - sw * (u.jxx * o.dvx + u.jyx * o.dvy);
  o.lry = lp.y - sw * (u.jxy * o.dvx + u.jyy * o.dvy);
  o.ls = lrdx * me.z + lrdy * me.w;
  const float lm = prm.mu * o.ls;
  o.lF = o.m > 0.f ? make_float2(lm * f.x / o.m, lm * f.y / o.m) : make_float2(0.f, 0.f);
  const float Q = f.z * f.z + f.w * f.w;
  const float lmean = prm.rate * o.ltn;
  o.lsc = Q > 0.f ? make_float2(lmean * f.z / Q, -lmean * f.w / Q) : make_float2(0.f, 0.f);
  o.lth = (1.f - prm.rate) * o.ltn + s * (-lrdx * me.w + lrdy * me.z);
  return o;
}

// the turn towards the mean heading, wrapped
__device__ __forceinline__ double mean_turn(float4 f, float theta) {
  double delta = atan2((double)f.w, (double)f.z) - (double)theta;
  if (delta > kPi) delta -= 2.0 * kPi;
  else if (delta <= -kPi) delta += 2.0 * kPi;
  return delta;
}

// parameter gradients and the velocity loss of particle g, accumulated in FP64 (true units); sum: the
// accumulators as they stand, loaded early
__device__ __forceinline__ void adj_accumulate(const StepParams& prm, const AdjLocal& o, float4 f, double delta,
                                               double unscale, const double (&sum)[kAdjAcc], double* acc, size_t ntot,
                                               int g) {
  const double tau = prm.dt64 / prm.rate64;
  acc[g] = sum[0] + unscale * (double)o.ls;                                            // d v0
  acc[ntot + g] = sum[1] + unscale * (double)o.ls * (double)o.m;                       // d mu
  if (prm.k64 != 0.0)                                                          // d k
    acc[2 * ntot + g] = sum[2] + unscale * ((double)o.lF.x * f.x + (double)o.lF.y * f.y) / prm.k64;
  acc[3 * ntot + g] = sum[3] + unscale * (double)o.ltn * delta * (-prm.dt64 / (tau * tau));  // d tau
  acc[4 * ntot + g] = sum[4] + (double)o.wv * ((double)o.dvx * o.dvx + (double)o.dvy * o.dvy);  // loss
}

// each replica's max |lambda| over the wave: the wave's particles of one replica occupy a
// contiguous range of lanes, so an inclusive max-scan restricted to that range leaves the max on
// its last lane, which posts it (float bits of non-negative values order like the values;
// replicas are concatenated, so r never decreases along the wave). Every lane of the wave calls it.
__device__ __forceinline__ void post_replica_max(int r, float mx, unsigned* mx_out) {
  const int me_lane = (int)__lane_id();
  const int r_prev = __shfl_up(r, 1, 64), r_next = __shfl_down(r, 1, 64);
  const unsigned long long heads = __ballot(me_lane == 0 || r_prev != r);
  const unsigned long long upto = me_lane == 63 ? ~0ull : (2ull << me_lane) - 1ull;
  const int first = 63 - __clzll(heads & upto);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float up = __shfl_up(mx, o, 64);
    if (me_lane - o >= first) mx = fmaxf(mx, up);
  }
  if ((me_lane == 63 || r_next != r) && r >= 0 && mx > 0.f) atomicMax(&mx_out[r], __float_as_uint(mx));
}

// One particle's G lanes. PART: kFactors (step p's factors from lr_in, lt_in), kGather (step q's gather to
// lr_out, lt_out) or kBoth (step q's gather, then step p = q - 1's factors from it). The gather's sums
// are laid out over the G lanes like the step's (lane l adds entries l, l + G, .. of the row). A chain
// of dependent loads (vertex, row, entries, bucket heads, factors) on few waves: entries and heads are
// loaded side by side from clamped addresses, a neighbour's four factors in one load, and what needs
// no neighbour (the field, the accumulators' arc tangent) runs between the chain's first loads. With
// use_occ the occupancy mask, a bit per vertex, is asked first: on a large mesh the counts and slots of
// the mostly empty rows of sparse replicas are some 500 MB of lines a step (64 x 2,000 particles on
// 100,265 vertices), the masks stay in the L2s.
template <int G, int PART>
__global__ void __launch_bounds__(256) k_adj_reverse(MeshDev mesh, const ReplicaDesc* __restrict__ reps,
                                                    const int* __restrict__ rid, int ntot, LossDev L, RevStep a) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int g = tid / G, lane = tid & (G - 1);
  const int gc = min(g, ntot - 1);
  // every load that needs no other first, then the row's bounds
  int r = a.single ? 0 : rid[gc];
  int v = 0;
  float4 mine, me, pt, me_p, f = make_float4(0.f, 0.f, 0.f, 0.f);  // f: step p's (Fx, Fy, sum cos, sum sin)
  float th_p = 0.f;
  int quarter = 0;
  // the accumulators: with wide groups (few waves) loaded first, so that nothing waits for them at the
  // end (1,000 particles 10.6 -> 9.7 us a step); with narrow ones (64 x 2,000) that delays the chain's
  // own loads (2 %)
  double sum[kAdjAcc] = {};
  auto load_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kAdjAcc; ++k) sum[k] = a.acc[(size_t)k * ntot + gc];
  };
  if constexpr (PART != kFactors) {
    v = a.vid_q[gc];
    mine = a.g4_in[gc];
    me = a.xycs_q[gc];
    pt = a.part_in[gc];
  }
  if constexpr (PART != kGather) {
    me_p = a.xycs_p[gc];
    f = a.fs_p[gc];
    th_p = a.th_p[gc];
    quarter = a.quarter_p[gc];
    if constexpr (G >= 8) load_sums();
  }
  int rs = 0, re = 0;
  if constexpr (PART != kFactors) {
    rs = load_at(mesh.row_ptr, v);
    re = load_at(mesh.row_ptr, v + 1);
  }
  const ReplicaDesc& rep = reps[r];
  const bool halted = a.halt[r] != 0u;
  if (g >= ntot) r = -1;  // past the end (the lanes stay for the wave reduction)
  float mx = 0.f;         // |lambda| of this particle (on lane 0 of its group)
  if (r >= 0) {
    const StepParams& prm = rep.prm;
    // the scaling of this launch's factors; the replica's first particle carries the exponent forward
    // and clears the max slot of the next launch
    int s_up = 0, E = 0;
    if constexpr (PART != kGather) {
      s_up = rescale_exponent(a.mx_in[r], PART == kBoth ? a.sup_in[r] : 0);
      E = a.sexp_in[r] + s_up;
      if (g == rep.off && lane == 0) {
        a.sexp_out[r] = E;
        a.sup_out[r] = s_up;
        a.mx_clear[r] = 0u;
      }
    }
    float2 lr = make_float2(0.f, 0.f);
    float lt = 0.f;
    Field u{};
    double delta = 0.0;
    if constexpr (PART == kFactors) {
      lr = a.lr_in[g];
      lt = a.lt_in[g];
      u = field_eval<G>(L, me_p.x, me_p.y, lane);
      delta = mean_turn(f, th_p);
    } else if (!halted) {
      const int nv = mesh.nv;
      const BucketsIn b = replica_in(a.bs, r, nv, rep.off);
      if constexpr (PART == kBoth) u = field_eval<G>(L, me_p.x, me_p.y, lane);
      float ax = 0.f, ay = 0.f, aS = 0.f, aC = 0.f;
      auto add = [&](float c, int j, const float4& o) __attribute__((always_inline)) {
        if (j != g) {
          ax += c * (mine.x - o.x);
          ay += c * (mine.y - o.y);
        }
        aS += o.z;
        aC += o.w;
      };
      constexpr int kChunk = G >= 8 ? 2 : 4;
      int2 ent[kChunk];
      auto load_entries = [&](int base) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          const int e = base + k * G;
          ent[k] = table_entry(mesh.nbr, min(e, re - 1));
          if (e >= re) ent[k].y = 0x7f800000;
        }
      };
      int base = rs + lane;
      load_entries(base);
      if constexpr (PART == kBoth) delta = mean_turn(f, th_p);
      for (;;) {
        int c[kChunk];
        int2 s[kChunk];
        bool want[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) want[k] = __int_as_float(ent[k].y) <= prm.t_near;
        if (a.use_occ) {  // uniform
          const unsigned* occ = a.bs.occ + (size_t)r * occ_words(nv);
          unsigned word[kChunk];
#pragma unroll
          for (int k = 0; k < kChunk; ++k) word[k] = load_at(occ, (want[k] ? ent[k].x : 0) >> 5);
#pragma unroll
          for (int k = 0; k < kChunk; ++k) want[k] = want[k] && ((word[k] >> (ent[k].x & 31)) & 1u) != 0u;
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          const int w = want[k] ? ent[k].x : 0;
          c[k] = load_at(b.count, w);
          s[k] = load_at(reinterpret_cast<const int2*>(b.slot), w * (kSlots / 2));
        }
        // the first two particles of every entry, side by side
        float4 o0[kChunk], o1[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          if (!want[k]) c[k] = 0;
          if (c[k] == 2 && !b.sorted && s[k].x > s[k].y) s[k] = make_int2(s[k].y, s[k].x);
          o0[k] = load_at(a.g4_in, c[k] == 1 || c[k] == 2 ? s[k].x : 0);
          o1[k] = load_at(a.g4_in, c[k] == 2 ? s[k].y : 0);
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          if (c[k] == 0) continue;
          const float co = pair_coef(__int_as_float(ent[k].y), prm);
          if (c[k] <= 2) {
            add(co, s[k].x, o0[k]);
            if (c[k] == 2) add(co, s[k].y, o1[k]);
          } else {
            for_bucket(b, ent[k].x, [&](int j) { add(co, j, load_at(a.g4_in, j)); });
          }
        }
        if (__int_as_float(ent[kChunk - 1].y) > prm.t_near) break;  // rows ascend in distance
        base += kChunk * G;
        load_entries(base);
      }
      ax = group_sum<G>(ax);
      ay = group_sum<G>(ay);
      aS = group_sum<G>(aS);
      aC = group_sum<G>(aC);
      lr = make_float2(pt.x + ax, pt.y + ay);
      lt = pt.z + me.z * aS - me.w * aC;
      if (lane == 0) mx = fmaxf(fabsf(lr.x), fmaxf(fabsf(lr.y), fabsf(lt)));  // fmaxf skips NaN
    }
    if constexpr (PART == kGather) {
      if (lane == 0) {
        a.lr_out[g] = lr;
        a.lt_out[g] = lt;
      }
    } else if (halted) {
      if (lane == 0) {
        a.g4_out[g] = make_float4(0.f, 0.f, 0.f, 0.f);
        a.part_out[g] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    } else {
      const AdjLocal o = adj_local(prm, L, u, rep.n, ldexpf(1.f, -s_up), ldexpf(1.f, -E), me_p, f, quarter, lr, lt);
      if (lane == 0) {
        a.g4_out[g] = make_float4(o.lF.x, o.lF.y, o.lsc.x, o.lsc.y);
        a.part_out[g] = make_float4(o.lrx, o.lry, o.lth, 0.f);
        if constexpr (G < 8) load_sums();
        adj_accumulate(prm, o, f, delta, ldexp(1.0, E), sum, a.acc, (size_t)ntot, g);
      }
    }
  }
  if constexpr (PART != kFactors) post_replica_max(r, mx, a.mx_out);
}

// one block per replica: sums of the per-particle accumulators
__global__ void k_adj_reduce(const ReplicaDesc* reps, int ntot, const double* acc, double* out) {
  __shared__ double tmp[kAdjBlock / 64];
  const int r = blockIdx.x;
  const int off = reps[r].off, n = reps[r].n;
  for (int k = 0; k < kAdjAcc; ++k) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += acc[(size_t)k * ntot + off + i];
    s = block_sum(s, tmp);
    if (threadIdx.x == 0) out[kAdjAcc * r + k] = s;
  }
}

inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

}  // namespace

hipError_t launch_adj_seed(int R, const ReplicaDesc* reps, const float4* xycs, const LossDev& L, const unsigned* halt,
                           float2* lr, float* lt, double* out, unsigned* mx, hipStream_t st) {
  hipLaunchKernelGGL(k_adj_seed, dim3(R), dim3(kAdjBlock), 0, st, reps, xycs, L, halt, lr, lt, out, mx);
  return hipGetLastError();
}

hipError_t launch_adj_reverse(int lanes, int part, const MeshDev& mesh, const ReplicaDesc* reps, const int* rid, int ntot,
                              const LossDev& L, const RevStep& a, hipStream_t st) {
  // (kFactors takes the gather's lanes too, which evaluate the field's modes side by side: 1,000 particles in
  // segments 5.2 ms at 16 lanes, 5.35 at one; at the 2 lanes of 64 x 2,000 6.52 against 6.46)
  // few waves: one a workgroup, so that each has a CU to itself (1,000 particles 11.2 -> 10.6 us a step)
  const int block = (long)ntot * lanes <= 65536 ? 64 : 256;
#define TISSUE_ADJ_PART(G, PART)                                                                                    \
  hipLaunchKernelGGL((k_adj_reverse<G, PART>), dim3(cdiv((long)ntot * G, block)), dim3(block), 0, st, mesh, reps, rid, ntot, \
                     L, a)
#define TISSUE_ADJ_LANES(G)                                                   \
  case G:                                                                     \
    if (part == kFactors) TISSUE_ADJ_PART(G, kFactors);                       \
    else if (part == kGather) TISSUE_ADJ_PART(G, kGather);                    \
    else if (part == kBoth) TISSUE_ADJ_PART(G, kBoth);                        \
    else return hipErrorInvalidValue;                                         \
    break
  switch (lanes) {
    TISSUE_ADJ_LANES(1);
    TISSUE_ADJ_LANES(2);
    TISSUE_ADJ_LANES(4);
    TISSUE_ADJ_LANES(8);
    TISSUE_ADJ_LANES(16);
    default: return hipErrorInvalidValue;
  }
#undef TISSUE_ADJ_LANES
#undef TISSUE_ADJ_PART
  return hipGetLastError();
}

hipError_t launch_adj_reduce(int R, const ReplicaDesc* reps, int ntot, const double* acc, double* out, hipStream_t st) {
  hipLaunchKernelGGL(k_adj_reduce, dim3(R), dim3(kAdjBlock), 0, st, reps, ntot, acc, out);
  return hipGetLastError();
}

}  // namespace tissue
