// Launchers and device-side constants of the reverse pass (adjoint.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "launch.h"

namespace tissue {

constexpr int kMaxModes = 16;  // modes of the target velocity field
constexpr int kAdjBlock = 256; // threads of the per-replica reduction kernels
constexpr int kAdjAcc = 5;     // per-particle FP64 accumulators: d v0, d mu, d k, d tau, velocity loss

// loss of a trajectory: w_order (phi_T - target)^2 + w_velocity mean_{t<T,i} |rdot - u(r)|^2 with
// u_c(x, y) = sum over modes of component c of amp sin(kx x + ky y + phase)
struct LossDev {
  float amp[kMaxModes], kx[kMaxModes], ky[kMaxModes], phase[kMaxModes];
  int comp[kMaxModes];
  int n_modes;
  int n_steps;  // T
  float target, w_order, w_velocity;
};

// per replica: out[2r] = phi_T, out[2r+1] = order loss; seeds lr = 0, lt = d loss / d theta_T, mx[r] = max |lt|
// (float bits)
hipError_t launch_adj_seed(int R, const ReplicaDesc* reps, const float4* xycs, const LossDev& L, const unsigned* halt,
                           float2* lr, float* lt, double* out, unsigned* mx, hipStream_t st);
// One launch of the reverse pass (adjoint.hip), by `lanes` (1 to 16) lanes per particle: kFactors: step p's
// factors from the adjoint (lr_in, lt_in) of the state after it; kGather: the adjoint (lr_out, lt_out)
// of the state before step q from step q's factors; kBoth: kGather of q, then kFactors of p = q - 1.
// Accumulators acc[kAdjAcc][ntot]. The adjoint state of replica r is stored scaled by 2^-E_r: the
// factors' exponent is sexp_in, raised by s_up when the max |lambda| in mx_in (float bits; kFactors: of
// its input, kBoth: of the step before, from which sup_in has been taken already) exceeds 2^21, and
// goes with s_up to sexp_out and sup_out; a gather posts its max to mx_out with atomicMax; mx_clear is
// zeroed for a later launch.
enum RevPart { kFactors = 0, kGather = 1, kBoth = 2 };
struct RevStep {
  BucketSet bs;             // vertex buckets of step q's input state
  const unsigned* halt;     // [R]
  int single;               // 1: one replica (rid is not read)
  int use_occ;              // 1: bs holds its occupancy mask, and few vertices are occupied
  const float4* xycs_q;     // step q's input state
  const int* vid_q;
  const float4* g4_in;      // step q's factors: (lF.x, lF.y, d loss / d sum sin, d loss / d sum cos)
  const float4* part_in;    // and the particles' own terms (x, y, theta)
  const float4* xycs_p;     // step p's input state and tape
  const float* th_p;
  const float4* fs_p;
  const int* quarter_p;
  const float2* lr_in;
  const float* lt_in;
  float4* g4_out;
  float4* part_out;
  float2* lr_out;
  float* lt_out;
  double* acc;
  const int* sexp_in;
  const int* sup_in;
  const unsigned* mx_in;
  int* sexp_out;
  int* sup_out;
  unsigned* mx_out;
  unsigned* mx_clear;
};
hipError_t launch_adj_reverse(int lanes, int part, const tdev::MeshDev& mesh, const ReplicaDesc* reps, const int* rid,
                              int ntot, const LossDev& L, const RevStep& a, hipStream_t st);
// out[kAdjAcc r + k] = sum over replica r of acc[k]
hipError_t launch_adj_reduce(int R, const ReplicaDesc* reps, int ntot, const double* acc, double* out, hipStream_t st);

}  // namespace tissue
