// Adjoint of n_steps of the step (engine side) and its C-ABI entry points.
//
// Whole tape (the rule when it fits in about 16 GB): the forward pass is the recording variant of the step
// kernel, which stores every pre-step state, the force and alignment sums and the seam-wrap turns, 44
// bytes per particle-step; nothing is recomputed. The reverse pass needs the vertex buckets of every
// state: the forward pass keeps them when they fit too, else they are made again from the recorded
// vertex ids, a few states ahead of the reverse pass on a stream of their own. Per reverse step one
// kernel: the transposed neighbour gather and the factors of the step before; two, in a second pass, where the
// adjoint grows too fast for that (adjoint.hip).
// Checkpoints (longer runs, and runs that stream or check every step): the tiled step kernel, with the
// state copied to a checkpoint every ckpt_every steps; in reverse, segment by segment from the last, the
// segment is recomputed from its checkpoint by the recording variant (bitwise the forward's states),
// which keeps the vertex buckets of every state of the segment when they fit (otherwise each reverse
// step rebuilds its state's buckets), and two kernels per step (factors, gather) go backwards through
// it. With several tapes the recomputes of the next segments run on their own streams meanwhile.
// Every form gives the same gradients (adjoint.hip).
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdlib>
#include <cmath>
#include <cstring>

#include "engine.h"

namespace tissue {

namespace {

LossDev make_loss(const tissue_loss& l, int n_steps) {
  if (l.n_modes < 0 || l.n_modes > kMaxModes) throw ApiError(TISSUE_E_INVALID_ARG, "n_modes out of range");
  const double sc[] = {l.target_order, l.w_order, l.w_velocity};
  for (double x : sc)
    if (!std::isfinite(x)) throw ApiError(TISSUE_E_INVALID_ARG, "non-finite loss weight");
  LossDev d{};
  d.n_modes = l.n_modes;
  d.n_steps = n_steps;
  d.target = (float)l.target_order;
  d.w_order = (float)l.w_order;
  d.w_velocity = (float)l.w_velocity;
  for (int m = 0; m < l.n_modes; ++m) {
    if (l.component[m] != 0 && l.component[m] != 1) throw ApiError(TISSUE_E_INVALID_ARG, "mode component must be 0 or 1");
    const double v[] = {l.amp[m], l.kx[m], l.ky[m], l.phase[m]};
    for (double x : v)
      if (!std::isfinite(x)) throw ApiError(TISSUE_E_INVALID_ARG, "non-finite field mode");
    d.comp[m] = l.component[m];
    d.amp[m] = (float)l.amp[m];
    d.kx[m] = (float)l.kx[m];
    d.ky[m] = (float)l.ky[m];
    d.phase[m] = (float)l.phase[m];
  }
  return d;
}

// n floats at p (a loop without branches)
bool all_finite(const void* p, size_t n) {
  uint32_t bad = 0;
  for (size_t i = 0; i < n; ++i) {
    uint32_t w;
    std::memcpy(&w, static_cast<const char*>(p) + 4 * i, 4);
    bad |= (w & 0x7f800000u) == 0x7f800000u ? 1u : 0u;
  }
  return bad == 0;
}

}  // namespace

void Engine::free_tape(Tape& t) {
  dfree(t.xycs); dfree(t.th); dfree(t.vid); dfree(t.fs); dfree(t.q);
  for (BucketSet& b : t.sbs) free_bucket_set(b);
  t.sbs.clear();
  dfree(t.vx); dfree(t.vy); dfree(t.r3x); dfree(t.r3y); dfree(t.r3z); dfree(t.face); dfree(t.nbr);
  dfree(t.rows); dfree(t.first_bad); dfree(t.partial);
  t.partial_n = 0;
}

void Engine::adjoint_release() {
  AdjointBuffers& a = adj;
  for (hipStream_t st : a.rec_stream)
    if (st) (void)hipStreamSynchronize(st);
  dfree(a.ck_xycs); dfree(a.ck_th); dfree(a.ck_vid);
  for (Tape& t : a.tp) free_tape(t);
  for (int k = 0; k < 2; ++k) { dfree(a.lr[k]); dfree(a.lt[k]); }
  for (int k = 0; k < 2; ++k) { dfree(a.g4[k]); dfree(a.part[k]); }
  dfree(a.acc); dfree(a.out_seed); dfree(a.out_red);
  dfree(a.sexp); dfree(a.sup); dfree(a.mx);
  free_whole_tape();
  if (a.ev_fwd) (void)hipEventDestroy(a.ev_fwd);
  for (int k = 0; k < kMaxTapes; ++k) {
    if (a.ev_ck[k]) (void)hipEventDestroy(a.ev_ck[k]);
    if (a.ev_rec[k]) (void)hipEventDestroy(a.ev_rec[k]);
    if (a.ev_rev[k]) (void)hipEventDestroy(a.ev_rev[k]);
  }
  for (hipStream_t st : a.rec_stream)
    if (st) (void)hipStreamDestroy(st);
  a = AdjointBuffers{};
}

void Engine::free_whole_tape() {
  free_tape(adj.whole);
  adj.whole_T = 0;
  free_set_slab();
}

void Engine::free_set_slab() {
  dfree(adj.set_slab);
  adj.sets.clear();
}

// bytes of a tape of T steps: T + 1 states, and T steps' sums and turns
size_t Engine::tape_bytes(int T) const { return ((size_t)T + 1) * ntot * 24 + (size_t)T * ntot * 20; }

// n bucket sets in one allocation
void Engine::alloc_set_slab(std::vector<BucketSet>& sets, int n) {
  const size_t cells = (size_t)R * md.nv, words = (size_t)R * tdev::occ_words(md.nv);
  size_t o = 0;
  auto place = [&](size_t bytes) {
    const size_t at = o;
    o += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t slot = place(cells * tdev::kSlots * 4), count = place(cells * 4), occ = place(words * 4),
               ovf = place((size_t)ntot * 8), multi = place((size_t)ntot * 4), big = place((size_t)ntot * 4),
               ovf_n = place((size_t)R * 4), big_n = place((size_t)R * 4);
  adj.set_slab = dalloc<unsigned char>(o * n);
  sets.resize(n);
  for (int k = 0; k < n; ++k) {
    unsigned char* p = adj.set_slab + o * k;
    sets[k] = BucketSet{(unsigned*)(p + occ), (int*)(p + count), (int*)(p + slot), (int*)(p + ovf_n), (int2*)(p + ovf),
                        (int*)(p + multi), (int*)(p + big_n), (int*)(p + big), raw_buckets ? 0 : 1};
  }
}

// the memory the tapes and their bucket sets may take: 16 GB, or TISSUE_ADJOINT_BUCKET_KB kilobytes
// when that is set (a smaller one selects the other forms, which give the same gradients)
static size_t adjoint_budget() {
  size_t budget = size_t(16) << 30;
  if (const char* e = std::getenv("TISSUE_ADJOINT_BUCKET_KB")) {
    const long long kb = std::atoll(e);
    if (kb >= 0) budget = (size_t)kb << 10;
  }
  return budget;
}

// a whole tape of T steps, when it may be used and fits: with the bucket sets of every state, or with
// two halves of kRingHalf sets. What is held stays as long as it can, so that horizons that take turns do
// not allocate anew (20 and 100 steps of 64 x 2,000 particles in turn 17.5 -> 13.9 ms): the tape where a run fits
// in it, the sets where there are enough.
bool Engine::whole_tape(int T) {
  AdjointBuffers& a = adj;
  const size_t N = ntot, budget = adjoint_budget(), set = bucket_set_bytes() + 4096;
  if (rec || d_visit) return false;
  auto sets_beside = [&](int len) { return tape_bytes(len) > budget ? 0 : (budget - tape_bytes(len)) / set; };
  int len = std::max(T, a.whole_T);
  if (sets_beside(len) < 2 * kRingHalf) len = T;
  const size_t most = sets_beside(len);
  if (most < 2 * kRingHalf) return false;
  a.keep_sets = most >= (size_t)T + 2;
  const size_t n_sets = a.keep_sets ? (size_t)T + 2 : 2 * kRingHalf;
  const bool new_tape = len != a.whole_T, new_sets = a.sets.size() < n_sets || a.sets.size() > most;
  if (!new_tape && !new_sets) return true;
  HIP_OK(hipStreamSynchronize(stream));
  if (new_tape) {
    free_tape(a.whole);
    a.whole_T = 0;
  }
  if (new_sets) free_set_slab();
  free_tapes();  // either form's memory, not both
  try {
    Tape& t = a.whole;
    if (new_tape) {
      t.xycs = dalloc<float4>((size_t)(len + 1) * N);
      t.th = dalloc<float>((size_t)(len + 1) * N);
      t.vid = dalloc<int>((size_t)(len + 1) * N);
      t.fs = dalloc<float4>((size_t)len * N);
      t.q = dalloc<int>((size_t)len * N);
      a.whole_T = len;
    }
    if (new_sets) alloc_set_slab(a.sets, (int)n_sets);
  } catch (const ApiError&) {  // less memory free than that: checkpoints need less
    free_whole_tape();
    return false;
  }
  return true;
}

// the segments' tapes
void Engine::free_tapes() {
  for (Tape& t : adj.tp) free_tape(t);
  adj.K = adj.ntape = 0;
}

// what every form needs
void Engine::adjoint_common() {
  AdjointBuffers& a = adj;
  const size_t N = ntot;
  if (a.lr[0]) return;
  try {
    for (int k = 0; k < 2; ++k) { a.lr[k] = dalloc<float2>(N); a.lt[k] = dalloc<float>(N); }
    for (int k = 0; k < 2; ++k) { a.g4[k] = dalloc<float4>(N); a.part[k] = dalloc<float4>(N); }
    a.acc = dalloc<double>(kAdjAcc * N);
    a.out_seed = dalloc<double>(2 * (size_t)R);
    a.out_red = dalloc<double>(kAdjAcc * (size_t)R);
    a.sexp = dalloc<int>(2 * (size_t)R);
    a.sup = dalloc<int>(2 * (size_t)R);
    a.mx = dalloc<unsigned>(3 * (size_t)R);
    for (hipStream_t& st : a.rec_stream) HIP_OK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    HIP_OK(hipEventCreateWithFlags(&a.ev_fwd, hipEventDisableTiming));
    for (int k = 0; k < kMaxTapes; ++k) {
      HIP_OK(hipEventCreateWithFlags(&a.ev_ck[k], hipEventDisableTiming));
      HIP_OK(hipEventCreateWithFlags(&a.ev_rec[k], hipEventDisableTiming));
      HIP_OK(hipEventCreateWithFlags(&a.ev_rev[k], hipEventDisableTiming));
    }
  } catch (...) {  // all of them or none
    adjoint_release();
    throw;
  }
}

void Engine::adjoint_buffers(int K, int C) {
  AdjointBuffers& a = adj;
  const size_t N = ntot;
  free_whole_tape();
  if (C > a.C) {
    dfree(a.ck_xycs); dfree(a.ck_th); dfree(a.ck_vid);
    a.C = 0;
    a.ck_xycs = dalloc<float4>((size_t)C * N); a.ck_th = dalloc<float>((size_t)C * N); a.ck_vid = dalloc<int>((size_t)C * N);
    a.C = C;
  }
  // as many tapes (up to three) as have their bucket sets within about 16 GB together: the
  // recomputes of two segments then run side by side while the reverse pass of a third runs;
  // else one tape, with its states' bucket sets when they fit (otherwise each reverse step
  // re-buckets its state), and everything in order on the engine's stream
  const size_t sets = (size_t)K + 2, budget = adjoint_budget();
  int ntape = 1;
  while (ntape < kMaxTapes && (size_t)(ntape + 1) * sets * bucket_set_bytes() <= budget) ++ntape;
  const bool with_sets = sets * bucket_set_bytes() <= budget;
  if (K > a.K || ntape != a.ntape || with_sets != !a.tp[0].sbs.empty()) {
    free_tapes();
    for (int k = 0; k < ntape; ++k) {
      Tape& t = a.tp[k];
      t.xycs = dalloc<float4>((size_t)(K + 1) * N);
      t.th = dalloc<float>((size_t)(K + 1) * N);
      t.vid = dalloc<int>((size_t)(K + 1) * N);
      t.fs = dalloc<float4>((size_t)K * N);
      t.q = dalloc<int>((size_t)K * N);
      if (with_sets) {
        t.sbs.resize(sets);
        for (BucketSet& b : t.sbs) alloc_bucket_set(b);
      }
      t.vx = dalloc<float>(N); t.vy = dalloc<float>(N);
      t.r3x = dalloc<float>(N); t.r3y = dalloc<float>(N); t.r3z = dalloc<float>(N);
      t.face = dalloc<int>(N); t.nbr = dalloc<int>(N);
      t.rows = dalloc<unsigned>(3 * (size_t)R);
      t.first_bad = dalloc<int>(R);
    }
    a.K = K;
    a.ntape = ntape;
  }
  for (int k = 0; k < ntape; ++k) {
    Tape& t = a.tp[k];
    const int np = n_logical * partials_per_tile(kStepMaxBlock);  // written, not read: sized for any shape
    if (t.partial_n < np) {
      regrow(t.partial, t.partial_n, np);
    }
  }
}

int32_t Engine::adjoint(int T, const float* nz, size_t stride, int K, const tissue_loss& loss, tissue_grads* g,
                        double* d_theta0, double* d_x0, double* d_y0) {
  if (!has_state) throw ApiError(TISSUE_E_INVALID_ARG, "no state: call init_random or set_state first");
  if (T < 1 || K < 1) throw ApiError(TISSUE_E_INVALID_ARG, "n_steps and ckpt_every must be positive");
  if (!g) throw ApiError(TISSUE_E_INVALID_ARG, "null gradient output");
  const LossDev L = make_loss(loss, T);
  K = std::min(K, T);
  const int C = (T + K - 1) / K;
  const Shape s = resolve_tiled();
  // the reverse gather walks the same rows as the forward with at most 16 lanes per particle: wider
  // groups shorten the forward's critical path but not the gather's (1,000 particles: reverse
  // 16.0 us per step at 16 lanes, 18.2 us at 32)
  const int gather_lanes = std::min(s.lanes, 16);
  ensure_buckets();
  ensure_tiles(s);
  adjoint_common();
  AdjointBuffers& a = adj;
  const size_t N = ntot;
  double fwd_ms = 0.0;
  int32_t status = TISSUE_OK;
  float2* lr_end = nullptr;  // the adjoint of the initial state and its exponents
  float* lt_end = nullptr;
  int* sexp_end = nullptr;
  RevStep v{};
  v.halt = d_halt;
  v.single = R == 1 ? 1 : 0;
  v.acc = a.acc;
  std::vector<double> seed, red;
  std::vector<float2> lr;
  std::vector<float> lt;
  std::vector<int> sexp;
  double rev_ms = 0.0;
  // mx_slot: the slot of mx that the first factors read
  auto begin_reverse = [&](int mx_slot) {
    HIP_OK(hipEventRecord(ev0, stream));
    HIP_OK(hipMemsetAsync(a.acc, 0, kAdjAcc * N * sizeof(double), stream));
    HIP_OK(hipMemsetAsync(a.sexp, 0, 2 * R * sizeof(int), stream));
    HIP_OK(hipMemsetAsync(a.sup, 0, 2 * R * sizeof(int), stream));
    HIP_OK(hipMemsetAsync(a.mx, 0, 3 * R * sizeof(unsigned), stream));
    HIP_OK(launch_adj_seed(R, d_reps, xycs[sphase], L, d_halt, a.lr[0], a.lt[0], a.out_seed, a.mx + mx_slot * R, stream));
  };
  auto end_reverse = [&] {
    HIP_OK(launch_adj_reduce(R, d_reps, ntot, a.acc, a.out_red, stream));
    HIP_OK(hipEventRecord(ev1, stream));
    seed.resize(2 * (size_t)R);
    red.resize(kAdjAcc * (size_t)R);
    lr.resize(N);
    lt.resize(N);
    sexp.resize(R);
    HIP_OK(hipMemcpyAsync(seed.data(), a.out_seed, seed.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
    HIP_OK(hipMemcpyAsync(red.data(), a.out_red, red.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
    HIP_OK(hipMemcpyAsync(lr.data(), lr_end, N * sizeof(float2), hipMemcpyDeviceToHost, stream));
    HIP_OK(hipMemcpyAsync(lt.data(), lt_end, N * sizeof(float), hipMemcpyDeviceToHost, stream));
    HIP_OK(hipMemcpyAsync(sexp.data(), sexp_end, R * sizeof(int), hipMemcpyDeviceToHost, stream));
    HIP_OK(hipStreamSynchronize(stream));
    float ms = 0.f;
    HIP_OK(hipEventElapsedTime(&ms, ev0, ev1));
    rev_ms += ms;
  };
  // whether the adjoint stayed within FP32 (adjoint.hip); a sum alone may be beyond FP64 of itself
  auto in_range = [&] {
    for (int r = 0; r < R; ++r)
      for (int k = 0; k < kAdjAcc; ++k)
        if (!std::isfinite(red[kAdjAcc * r + k]) && sexp[r] < 512) return false;
    return all_finite(lr.data(), 2 * N) && all_finite(lt.data(), N);
  };
  if (whole_tape(T)) {
    Tape& tp = a.whole;
    HIP_OK(hipMemcpyAsync(tp.xycs, xycs[sphase], N * sizeof(float4), hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(tp.th, th[sphase], N * sizeof(float), hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(tp.vid, vid[sphase], N * sizeof(int), hipMemcpyDeviceToDevice, stream));
    BucketSet* sets = a.keep_sets ? a.sets.data() : bs;
    HIP_OK(launch_clear_sets(R, md.nv, sets + 1, 2, stream));
    bucket_state_into(tp.vid, sets[0]);
    buckets_stale = true;  // the sets no longer follow the engine's own phase
    status = run_once(s, T, nz, stride, 0, &tp);
    fwd_ms = last_ms;
    HIP_OK(hipMemcpyAsync(xycs[sphase], tp.xycs + T * N, N * sizeof(float4), hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(th[sphase], tp.th + T * N, N * sizeof(float), hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(vid[sphase], tp.vid + T * N, N * sizeof(int), hipMemcpyDeviceToDevice, stream));
    // half h of the ring: the buckets of the states T - 1 - h kRingHalf .. downwards
    const int halves = (T + kRingHalf - 1) / kRingHalf;
    hipStream_t side = a.rec_stream[0];
    auto ring_set = [&](int q) -> BucketSet& { return a.sets[(T - 1 - q) % (2 * kRingHalf)]; };
    auto fill = [&](int h) {
      if (h >= halves) return;
      if (h >= 2) HIP_OK(hipStreamWaitEvent(side, a.ev_rev[h & 1], 0));
      for (int q = T - 1 - h * kRingHalf; q >= std::max(0, T - (h + 1) * kRingHalf); --q)
        bucket_state_into(tp.vid + q * N, ring_set(q), side, h >= 2 ? tp.vid + (q + 2 * kRingHalf) * N : nullptr);
      HIP_OK(hipEventRecord(a.ev_rec[h & 1], side));
    };
    v.use_occ = !a.keep_sets && 8L * nmax < md.nv ? 1 : 0;
    v.lt_out = a.lt[1];
    v.lr_out = a.lr[1];
    lr_end = a.lr[1];
    lt_end = a.lt[1];
    // fused: one launch a step (kBoth); else two, for adjoints that grow faster than FP32 lets it follow
    auto reverse_whole = [&](bool fused) {
      begin_reverse(2);
      if (!a.keep_sets) {
        fill(0);
        fill(1);
      }
      // launch j: factors and maxima from slots that launch j - 1 wrote, to the next ones; e: the slot of the
      // exponents, which the launches with factors move on
      int j = 0, e = 0;
      v.lr_in = a.lr[0];
      v.lt_in = a.lt[0];
      auto launch = [&](int part, int q, int p) {
        v.sexp_in = a.sexp + e * R; v.sexp_out = a.sexp + (1 - e) * R;
        v.sup_in = a.sup + e * R; v.sup_out = a.sup + (1 - e) * R;
        v.mx_in = a.mx + (j + 2) % 3 * R; v.mx_out = a.mx + j % 3 * R; v.mx_clear = a.mx + (j + 1) % 3 * R;
        v.g4_in = a.g4[1 - (j & 1)]; v.part_in = a.part[1 - (j & 1)];
        v.g4_out = a.g4[j & 1]; v.part_out = a.part[j & 1];
        if (q >= 0) {
          v.bs = a.keep_sets ? a.sets[q] : ring_set(q);
          v.xycs_q = tp.xycs + q * N; v.vid_q = tp.vid + q * N;
        }
        if (p >= 0) {
          v.xycs_p = tp.xycs + p * N; v.th_p = tp.th + p * N; v.fs_p = tp.fs + p * N; v.quarter_p = tp.q + p * N;
        }
        HIP_OK(launch_adj_reverse(gather_lanes, part, md, d_reps, d_rid, ntot, L, v, stream));
        ++j;
        if (part != kGather) e = 1 - e;
      };
      launch(kFactors, -1, T - 1);
      v.lr_in = a.lr[1];
      v.lt_in = a.lt[1];
      for (int q = T - 1; q >= 0; --q) {
        const int at = T - 1 - q, h = at / kRingHalf;
        if (!a.keep_sets && at % kRingHalf == 0) HIP_OK(hipStreamWaitEvent(stream, a.ev_rec[h & 1], 0));
        launch(fused && q > 0 ? kBoth : kGather, q, q - 1);
        if (!fused && q > 0) launch(kFactors, -1, q - 1);
        if (!a.keep_sets && (at % kRingHalf == kRingHalf - 1 || q == 0)) {
          HIP_OK(hipEventRecord(a.ev_rev[h & 1], stream));
          fill(h + 2);
        }
      }
      sexp_end = a.sexp + e * R;
      end_reverse();
    };
    reverse_whole(true);
    if (!in_range()) reverse_whole(false);
  } else {
  adjoint_buffers(K, C);

  // recomputes: with nt > 1 tapes, segment c goes to tape c % nt on recompute stream c % (nt - 1),
  // nt - 1 segments ahead of the reverse passes (tapes are handed over by events); with one tape
  // everything runs in order on the engine's stream
  // (the last nt - 1 segments are recomputed as soon as their checkpoints are written, while the
  // forward still runs)
  const int nt = a.ntape, ns = nt - 1;
  const bool overlap = nt > 1;
  auto rs_of = [&](int c) { return overlap ? a.rec_stream[c % ns] : stream; };
  auto segment_set = [&](Tape& tp, int kc, int q) -> BucketSet& {
    return tp.sbs.size() >= (size_t)kc + 2 ? tp.sbs[q] : bs[q % 3];
  };
  // recompute segment c from its checkpoint into tape c % nt, recording the tape; ready: an
  // event on the engine's stream after which checkpoint c is written
  auto recompute = [&](int c, hipEvent_t ready) {
    const int t0 = c * K, kc = std::min(K, T - t0);
    Tape& tp = a.tp[c % nt];
    hipStream_t rs = rs_of(c);
    if (overlap) {
      HIP_OK(hipStreamWaitEvent(rs, ready, 0));
      if (c + nt <= C - 1) HIP_OK(hipStreamWaitEvent(rs, a.ev_rev[c % nt], 0));  // segment c + nt is done with it
    }
    HIP_OK(hipMemcpyAsync(tp.xycs, a.ck_xycs + c * N, N * sizeof(float4), hipMemcpyDeviceToDevice, rs));
    HIP_OK(hipMemcpyAsync(tp.th, a.ck_th + c * N, N * sizeof(float), hipMemcpyDeviceToDevice, rs));
    HIP_OK(hipMemcpyAsync(tp.vid, a.ck_vid + c * N, N * sizeof(int), hipMemcpyDeviceToDevice, rs));
    clear_bucket_set(segment_set(tp, kc, 1), rs);
    clear_bucket_set(segment_set(tp, kc, 2), rs);
    bucket_state_into(tp.vid, segment_set(tp, kc, 0), rs);
    HIP_OK(launch_flags_begin(R, d_halt, tp.rows, tp.first_bad, rs));
    for (int q = 0; q < kc; ++q) {
      TiledIO io{};
      io.xycs_in = tp.xycs + q * N; io.th_in = tp.th + q * N; io.vid_in = tp.vid + q * N;
      io.xycs_out = tp.xycs + (q + 1) * N; io.th_out = tp.th + (q + 1) * N; io.vid_out = tp.vid + (q + 1) * N;
      io.vx = tp.vx; io.vy = tp.vy; io.r3x = tp.r3x; io.r3y = tp.r3y; io.r3z = tp.r3z; io.face = tp.face;
      io.nbr = tp.nbr;
      io.noise = nz ? nz + (size_t)(t0 + q) * stride : nullptr;
      io.partial = tp.partial;
      io.halt_in = tp.rows + (size_t)(q % 3) * R;
      io.halt_out = tp.rows + (size_t)((q + 1) % 3) * R;
      io.halt_clr = tp.rows + (size_t)((q + 2) % 3) * R;
      io.first_bad = tp.first_bad;
      io.step = q;
      io.areas = step_areas(nmax, s.block, phys_lanes(s));
      io.tape_fs = tp.fs + q * N;
      io.tape_q = tp.q + q * N;
      HIP_OK(launch_step_tiled(s.lanes, phys_lanes(s), s.block, true, !raw_buckets, md, d_reps, d_tiles, n_phys, segment_set(tp, kc, q),
                               segment_set(tp, kc, q + 1), segment_set(tp, kc, q + 2), io, rs));
      if (!raw_buckets)
        HIP_OK(launch_bucket_finalize(s.block, d_reps, d_tiles, n_phys, md.nv, R == 1 ? ntot : 0,
                                      segment_set(tp, kc, q + 1), rs));
    }
    if (overlap) HIP_OK(hipEventRecord(a.ev_rec[c % nt], rs));
  };
  // lr[cur], lt[cur]: the adjoint of the current state; slot cur of sexp and mx: its exponent and max
  int cur = 0;
  // backwards through segment c
  auto reverse = [&](int c) {
    const int t0 = c * K, kc = std::min(K, T - t0);
    Tape& tp = a.tp[c % nt];
    const bool keep = tp.sbs.size() >= (size_t)kc + 2;
    if (overlap) HIP_OK(hipStreamWaitEvent(stream, a.ev_rec[c % nt], 0));
    for (int q = kc - 1; q >= 0; --q) {
      if (!keep) bucket_state_into(tp.vid + q * N, bs[0], stream);
      v.bs = keep ? tp.sbs[q] : bs[0];
      v.xycs_q = v.xycs_p = tp.xycs + q * N; v.vid_q = tp.vid + q * N; v.th_p = tp.th + q * N;
      v.fs_p = tp.fs + q * N; v.quarter_p = tp.q + q * N;
      v.lr_in = a.lr[cur]; v.lt_in = a.lt[cur]; v.lr_out = a.lr[1 - cur]; v.lt_out = a.lt[1 - cur];
      v.g4_in = v.g4_out = a.g4[0]; v.part_in = v.part_out = a.part[0];
      v.sexp_in = a.sexp + cur * R; v.sexp_out = a.sexp + (1 - cur) * R;
      v.sup_in = a.sup + cur * R; v.sup_out = a.sup + (1 - cur) * R;
      v.mx_in = a.mx + cur * R; v.mx_out = v.mx_clear = a.mx + (1 - cur) * R;
      HIP_OK(launch_adj_reverse(gather_lanes, kFactors, md, d_reps, d_rid, ntot, L, v, stream));
      HIP_OK(launch_adj_reverse(gather_lanes, kGather, md, d_reps, d_rid, ntot, L, v, stream));
      cur = 1 - cur;
    }
    if (overlap) HIP_OK(hipEventRecord(a.ev_rev[c % nt], stream));
  };
  // forward, with a checkpoint at the start of every segment
  for (int c = 0; c < C; ++c) {
    const int t0 = c * K, kc = std::min(K, T - t0);
    HIP_OK(hipMemcpyAsync(a.ck_xycs + c * N, xycs[sphase], N * sizeof(float4), hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(a.ck_th + c * N, th[sphase], N * sizeof(float), hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(a.ck_vid + c * N, vid[sphase], N * sizeof(int), hipMemcpyDeviceToDevice, stream));
    if (overlap && c >= C - ns) {
      HIP_OK(hipEventRecord(a.ev_ck[c % nt], stream));
      recompute(c, a.ev_ck[c % nt]);
    }
    const int32_t st = run_shape(s, kc, nz, stride, t0);
    fwd_ms += last_ms;
    if (st != TISSUE_OK && status == TISSUE_OK) status = st;
  }
  // reverse
  begin_reverse(0);
  if (overlap) {
    HIP_OK(hipEventRecord(a.ev_fwd, stream));  // every checkpoint is written
    for (int c = C - 1; c >= 0; --c) {
      reverse(c);
      if (c - ns >= 0) recompute(c - ns, a.ev_fwd);
    }
  } else {
    recompute(C - 1, nullptr);
    for (int c = C - 1; c >= 0; --c) {
      reverse(c);
      if (c >= 1) recompute(c - 1, nullptr);
    }
  }
  lr_end = a.lr[cur];
  lt_end = a.lt[cur];
  sexp_end = a.sexp + cur * R;
  end_reverse();
  }
  buckets_stale = true;  // the reverse pass used the bucket sets
  for (int r = 0; r < R; ++r) {
    tissue_grads& o = g[r];
    o.phi_final = seed[2 * r];
    o.loss_order = seed[2 * r + 1];
    o.loss_velocity = red[kAdjAcc * r + 4];
    o.loss = o.loss_order + o.loss_velocity;
    o.d_v0 = red[kAdjAcc * r + 0];
    o.d_mu = red[kAdjAcc * r + 1];
    o.d_k = red[kAdjAcc * r + 2];
    o.d_tau = red[kAdjAcc * r + 3];
    o.forward_ms = fwd_ms;
    o.reverse_ms = rev_ms;
  }
  for (int r = 0; r < R; ++r) {
    const double sc = std::ldexp(1.0, sexp[r]);
    for (int i = off[r]; i < off[r] + n[r]; ++i) {
      if (d_theta0) d_theta0[i] = sc * (double)lt[i];
      if (d_x0) d_x0[i] = sc * (double)lr[i].x;
      if (d_y0) d_y0[i] = sc * (double)lr[i].y;
    }
  }
  last_ms = fwd_ms + rev_ms;
  return status;
}

}  // namespace tissue

extern "C" {

int32_t tissue_adjoint(tissue_sim* s, int32_t n_steps, int32_t first_row, int32_t ckpt_every, const tissue_loss* loss,
                       tissue_grads* g, double* d_theta0, double* d_x0, double* d_y0) {
  return guarded([&] {
    if (!s || !s->e) throw ApiError(TISSUE_E_INVALID_ARG, "null simulation handle");
    if (!loss) throw ApiError(TISSUE_E_INVALID_ARG, "null loss");
    auto& e = *s->e;
    HIP_OK(hipSetDevice(e.device));
    const float* nz = first_row >= 0 ? e.staged_rows(first_row, n_steps) : nullptr;
    return e.adjoint(n_steps, nz, (size_t)e.ntot, ckpt_every, *loss, g, d_theta0, d_x0, d_y0);
  });
}

int32_t tissue_batch_adjoint(tissue_batch* b, int32_t n_steps, int32_t first_row, int32_t ckpt_every,
                             const tissue_loss* loss, tissue_grads* g, double* d_theta0, double* d_x0, double* d_y0) {
  return guarded([&] {
    if (!b || !b->e) throw ApiError(TISSUE_E_INVALID_ARG, "null batch handle");
    if (!loss) throw ApiError(TISSUE_E_INVALID_ARG, "null loss");
    auto& e = *b->e;
    HIP_OK(hipSetDevice(e.device));
    const float* nz = first_row >= 0 ? e.staged_rows(first_row, n_steps) : nullptr;
    return e.adjoint(n_steps, nz, (size_t)e.ntot, ckpt_every, *loss, g, d_theta0, d_x0, d_y0);
  });
}

}  // extern "C"
