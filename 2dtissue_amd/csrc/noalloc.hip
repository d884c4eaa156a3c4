// tissue_step_noalloc: one step of one system for callers that cannot allocate device memory
// (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
//
// The caller passes the state and the outputs as device pointers. Everything else the step
// kernel needs (the packed state, three vertex-bucket sets, the tile and replica descriptors, the
// order-parameter partials and the flag rows) lives in `scratch`, a file-scope device array of
// kScratchBytes that each GPU the library runs on holds until the process ends. The entry point
// calls no hipMalloc, hipFree or allocating library routine, and no hipMemsetAsync: buffers that
// must start at zero are cleared by the set-up kernel. A call is four kernels (five where buckets are
// sorted), each some 4 us at these sizes whatever it does: set-up, bucketing of the input state, the
// step, and one for all that follows it. It launches the same step kernel as
// tissue_step with the same default launch shape, so its results equal one tissue_step bit for
// bit. Calls that overlap on one GPU share its scratch and race; the array keeps the last call's
// contents.
#include <hip/hip_runtime.h>

#include <array>
#include <climits>
#include <mutex>

#include "capi_common.h"
#include "step_kernel.h"

namespace {

using tissue::BucketSet;
using tissue::OrderPartial;
using tissue::ReplicaDesc;
using tissue::TileDesc;
using tissue::TiledIO;

constexpr int kMaxParticles = TISSUE_NOALLOC_MAX_PARTICLES;
constexpr int kMaxVertices = TISSUE_NOALLOC_MAX_UV_VERTICES;
// tiles of the default launch shape: 2 particles per tile (32 lanes in 64 threads) up to 4,096
// particles, 8 up to 8,192 and 16 beyond (the physical lanes: 16 and 8 in 128 threads), so at most 2,048
constexpr int kMaxTiles = 2048;

constexpr size_t al(size_t x) { return (x + 255) & ~(size_t)255; }

// byte offsets of the scratch regions
struct Layout {
  static constexpr size_t xycs_in = 0;
  static constexpr size_t xycs_out = xycs_in + al(sizeof(float4) * kMaxParticles);
  static constexpr size_t vid = xycs_out + al(sizeof(float4) * kMaxParticles);
  // one bucket set: occupancy mask, count[V], slot[V * kSlots], ovf[N] (int2), multi[N], big[N],
  // counters[2]
  static constexpr size_t set_occ = 0;
  static constexpr size_t set_count = set_occ + al(sizeof(unsigned) * tdev::occ_words(kMaxVertices));
  static constexpr size_t set_slot = set_count + al(sizeof(int) * kMaxVertices);
  static constexpr size_t set_ovf = set_slot + al(sizeof(int) * kMaxVertices * tdev::kSlots);
  static constexpr size_t set_multi = set_ovf + al(sizeof(int2) * kMaxParticles);
  static constexpr size_t set_big = set_multi + al(sizeof(int) * kMaxParticles);
  static constexpr size_t set_ctr = set_big + al(sizeof(int) * kMaxParticles);
  static constexpr size_t set_bytes = set_ctr + al(sizeof(int) * 2);
  static constexpr size_t sets = vid + al(sizeof(int) * kMaxParticles);
  static constexpr size_t partial = sets + 3 * set_bytes;
  static constexpr size_t tiles = partial + al(sizeof(OrderPartial) * kMaxTiles * (tissue::kStepMaxBlock / 64));
  static constexpr size_t rep = tiles + al(sizeof(TileDesc) * kMaxTiles);
  static constexpr size_t rows = rep + al(sizeof(ReplicaDesc));
  static constexpr size_t first_bad = rows + al(sizeof(unsigned) * 3);
  static constexpr size_t bad = first_bad + al(sizeof(int));  // bad vertex ids of the call, else 0
  static constexpr size_t total = bad + al(sizeof(unsigned));
};
constexpr size_t kScratchBytes = TISSUE_NOALLOC_SCRATCH_BYTES;
static_assert(Layout::total <= kScratchBytes, "scratch regions exceed the declared scratch size");

// The scratch array. In host code its name is a host-side stand-in, not a device address: host
// code uses only the per-device address from hipGetSymbolAddress (scratch_base).
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_mu;
std::array<unsigned char*, 64> g_base{};  // per device, from hipGetSymbolAddress

unsigned char* scratch_base(int device) {
  if (device < 0 || device >= (int)g_base.size()) throw ApiError(TISSUE_E_INVALID_ARG, "device index out of range");
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_base[device]) {
    void* p = nullptr;
    HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw ApiError(TISSUE_E_HIP, "hipGetSymbolAddress returned a null scratch address");
    g_base[device] = (unsigned char*)p;
  }
  return g_base[device];
}

BucketSet set_at(unsigned char* base, int k, int sorted) {
  unsigned char* s = base + Layout::sets + (size_t)k * Layout::set_bytes;
  int* ctr = (int*)(s + Layout::set_ctr);
  BucketSet b;
  b.occ = (unsigned*)(s + Layout::set_occ);
  b.count = (int*)(s + Layout::set_count);
  b.slot = (int*)(s + Layout::set_slot);
  b.ovf = (int2*)(s + Layout::set_ovf);
  b.multi = (int*)(s + Layout::set_multi);
  b.big = (int*)(s + Layout::set_big);
  b.ovf_n = ctr;
  b.big_n = ctr + 1;
  b.sorted = sorted;
  return b;
}

struct SetupArgs {
  int n, nv, n_tiles, per_tile;
  const float* x;
  const float* y;
  const float* th;
  float4* xycs;
  BucketSet sets[3];
  TileDesc* tiles;
  ReplicaDesc* rep;
  unsigned* rows;
  int* first_bad;
  unsigned* bad;
  ReplicaDesc rep_value;
};

// packs the state (x, y, cos theta, sin theta), clears the bucket sets (counts, occupancy masks, list
// lengths) and the flag words, and writes the tile and replica descriptors
__global__ void k_noalloc_setup(SetupArgs a) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < a.n) {
    float s, c;
    sincosf(a.th[t], &s, &c);
    a.xycs[t] = make_float4(a.x[t], a.y[t], c, s);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (t < a.nv) a.sets[k].count[t] = 0;
    if (t < tdev::occ_words(a.nv)) a.sets[k].occ[t] = 0u;
    if (t == 0) *a.sets[k].ovf_n = *a.sets[k].big_n = 0;
  }
  if (t < a.n_tiles) a.tiles[t] = TileDesc{0, t * a.per_tile, t, t, tissue::clear_end(a.nv, t - 1, a.n_tiles),
                                            tissue::clear_end(a.nv, t, a.n_tiles)};
  if (t < 3) a.rows[t] = 0u;
  if (t == 0) {
    *a.rep = a.rep_value;
    *a.first_bad = INT_MAX;
    *a.bad = 0u;
  }
}

// copies the vertex ids (an id outside the mesh is replaced by 0 and reported with TISSUE_FLAG_BAD_INPUT,
// so no later access leaves its table) and buckets the particles
__global__ void k_noalloc_insert(int n, int nv, const int* vid_in, int* vid, unsigned* bad, BucketSet set) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int v = vid_in[t];
  const bool ok = v >= 0 && v < nv;
  vid[t] = ok ? v : 0;
  if (!ok) atomicOr(bad, TISSUE_FLAG_BAD_INPUT);
  tissue::bucket_insert<true>(tissue::replica_out(set, 0, nv, 0), ok ? v : 0, t);
}

// splits the new packed positions into the caller's x and y; workgroup 0 also reduces the order parameters
// and reports the step's flags
__global__ void __launch_bounds__(tissue::kPhiBlock) k_noalloc_finish(int n, const float4* xycs, float* x, float* y,
                                                                     const OrderPartial* partial, int n_partials,
                                                                     double* phi, const unsigned* halt_out,
                                                                     const unsigned* bad, unsigned* flags_out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) {
    const float4 q = xycs[t];
    x[t] = q.x;
    y[t] = q.y;
  }
  if (t == 0) *flags_out = *bad | *halt_out;
  if (blockIdx.x == 0) tissue::block_phi(partial, 0, n_partials, n, phi);
}

inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

}  // namespace

extern "C" int32_t tissue_step_noalloc(const tissue_mesh* mc, const tissue_params* p, int32_t n, const float* x_in,
                                       const float* y_in, const float* theta_in, const int32_t* vid_in,
                                       const float* noise, float* x_out, float* y_out, float* theta_out,
                                       int32_t* vid_out, float* vx, float* vy, float* r3x, float* r3y, float* r3z,
                                       int32_t* face, int32_t* nbr, double* phi, uint32_t* flags, void* stream) {
  return guarded([&] {
    if (!mc || !p) throw ApiError(TISSUE_E_INVALID_ARG, "null mesh or params");
    if (n < 1 || n > kMaxParticles)
      throw ApiError(TISSUE_E_INVALID_ARG, "tissue_step_noalloc: particle count must be in 1.." +
                                               std::to_string(kMaxParticles));
    const float* ins[] = {x_in, y_in, theta_in};
    float* outs[] = {x_out, y_out, theta_out, vx, vy, r3x, r3y, r3z};
    for (const float* q : ins)
      if (!q) throw ApiError(TISSUE_E_INVALID_ARG, "null state pointer");
    for (float* q : outs)
      if (!q) throw ApiError(TISSUE_E_INVALID_ARG, "null output pointer");
    if (!vid_in || !vid_out || !face || !nbr || !phi || !flags)
      throw ApiError(TISSUE_E_INVALID_ARG, "null output pointer");
    auto* m = const_cast<tissue_mesh*>(mc);
    int dev = 0;
    HIP_OK(hipGetDevice(&dev));
    const tdev::MeshDev md = m->resident_view(dev);
    if (md.nv > kMaxVertices)
      throw ApiError(TISSUE_E_INVALID_ARG, "tissue_step_noalloc: the mesh has more than " +
                                               std::to_string(kMaxVertices) + " UV vertices");
    check_params(p, m->sigma_max);
    unsigned char* base = scratch_base(dev);
    auto st = (hipStream_t)stream;

    int lanes = 0, block = 0;
    tissue::tiled_default_shape(1, n, n, md.nv, &lanes, &block);
    const int phys = tissue::phys_lanes(lanes, n, n, md.nv, block), per = block / phys;
    const int n_tiles = cdiv(n, per);
    if (n_tiles > kMaxTiles) throw ApiError(TISSUE_E_INVALID_ARG, "tissue_step_noalloc: too many tiles");
    const int sorted = tissue::raw_buckets_for(n, md.nv) ? 0 : 1;
    BucketSet b[3] = {set_at(base, 0, sorted), set_at(base, 1, sorted), set_at(base, 2, sorted)};

    SetupArgs a{};
    a.n = n;
    a.nv = md.nv;
    a.n_tiles = n_tiles;
    a.per_tile = per;
    a.x = x_in;
    a.y = y_in;
    a.th = theta_in;
    a.xycs = (float4*)(base + Layout::xycs_in);
    int* vid = (int*)(base + Layout::vid);
    for (int k = 0; k < 3; ++k) a.sets[k] = b[k];
    a.tiles = (TileDesc*)(base + Layout::tiles);
    a.rep = (ReplicaDesc*)(base + Layout::rep);
    a.rows = (unsigned*)(base + Layout::rows);
    a.first_bad = (int*)(base + Layout::first_bad);
    a.bad = (unsigned*)(base + Layout::bad);
    a.rep_value = ReplicaDesc{0, n, make_step_params(*p)};
    const int span = std::max(std::max(n, md.nv), n_tiles);
    hipLaunchKernelGGL(k_noalloc_setup, dim3(cdiv(span, 256)), dim3(256), 0, st, a);
    HIP_OK(hipGetLastError());

    // buckets of the input state (set 0), sorted when the engine's rule sorts them
    BucketSet in = b[0];
    if (!sorted) in.multi = nullptr;  // no finalize pass reads the marks
    hipLaunchKernelGGL(k_noalloc_insert, dim3(cdiv(n, 256)), dim3(256), 0, st, n, md.nv, vid_in, vid, a.bad, in);
    HIP_OK(hipGetLastError());
    if (sorted) HIP_OK(tissue::launch_bucket_finalize(block, a.rep, a.tiles, n_tiles, md.nv, n, b[0], st));

    TiledIO io{};
    io.xycs_in = a.xycs;
    io.th_in = theta_in;
    io.vid_in = vid;
    io.xycs_out = (float4*)(base + Layout::xycs_out);
    io.th_out = theta_out;
    io.vid_out = vid_out;
    io.vx = vx;
    io.vy = vy;
    io.r3x = r3x;
    io.r3y = r3y;
    io.r3z = r3z;
    io.face = face;
    io.nbr = nbr;
    io.noise = noise;
    io.noise_row0 = nullptr;
    io.noise_stride = 0;
    io.partial = (OrderPartial*)(base + Layout::partial);
    io.halt_in = a.rows;
    io.halt_out = a.rows + 1;
    io.halt_clr = a.rows + 2;
    io.first_bad = a.first_bad;
    io.step = 0;
    io.areas = tissue::step_areas(n, block, phys);
    HIP_OK(tissue::launch_step_tiled(lanes, phys, block, false, sorted != 0, md, a.rep, a.tiles, n_tiles, b[0], b[1], b[2], io, st));
    hipLaunchKernelGGL(k_noalloc_finish, dim3(cdiv(n, tissue::kPhiBlock)), dim3(tissue::kPhiBlock), 0, st, n, io.xycs_out,
                       x_out, y_out, io.partial, n_tiles * tissue::partials_per_tile(block), phi, io.halt_out, a.bad,
                       flags);
    HIP_OK(hipGetLastError());
    return TISSUE_OK;
  });
}
