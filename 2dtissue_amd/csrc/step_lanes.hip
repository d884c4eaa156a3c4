// The step kernel for one layout of its sums (STEP_LANES) and number of physical lanes (STEP_P), both given
// by the build: the instantiations are compiled side by side.
#define TISSUE_STEP_KERNEL
#include "step_kernel.h"

namespace tissue {

#define STEP_NAME2(L, P) launch_step_l##L##_p##P
#define STEP_NAME(L, P) STEP_NAME2(L, P)

hipError_t STEP_NAME(STEP_LANES, STEP_P)(int block, bool tape, bool wave, const MeshDev& mesh, const ReplicaDesc* reps,
                                         const TileDesc* tiles, int n_tiles, const BucketSet& bin,
                                         const BucketSet& bout, const BucketSet& bclr, const TiledIO& io,
                                         hipStream_t st) {
  constexpr int L = STEP_LANES, P = STEP_P;
  if constexpr (P <= L) {
    if (stage_occupancy(mesh.nv, block, L, P)) {
      launch_tiled_variant<L, P, true>(block, tape, wave, mesh, reps, tiles, n_tiles, bin, bout, bclr, io, st);
      return hipGetLastError();
    }
  }
  launch_tiled_variant<L, P, false>(block, tape, wave, mesh, reps, tiles, n_tiles, bin, bout, bclr, io, st);
  return hipGetLastError();
}

}  // namespace tissue
