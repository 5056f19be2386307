// Instances of the fused 0D solver kernels for the window width W = 12 (the tile counts
// of this window, and the register levels of the one-pivot-a-step form).  One translation
// unit per window keeps the builds parallel.
#include "bz_ee_lane.h"
#include "bz_solver0d.h"

namespace bz0d {

int steady_w12(const GridDev& g, const BatchDev& b, hipStream_t s, const EEDev* ee) {
  if (g.nslots % 64 == 0) {
    BZ0D_FOR_LEVELS(12, launch_newton_lane, g, b, s, ee)
  }
  BZ0D_FOR_TILES(12, launch_newton, g, b, s, ee)
}

int transient_w12(const GridDev& g, const BatchDev& b, double cdt, const double* ustart, double* avg,
                   hipStream_t s) {
  BZ0D_FOR_TILES(12, launch_transient, g, b, cdt, ustart, avg, s)
}

int ee_factor_w12(const GridDev& g, const BatchDev& b, const int* active, double* lprof, double* z1, double* s1,
                   hipStream_t s) {
  if (g.nslots % 64 != 0) {
    BZ0D_FOR_TILES(12, launch_ee_factor_tiles, g, b, active, lprof, z1, s1, s)
  }
  BZ0D_FOR_LEVELS(12, launch_ee_factor, g, b, active, lprof, z1, s1, s)
}

int ee_apply_w12(const GridDev& g, const BatchDev& b, const int* active, const double* lprof, const double* z1,
                  const double* s1, const double* v, double* out, double* outT, hipStream_t s) {
  return launch_ee_apply<12>(g, b, active, lprof, z1, s1, v, out, outT, s);
}

}  // namespace bz0d
