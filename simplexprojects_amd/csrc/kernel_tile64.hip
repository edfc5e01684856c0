// kernel_tile64.hip -- the 2-D block kernel in FP64.
#include "tile_device.hpp"

namespace blpg {

#define X(id, nw, tc, rpt, cpt, vr32, vr32w, vr64, vr64w, b32, b64)                    \
  BLPG_TILE_KERNEL(k_tile_f64_##id, double, nw, tc, rpt, cpt, vr64, 2, false)           \
  BLPG_TILE_KERNEL(k_tile_f64w_##id, double, nw, tc, rpt, cpt, vr64w, 2, b64 != 0)
BLPG_TILE_VARIANTS(X)
#undef X

// warm: the batch carries warm-start lists (block crash where the variant has it)
const void* tile_fn64(int v, bool warm) {
  switch (v) {
#define X(id, nw, tc, rpt, cpt, vr32, vr32w, vr64, vr64w, b32, b64)                    \
  case id:                                                                            \
    return warm ? reinterpret_cast<const void*>(&k_tile_f64w_##id)                    \
                : reinterpret_cast<const void*>(&k_tile_f64_##id);
    BLPG_TILE_VARIANTS(X)
#undef X
    default: return nullptr;
  }
}

}  // namespace blpg
