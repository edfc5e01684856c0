// kernel_tile.hip -- the 2-D block kernel in FP32 and the host side of both precisions.
#include "tile_device.hpp"

namespace blpg {

#define X(id, nw, tc, rpt, cpt, vr32, vr32w, vr64, vr64w, b32, b64)                    \
  BLPG_TILE_KERNEL(k_tile_f32_##id, float, nw, tc, rpt, cpt, vr32, 1, false)           \
  BLPG_TILE_KERNEL(k_tile_f32w_##id, float, nw, tc, rpt, cpt, vr32w, 1, b32 != 0)
BLPG_TILE_VARIANTS(X)
BLPG_TILE_VARIANTS_F32(X)
#undef X

// warm: the batch carries warm-start lists (block crash where the variant has it)
const void* tile_fn32(int v, bool warm) {
  switch (v) {
#define X(id, nw, tc, rpt, cpt, vr32, vr32w, vr64, vr64w, b32, b64)                    \
  case id:                                                                            \
    return warm ? reinterpret_cast<const void*>(&k_tile_f32w_##id)                    \
                : reinterpret_cast<const void*>(&k_tile_f32_##id);
    BLPG_TILE_VARIANTS(X)
    BLPG_TILE_VARIANTS_F32(X)
#undef X
    default: return nullptr;
  }
}

const void* tile_fn64(int v, bool warm);  // kernel_tile64.hip

constexpr int kTileVariants = 14;
constexpr int kTileDefault = 7;  // static routing by size uses variants 0..6

int tile_variant_count(int) { return kTileVariants; }
int tile_default_variants() { return kTileDefault; }

TileVariant tile_variant(int precision, int v) {
  if (precision == 0 && v >= 13) return TileVariant{1, 8, 1, 1};  // FP32 only
  switch (v) {
#define X(id, nw, tc, rpt, cpt, vr32, vr32w, vr64, vr64w, b32, b64) \
  case id: return TileVariant{nw, (nw * 64) / tc, rpt, cpt};
    BLPG_TILE_VARIANTS(X)
    BLPG_TILE_VARIANTS_F32(X)
#undef X
    default: return TileVariant{1, 8, 1, 1};
  }
}

// the smaller of the cold and warm instantiations' residency
int tile_max_blocks_per_cu(int precision, int v) {
  int best = -1;
  for (int warm = 0; warm < 2; ++warm) {
    const void* fn = precision == 0 ? tile_fn64(v, warm) : tile_fn32(v, warm);
    if (!fn) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, tile_variant(precision, v).nw * 64,
                                                     0) != hipSuccess)
      return 0;
    best = best < 0 || nb < best ? nb : best;
  }
  return best;
}

hipError_t launch_tile(const TileLaunch& L, hipStream_t st) {
  const bool warm = L.warm != nullptr;
  const void* fn = L.precision == 0 ? tile_fn64(L.variant, warm) : tile_fn32(L.variant, warm);
  if (!fn) return hipErrorInvalidValue;
  const int nt = tile_variant(L.precision, L.variant).nw * 64;
  if (L.precision == 0) {
    Opt<double> o{L.eps_d, L.eps_p, L.tol, L.max_iter, L.bland_after};
    void* args[] = {(void*)&L.desc, (void*)&L.pool, (void*)&L.spool, (void*)&L.idx,
                    (void*)&L.count, (void*)&L.count_dev, (void*)&L.queue, (void*)&L.out,
                    (void*)&o, (void*)&L.warm};
    return hipLaunchKernel(fn, dim3(L.grid), dim3(nt), args, 0, st);
  }
  Opt<float> o{(float)L.eps_d, (float)L.eps_p, (float)L.tol, L.max_iter, L.bland_after};
  void* args[] = {(void*)&L.desc, (void*)&L.pool, (void*)&L.spool, (void*)&L.idx,
                  (void*)&L.count, (void*)&L.count_dev, (void*)&L.queue, (void*)&L.out,
                  (void*)&o, (void*)&L.warm};
  return hipLaunchKernel(fn, dim3(L.grid), dim3(nt), args, 0, st);
}

}  // namespace blpg
