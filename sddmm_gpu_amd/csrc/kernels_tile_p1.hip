// Tile kernels, part 1: the instantiations for value mode 1 (out = val * dot, values in sorted order).
// The kernel template is compiled in several translation units side by side, which
// divides the build time of the slowest file.
#include "kernels_tile_impl.hpp"

namespace sddmm {

TileFn tile_kernel_part1(const TileVariant &v, int vmode, bool gather, int slice, int nwaves, bool ragged)
{
    if (ragged) return ragged_tile_kernel<1>(v, gather, slice, nwaves);
#define SDDMM_PICK_SLICE(g, kpl, vm, nw)                                                                     \
    (slice == 3 || slice == 5 ? fused_slices_kernel<g, kpl, vm, nw, false>(slice)                               \
     : slice == 4 ? (TileFn)sddmm_tile_kernel<g, kpl, vm, nw, false, 4>                                        \
                  : (TileFn)sddmm_tile_kernel<g, kpl, vm, nw, false, 0>)
#define SDDMM_PICK(g, kpl, vm)                                                                              \
    (gather ? gather_tile_kernel<g, kpl, vm>(slice)                                                         \
            : (nwaves == 12 ? SDDMM_PICK_SLICE(g, kpl, vm, 12) : SDDMM_PICK_SLICE(g, kpl, vm, 16)))
#define SDDMM_CASE(g, kpl)                                                                                  \
    if (v.G == g && v.KPL == kpl)                                                                           \
        return SDDMM_PICK(g, kpl, 1);
    SDDMM_CASE(4, 2) SDDMM_CASE(4, 4) SDDMM_CASE(4, 8) SDDMM_CASE(8, 1) SDDMM_CASE(8, 2) SDDMM_CASE(8, 4) SDDMM_CASE(8, 8)
    SDDMM_CASE(16, 4) SDDMM_CASE(16, 8) SDDMM_CASE(32, 4) SDDMM_CASE(32, 8)
#undef SDDMM_CASE
#undef SDDMM_PICK
#undef SDDMM_PICK_SLICE
    return nullptr;
}

}  // namespace sddmm
