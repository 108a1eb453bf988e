// The fused step's kernels D and P on the small fields' tiles, 8 to 24 cells a
// side (see pfs_step.hip).

#include "pfs_step_launch.h"

namespace pfs {

namespace {

template <int H, bool LAST, int TS>
__global__ __launch_bounds__((Geo<H, TS>::NT)) void k_diffuse(DiffuseArgs a) {
    diffuse_tile<H, LAST, TS>(a, xcd_tile(blockIdx.x, a.ntiles));
}

template <int TS>
DiffuseFn diffuse_for_ts(int H, bool last) {
    if (!last) return H == kMaxChunk ? k_diffuse<kMaxChunk, false, TS> : nullptr;
    switch (H) {
#define PFS_CASE(h) \
    case h:         \
        return k_diffuse<h, true, TS>;
        PFS_H_CASES(PFS_CASE)
#undef PFS_CASE
    }
    return nullptr;
}

}  // namespace

DiffuseFn diffuse_small_for(int H, bool last, int side) {
    switch (side) {
#define PFS_CASE(t) \
    case t:         \
        return diffuse_for_ts<t>(H, last);
        PFS_SMALL_SIDES(PFS_CASE)
#undef PFS_CASE
    }
    return nullptr;
}

PressureFn pressure_small_for(int H, bool last, int side) {
    switch (side) {
#define PFS_CASE(t) \
    case t:         \
        return pressure_for_ts<t>(H, last);
        PFS_SMALL_SIDES(PFS_CASE)
#undef PFS_CASE
    }
    return nullptr;
}

}  // namespace pfs
