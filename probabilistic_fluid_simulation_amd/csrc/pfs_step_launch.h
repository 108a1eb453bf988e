// The fused step's square-tile kernels by halo, place in the step and tile side;
// the sides of small fields compile in pfs_step_small.hip, the others in
// pfs_step.hip.
#pragma once

#include "pfs_internal.h"
#include "pfs_step_kernels.h"

namespace pfs {

using DiffuseFn = void (*)(DiffuseArgs);
using PressureFn = void (*)(PressureArgs);

// Halos of a last chunk; one that is not the last runs kMaxChunk or kLongChunk
// sweeps.
#define PFS_H_CASES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11)

// Tile sides of small fields, and of the others.
#define PFS_SMALL_SIDES(X) X(8) X(12) X(16) X(20) X(24)
#define PFS_LARGE_SIDES(X) X(32) X(36) X(40) X(48) X(56) X(64)

DiffuseFn diffuse_small_for(int H, bool last, int side);
PressureFn pressure_small_for(int H, bool last, int side);

namespace {

template <int H, bool LAST, int TS>
__global__ __launch_bounds__((Geo<H, TS>::NT)) void k_pressure(PressureArgs a) {
    pressure_tile<H, LAST, TS>(a, xcd_tile(blockIdx.x, a.ntiles));
}

template <int TS>
PressureFn pressure_for_ts(int H, bool last) {
    if (!last) return H == kLongChunk ? k_pressure<kLongChunk, false, TS> : k_pressure<kMaxChunk, false, TS>;
    switch (H) {
#define PFS_CASE(h) \
    case h:         \
        return k_pressure<h, true, TS>;
        PFS_H_CASES(PFS_CASE)
#undef PFS_CASE
    }
    return nullptr;
}

}  // namespace
}  // namespace pfs
