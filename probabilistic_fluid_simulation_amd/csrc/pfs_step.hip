// Fused, temporally blocked fluid step for gfx950.
//
// One call of the reference's simulate_fluid_step (src/fluid.cpp:298-310)
// is 2K+3 full-grid passes there.  Here it is two kernels (for K <= 10):
//
//   D: advect (src/fluid.cpp:24-70) + K diffusion sweeps (:129-196) +
//      divergence (:221-237), temporally blocked in LDS;
//   P: K pressure sweeps (:239-266) + gradient subtraction (:269-296),
//      temporally blocked in LDS, optionally followed by the dye advection
//      of the same cells (:72-127) when one call runs the whole timestep of
//      the reference driver (src/main.cpp:222-225).
//
// Each workgroup owns a tile of cells and stages it plus a halo of H = sweeps
// (+1 for the final stencil) cells, periodic wrap folded into the staged
// coordinates.  Two forms:
//   - square tiles (8 to 64 wide: kernel P, and kernel D on small fields, up to
//     side 24; pfs_step_kernels.h): thread (x, seg) owns column x of the staged region,
//     rows [seg*S, seg*S + S), in registers; every sweep it publishes its cells
//     (alpha-scaled for diffusion) to an LDS plane, waits at one barrier
//     (planes alternate), and updates its cells from the left/right columns in
//     LDS and its own registers above and below;
//   - wave tiles (kernel D on every larger field; pfs_wave_kernels.h):
//     a wavefront owns whole rows and takes its horizontal neighbours by DPP.
// Cells of the outer ring read clamped or missing neighbours and become
// garbage; that ring grows by one cell per sweep exactly as the valid region
// shrinks, so the tile is never touched by it.  Halo cells are recomputed by
// both neighbouring tiles with the same operations in the same order: every
// value is bit-identical to the reference's global sweep.  For K > 10 the
// sweeps run in chunks of 8 or 10 with the iterate in workspace planes between
// chunks.
//
// Buffer contract (equal to fluid.cpp's, derived from its pointer swaps):
// with P = vp and Q = tmp at entry, E = D^K if K is even else D^(K-1),
// warm = Q[2] if K is even else P[2] (the pressure start), p^0 = warm:
//   Q = (E.u, E.v, p^K, b)     P = (E - grad p^K, p^(K-1), b)
// b = divergence of D^K.  Kernel D only reads vp and tmp: it writes the
// pressure start, b and E to workspace planes (16 B per cell), so that
// kernel P's halo reads never race with its own writes, and kernel P writes
// both outputs whole (32 B per cell) without reading them.

#include <cmath>
#include <initializer_list>

#include "pfs_internal.h"
#include "pfs_step_launch.h"
#include "pfs_wave_kernels.h"

namespace pfs {

namespace {

// Larger fields.
template <int H, bool FIRST, bool LAST, int S>
__global__ __launch_bounds__(kWaveMax * 64, S == 2 ? 8 : 6) void k_diffuse_wave(DiffuseArgs a) {
    diffuse_wave<H, FIRST ? From::Advect : From::Plane, LAST ? To::Step : To::Plane, S>(
        a, xcd_tile(blockIdx.x, a.ntiles));
}

// Chunks of the pressure that are not the last, on larger fields.
__global__ __launch_bounds__(kWaveMax * 64, 8) void k_pressure_wave(PressureArgs a) {
    pressure_wave<kMaxChunk, From::Plane, To::Plane, 4>(a, xcd_tile(blockIdx.x, a.ntiles));
}

// The operators diffuse and computePressure.
template <int H, From FROM, To TO, int S>
__global__ __launch_bounds__(kWaveMax * 64, S == 2 ? 8 : 6) void k_diffuse_op(DiffuseArgs a) {
    diffuse_wave<H, FROM, TO, S>(a, xcd_tile(blockIdx.x, a.ntiles));
}

template <int H, From FROM, To TO, int S>
__global__ __launch_bounds__(kWaveMax * 64, S == 2 ? 8 : 6) void k_pressure_op(PressureArgs a) {
    pressure_wave<H, FROM, TO, S>(a, xcd_tile(blockIdx.x, a.ntiles));
}

// ---- host dispatch over the compile-time halo and tile side ----------------
template <int S>
DiffuseFn diffuse_wave_for(int H, bool first, bool last) {
    if (!last && H == kLongChunk)
        return first ? k_diffuse_wave<kLongChunk, true, false, S> : k_diffuse_wave<kLongChunk, false, false, S>;
    if (!last)
        return first ? k_diffuse_wave<kMaxChunk, true, false, S> : k_diffuse_wave<kMaxChunk, false, false, S>;
    switch (H) {
#define PFS_CASE(h) \
    case h:         \
        return first ? k_diffuse_wave<h, true, true, S> : k_diffuse_wave<h, false, true, S>;
        PFS_H_CASES(PFS_CASE)
#undef PFS_CASE
    }
    return nullptr;
}

PressureFn pressure_for(int H, bool last, int ts) {
    switch (ts) {
#define PFS_CASE(t) \
    case t:         \
        return pressure_for_ts<t>(H, last);
        PFS_LARGE_SIDES(PFS_CASE)
#undef PFS_CASE
    }
    return pressure_small_for(H, last, ts);
}

template <int TS>
int threads_for_ts(int H) {
    switch (H) {
#define PFS_CASE(h) \
    case h:         \
        return Geo<h, TS>::NT;
        PFS_H_CASES(PFS_CASE)
#undef PFS_CASE
    }
    return 0;
}

// The wave shape of one field's launch with halo H; sets the launch's tile
// counts (of DiffuseArgs or PressureArgs) to it.
template <typename Args>
WaveShape wave_args(Args &d, int H) {
    const WaveShape sh =
        wave_shape(H, device_cus(), [&](WaveShape s) { return wave_tiles(d.w, d.h, H, s); });
    d.tiles_x = wave_tiles_x(d.w, H);
    d.ntiles = (int)wave_tiles(d.w, d.h, H, sh);
    return sh;
}

// An operator's sweeps in launches.  The first reads the field and writes
// planes, the last reads planes and writes both fields (a launch that read a
// field and wrote one would race with its own halo reads), so there are at
// least two: 4 + the rest up to 8 sweeps, else 8 (or 10, sweeps_per_launch) at a
// time and the rest last.
struct OpPlan {
    int first, middles, last;
};
OpPlan op_plan(int iters, int w, int h) {
    if (iters <= kMaxChunk) return {4, 0, iters - 4};
    int n = kMaxChunk;
    if (iters > kLongChunk) {
        DiffuseArgs longer{};
        longer.w = w;
        longer.h = h;
        (void)wave_args(longer, kLongChunk);
        n = sweeps_per_launch(iters, longer.ntiles <= device_cus());
    }
    const int rest = (iters - 1) % n + 1;
    return {n, (iters - rest) / n - 1, rest};
}

template <int S>
DiffuseFn diffuse_op_for(int ns, From from, To to) {
    if (to == To::Plane) {
        if (from == From::Plane) return diffuse_wave_for<S>(ns, false, false);
        return ns == 4           ? k_diffuse_op<4, From::Field, To::Plane, S>
               : ns == kMaxChunk ? k_diffuse_op<kMaxChunk, From::Field, To::Plane, S>
                                 : k_diffuse_op<kLongChunk, From::Field, To::Plane, S>;
    }
    switch (ns) {
#define PFS_CASE(n) \
    case n:         \
        return k_diffuse_op<n, From::Plane, To::Field, S>;
        PFS_CASE(1) PFS_CASE(2) PFS_CASE(3) PFS_CASE(4) PFS_CASE(5) PFS_CASE(6) PFS_CASE(7) PFS_CASE(8)
        PFS_CASE(9) PFS_CASE(10)
#undef PFS_CASE
    }
    return nullptr;
}

template <int S>
PressureFn pressure_op_for(int ns, From from, To to) {
    if (to == To::Plane) {
        if (from == From::Plane)
            return ns == kMaxChunk ? k_pressure_op<kMaxChunk, From::Plane, To::Plane, S>
                                   : k_pressure_op<kLongChunk, From::Plane, To::Plane, S>;
        return ns == 4           ? k_pressure_op<4, From::Field, To::Plane, S>
               : ns == kMaxChunk ? k_pressure_op<kMaxChunk, From::Field, To::Plane, S>
                                 : k_pressure_op<kLongChunk, From::Field, To::Plane, S>;
    }
    switch (ns) {
#define PFS_CASE(n) \
    case n:         \
        return k_pressure_op<n, From::Plane, To::Field, S>;
        PFS_CASE(1) PFS_CASE(2) PFS_CASE(3) PFS_CASE(4) PFS_CASE(5) PFS_CASE(6) PFS_CASE(7) PFS_CASE(8)
        PFS_CASE(9) PFS_CASE(10)
#undef PFS_CASE
    }
    return nullptr;
}

}  // namespace

int threads_for(int H, int ts) {
    switch (ts) {
#define PFS_CASE(t) \
    case t:         \
        return threads_for_ts<t>(H);
        PFS_SMALL_SIDES(PFS_CASE)
        PFS_LARGE_SIDES(PFS_CASE)
#undef PFS_CASE
    }
    return 0;
}

size_t fused_workspace_bytes(int w, int h) {
    return scene_ws_floats(w, h, kMaxChunk + 1) * sizeof(float);
}

// The side of the square tiles for a step: the smallest of its class (of all,
// tile 0) whose tiles the CUs hold at once.  Small tiles keep a launch's
// chain of phases short, a second round of workgroups on part of the CUs costs
// up to half the launch again.  Diffusion + pressure at 8 sweeps, us, by side:
// 128^2 8: 8.7, 12: 9.3, 16: 10.2; 320x240 16 (300 tiles): 13.8, 20: 11.5, 24:
// 12.4; 360^2 24: 13.1, 32: 15.2.  The pressure alone: 611x397 32 (260 tiles) 12.8,
// 36: 8.7; 800x600 48: 12.2, 56: 13.6, 64: 15.2; past a tile a CU at 64, two at 48
// or 56: 1100x1024 48: 19.2, 56: 21.4, 64: 24.5, 1200x1024 56: 21.8, 64: 25.0.  Where
// 64 just fits, pairs of 48 depend on the sweeps: a 1024^2 step 36.6 (48) against
// 37.9 (64) at 8, 55.2 against 56.6 at 16, but 33.0 against 31.4 at 4: left at 64.
int tile_side(int tile, int w, int h) {
    const int cus = device_cus();
    auto smallest = [&](std::initializer_list<int> sides) {
        for (int side : sides)
            if (tile_count(w, h, side) <= cus) return side;
        return 0;
    };
    int side = 0;
    if (tile == 16 || tile == 0) side = smallest({8, 12, 16, 20, 24});
    if (side || tile == 16) return side ? side : 16;
    if (tile == 32 || tile == 0) side = smallest({32, 36, 40});
    if (side || tile == 32) return side ? side : 32;
    if ((side = smallest({48, 56, 64}))) return side;
    for (int two : {48, 56})  // two workgroups a CU
        if (tile_count(w, h, two) <= 2 * cus) return two;
    return 64;
}

int fused_step(const StepArgs &s, float *ws, hipStream_t stream, hipEvent_t *ev, int reps) {
    if (s.iters < 1) return set_error(PFS_ERR_INVALID, "fused step needs iters >= 1");
    Chunk plan[64], pplan[64];  // the diffusion's and the pressure's launches
    if (s.iters > 64 * kMaxChunk)
        return set_error(PFS_ERR_UNSUPPORTED, "iters too large for one step plan");
    if (s.tile != 0 && !valid_tile_side(s.tile))
        return set_error(PFS_ERR_INVALID, "tile side must be 16, 32 or 64");
    const int side = tile_side(s.tile, s.w, s.h);
    const bool small = side <= 24;
    DiffuseArgs d = diffuse_args(s.P, s.Q, s.w, s.h, s.dt, s.visc, s.iters, ws, side);
    PressureArgs p = pressure_args(s.P, s.Q, s.image, s.itmp, s.w, s.h, s.dt, ws, side);
    const dim3 grid(d.ntiles);
    DiffuseArgs longer = d;
    if (!small) (void)wave_args(longer, kLongChunk);
    const int nd = chunk_plan(s.iters, plan, 64,
                              sweeps_per_launch(s.iters, !small && longer.ntiles <= device_cus()));
    const int np = chunk_plan(s.iters, pplan, 64, sweeps_per_launch(s.iters, d.ntiles <= device_cus()));

    if (!ev) reps = 1;
    if (ev) PFS_HIP_TRY(hipEventRecord(ev[0], stream));
    for (int r = 0; r < reps; ++r)
        for (int c = 0; c < nd; ++c) {
            diffuse_chunk(d, c, plan[c], ws);
            const Chunk &k = plan[c];
            if (small) {
                hipLaunchKernelGGL(diffuse_small_for(k.H, k.last, side), grid,
                                   dim3(threads_for(k.H, side)), 0, stream, d);
            } else {
                DiffuseArgs w = d;
                const WaveShape sh = wave_args(w, k.H);
                hipLaunchKernelGGL(sh.S == 2 ? diffuse_wave_for<2>(k.H, k.first, k.last)
                                             : diffuse_wave_for<4>(k.H, k.first, k.last),
                                   dim3(w.ntiles), dim3(64 * sh.nw), 0, stream, w);
            }
            PFS_TRY(check_launch("fused diffuse"));
        }
    if (ev) PFS_HIP_TRY(hipEventRecord(ev[1], stream));
    if (ev) PFS_HIP_TRY(hipEventRecord(ev[2], stream));
    for (int r = 0; r < reps; ++r)
        for (int c = 0; c < np; ++c) {
            pressure_chunk(p, c, pplan[c], ws, s.image, s.itmp, nd);
            const Chunk &k = pplan[c];
            PressureArgs w = p;
            // Only whole chunks of fields with two workgroups for every CU:
            // below that the square tiles are as fast (2048^2: 22.5 us against
            // 24; 1024^2: equal).
            const WaveShape sh = k.last || side < 48 ? WaveShape{0, 0} : wave_args(w, k.H);
            if (sh.S == 4 && k.H == kMaxChunk && w.ntiles >= 2 * device_cus())
                hipLaunchKernelGGL(k_pressure_wave, dim3(w.ntiles), dim3(64 * sh.nw), 0, stream, w);
            else
                hipLaunchKernelGGL(pressure_for(k.H, k.last, side), grid,
                                   dim3(threads_for(k.H, side)), 0, stream, p);
            PFS_TRY(check_launch("fused pressure"));
        }
    if (ev) PFS_HIP_TRY(hipEventRecord(ev[3], stream));
    return PFS_OK;
}

// The operators' sweeps (include/fluid.hpp's diffuse and computePressure) in
// the step's wave tiles.  a holds the input; on return the last iterate is in
// `last` and the one before it in `before` (the two fields, in the order the
// reference's pointer swaps leave them).  Other channels keep their values.
// Workspace (floats, N = w*h): the iterates of u and v in [0, 2N) and [2N, 4N),
// the divergence in [4N, 5N) and the iterates of p in [5N, 6N) and [6N, 7N).  (Both
// operators in the same 4N: 640x480 at 30 sweeps, all operators in turn 65.7 us
// against 64.1, each one's planes then lying in the XCDs' L2s for the other.)
size_t op_workspace_bytes(int w, int h) { return 7 * (size_t)w * h * sizeof(float); }

int diffuse_op(const float *a, float *last, float *before, int w, int h, float dt, float visc,
               int iters, float *ws, hipStream_t stream) {
    DiffuseArgs d = diffuse_args(a, a, w, h, dt, visc, iters, ws);
    float2 *plane[2] = {reinterpret_cast<float2 *>(ws), reinterpret_cast<float2 *>(ws) + (size_t)w * h};
    d.field[0] = last;
    d.field[1] = before;
    const OpPlan plan = op_plan(iters, w, h);
    const int n = plan.middles + 2;
    for (int c = 0; c < n; ++c) {
        const int ns = c == 0 ? plan.first : c == n - 1 ? plan.last : plan.first;
        const From from = c == 0 ? From::Field : From::Plane;
        const To to = c == n - 1 ? To::Field : To::Plane;
        d.dsrc = plane[(c + 1) & 1];
        d.ddst = plane[c & 1];
        const WaveShape sh = wave_args(d, ns);
        hipLaunchKernelGGL(sh.S == 2 ? diffuse_op_for<2>(ns, from, to) : diffuse_op_for<4>(ns, from, to),
                           dim3(d.ntiles), dim3(64 * sh.nw), 0, stream, d);
        PFS_TRY(check_launch("diffuse"));
    }
    return PFS_OK;
}

int pressure_op(float *a, float *last, float *before, int w, int h, float dt, int iters, float *ws,
                hipStream_t stream) {
    PressureArgs p = pressure_args(a, a, nullptr, nullptr, w, h, dt, ws);
    float *plane[2] = {ws + 5 * (size_t)w * h, ws + 6 * (size_t)w * h};
    p.gamma = pressure_gamma(dt);
    p.bpl = p.bdst = ws + 4 * (size_t)w * h;
    p.field[0] = last;
    p.field[1] = before;
    const OpPlan plan = op_plan(iters, w, h);
    const int n = plan.middles + 2;
    for (int c = 0; c < n; ++c) {
        const int ns = c == 0 ? plan.first : c == n - 1 ? plan.last : plan.first;
        const From from = c == 0 ? From::Field : From::Plane;
        const To to = c == n - 1 ? To::Field : To::Plane;
        p.psrc = plane[(c + 1) & 1];
        p.pdst = plane[c & 1];
        const WaveShape sh = wave_args(p, ns);
        hipLaunchKernelGGL(sh.S == 2 ? pressure_op_for<2>(ns, from, to) : pressure_op_for<4>(ns, from, to),
                           dim3(p.ntiles), dim3(64 * sh.nw), 0, stream, p);
        PFS_TRY(check_launch("computePressure"));
    }
    return PFS_OK;
}

}  // namespace pfs
