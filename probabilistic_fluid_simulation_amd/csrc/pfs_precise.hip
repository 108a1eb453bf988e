// Precision form of the fluid step, and its FP64 twin.
//
// No counterpart in the reference, whose Jacobi loops run a fixed count in
// FP32 (src/fluid.cpp:151,239).  The precision form keeps the reference's
// step structure (src/fluid.cpp:298-310) and changes three things:
//
//   - the 5-term stencil sums of both Jacobi sweeps (src/fluid.cpp:19-21)
//     are compensated: Kahan's compensated summation of the neighbours,
//     the product by alpha with its exact FMA error, the diffusion's centre
//     term by TwoSum, so each numerator is rounded once from about twice FP32
//     precision before the division;
//   - every pressure sweep also accumulates, in FP64, the residual of its
//     input iterate, r = b + pL + pR + pT + pB - 4p (zero at the fixed point
//     of the sweep p' = (pL+pR+pT+pB+b)/4), from the compensated sum, and
//     sum b^2 once;
//   - the pressure iteration stops at the first iterate i >= 1 with
//     ||r(p^i)|| <= tol ||b||, at most K sweeps, decided on the device.
//
// Kernels (temporally blocked like the plain step, pfs_step.hip, in the same
// wave tiles, pfs_wave_kernels.h, and square tiles, pfs_step_kernels.h):
//
//   k_diffuse_wave_precise, on small fields k_diffuse_precise
//                         advect + C diffusion sweeps per launch (compensated),
//                         the last launch also the divergence and the
//                         pressure start (diffuse_wave / diffuse_tile with COMP
//                         = true); the first also clears the step's control block
//   k_pressure_precise    C pressure sweeps per launch from an iterate plane,
//                         with the FP64 residual of every iterate the launch
//                         reads on the tile's own cells; launch `launch`
//                         covers iterates launch*C .. launch*C + C.
//
// Every workgroup writes its per-row FP64 sums to its own slot (one per
// tile); the last workgroup of a launch to finish folds each row over the
// tiles in tile order (a fixed order: the totals, and so the early exit, do
// not depend on scheduling) and decides.  The next launch reads that
// decision at entry:
//   - no iterate converged, more sweeps to go: continue from the plane the
//     last launch wrote (planes rotate by launch: launch k reads k % 3 and
//     writes (k+1) % 3);
//   - iterate i converged: re-run the sweeps that end at i from the plane
//     that precedes them, still intact, then the gradient subtraction and the
//     outputs; later launches return at entry.
// The last chunk writes the outputs for Kp = K as it goes; one more launch
// fixes them up when the fold of that chunk finds an earlier converged
// iterate.  So the early exit costs no host round trip.
//
// Buffer contract, with Kd = K the diffusion sweeps and Kp <= K the pressure
// sweeps of the result: E = D^Kd if Kd is even else D^(Kd-1); the pressure
// starts from tmp[2] if Kd is even else vp[2];
//   tmp = (E.u, E.v, p^Kp, b)     vp = (E - grad p^Kp, p^(Kp-1), b)
// which is exactly the reference's step when Kp = Kd (the plain step's
// contract, see pfs_step.hip).
//
// The FP64 twin runs the same contract in double with plain arithmetic, up to
// 8 sweeps per launch and given (Kd, Kp): the yardstick the precision form's
// error is reported against.  With Kd = Kp = K it reproduces the
// reference's algorithm in double exactly.

#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <cstring>
#include <string>
#include <utility>

#include "pfs.h"
#include "pfs_internal.h"
#include "pfs_step_kernels.h"
#include "pfs_wave_kernels.h"

namespace pfs {
namespace {

constexpr int kMaxK = PFS_PRECISE_MAX_ITERS;

// ============================ FP64 twin ======================================
constexpr int kBX = 64, kBY = 4;
constexpr int kRows = 2;  // rows per thread: a block covers kBX x (kBY * kRows) cells

struct Cell {
    int i, j, im, ip, jm, jp;
    __device__ Cell(int w, int h, int i_, int j_) : i(i_), j(j_) {
        im = wrap_minus(i, w);
        ip = wrap_plus(i, w);
        jm = wrap_minus(j, h);
        jp = wrap_plus(j, h);
    }
};

// Calls f(cell) for each of this thread's cells: column blockIdx.x*kBX + x,
// rows kRows apart by kBY within the block's kBY*kRows rows.
template <typename F>
__device__ __forceinline__ void for_cells(int w, int h, F &&f) {
    const int i = blockIdx.x * kBX + threadIdx.x;
    const int j0 = blockIdx.y * (kBY * kRows) + threadIdx.y;
    if (i >= w) return;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int j = j0 + r * kBY;
        if (j < h) f(Cell(w, h, i, j));
    }
}

// Advection of vp[0,1] (src/fluid.cpp:24-70) into the iterate planes u, v.
__global__ __launch_bounds__(kBX *kBY) void k_t_advect(const double *__restrict__ P,
                                                      double *__restrict__ u,
                                                      double *__restrict__ v, int w, int h,
                                                      double dt, double fw, double fh,
                                                      double inv_w, double inv_h, int pow2_w,
                                                      int pow2_h) {
    for_cells(w, h, [&](const Cell &c) {
        const int cell = c.j * w + c.i;
        auto at = [&](int k) { return *reinterpret_cast<const Pair<double> *>(P + 4 * k); };
        const Pair<double> here = at(cell);
        const double xp = (double)c.i - div_n(dt * here.a, fw, inv_w, pow2_w);
        const double yp = (double)c.j - div_n(dt * here.b, fh, inv_h, pow2_h);
        const TraceT<double> t = trace(xp, yp, w, h, fw, fh);
        const Pair<double> f00 = at(t.j0 * w + t.i0), f10 = at(t.j0 * w + t.i1);
        const Pair<double> f01 = at(t.j1 * w + t.i0), f11 = at(t.j1 * w + t.i1);
        u[cell] = bilerp(t.sx, t.sy, f00.a, f10.a, f01.a, f11.a);
        v[cell] = bilerp(t.sx, t.sy, f00.b, f10.b, f01.b, f11.b);
    });
}

// Divergence of D^Kd (src/fluid.cpp:221-237) into b, and the pressure start
// (tmp[2] for even Kd, vp[2] for odd) into iterate plane 0.
__global__ __launch_bounds__(kBX *kBY) void k_t_divergence(const double *__restrict__ u,
                                                          const double *__restrict__ v,
                                                          const double *__restrict__ start,
                                                          double *__restrict__ b,
                                                          double *__restrict__ p0, int w, int h,
                                                          double gamma) {
    for_cells(w, h, [&](const Cell &c) {
        const int cell = c.j * w + c.i;
        const double uR = u[c.j * w + c.ip] - u[c.j * w + c.im];
        const double vT = v[c.jp * w + c.i] - v[c.jm * w + c.i];
        b[cell] = gamma * (uR + vT);
        p0[cell] = start[4 * cell + 2];
    });
}

// Gradient subtraction with p^Kp (src/fluid.cpp:269-296) and the output
// contract.
__global__ __launch_bounds__(kBX *kBY) void k_t_finalize(
    double *__restrict__ P, double *__restrict__ Q, const double *__restrict__ eu,
    const double *__restrict__ ev, const double *__restrict__ pk, const double *__restrict__ pkm1,
    const double *__restrict__ b, int w, int h, double dt) {
    for_cells(w, h, [&](const Cell &c) {
        const int cell = c.j * w + c.i;
        const double pL = pk[c.j * w + c.im], pR = pk[c.j * w + c.ip];
        const double pT = pk[c.jm * w + c.i], pB = pk[c.jp * w + c.i];
        const double gradX = (pR - pL) * dt / 2.0;
        const double gradY = (pB - pT) * dt / 2.0;
        const double ex = eu[cell], ey = ev[cell], bb = b[cell];
        P[4 * cell] = ex - gradX;
        P[4 * cell + 1] = ey - gradY;
        P[4 * cell + 2] = pkm1[cell];
        P[4 * cell + 3] = bb;
        Q[4 * cell] = ex;
        Q[4 * cell + 1] = ey;
        Q[4 * cell + 2] = pk[cell];
        Q[4 * cell + 3] = bb;
    });
}

__device__ __forceinline__ double from_left(double x) {
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true),
        __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double from_right(double x) {
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true),
        __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double own_register(double x) {
    double y;
    asm("v_mov_b64 %0, %1" : "=v"(y) : "v"(x));
    return y;
}

constexpr int kTwinSweeps = 8;  // sweeps per launch, at most

// A launch of ns Jacobi sweeps over planes of doubles; blockIdx.y picks the
// plane (u or v for the diffusion).
struct TwinArgs {
    int w, h, tiles_x, ns;
    const double *src[2];
    double *dst[2];   // the last sweep's iterate
    double *prev[2];  // the one before it, if not null
    const double *rhs;                 // pressure: the divergence
    double alpha, beta, rcp_beta;      // diffusion
    int fast_div;
};

// ns sweeps in the wave layout of pfs_wave_kernels.h: a wavefront owns S whole
// rows of a 128-cell region, two cells a lane, DPP to the sides, the outer
// rows exchanged through LDS.  u and v don't meet in a sweep, so each has its
// own workgroups and a sweep of either kind is one value a cell; the halo is
// ns cells (columns: rounded up to even).  DIFF: src/fluid.cpp:154-185, else
// src/fluid.cpp:240-257, operations and their order as there.  The division
// by beta is Markstein's (see div_fast) where the host allows it and a
// wavefront's numerators lie in [2^-900, 2^900), else IEEE division.
// One launch per sweep was bound by memory and the launches' ends (7.3 and 6.5
// us a sweep at 1001x751, 16 sweeps: 117 and 104 us);
// 8 sweeps a launch are bound by VALU issue and the exchange: 17.9 and 10.1 us a
// launch, 36 and 20 us.
template <int S, bool DIFF>
__global__ __launch_bounds__(kWaveMax * 64) void k_t_sweeps(TwinArgs a) {
    constexpr int XB = kWaveMax * 2 * 64;
    __shared__ double2 lds[2 * XB];
    const int H = a.ns, hx = H + (H & 1), w = a.w, h = a.h;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6, ry = nw * S, r0 = wave * S;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % a.tiles_x) * (kWaveRX - 2 * hx) - hx;
    const int y0 = (tile / a.tiles_x) * (ry - 2 * H) - H;
    const int xc = x0 + 2 * lane;
    const bool inside = x0 >= 0 && x0 + kWaveRX <= w;
    const int g0 = wrap_index(xc, w), g1 = wrap_index(xc + 1, w);
    const bool z = blockIdx.y != 0;
    const double *__restrict__ src = z ? a.src[1] : a.src[0];
    double *dst = z ? a.dst[1] : a.dst[0], *prev = z ? a.prev[1] : a.prev[0];

    auto load = [&](const double *row, double (&f)[2]) {
        Pair<double> c;
        if (inside) {
            c = *reinterpret_cast<const Pair<double> *>(row + xc);
        } else {
            c.a = row[g0];
            c.b = row[g1];
        }
        f[0] = c.a;
        f[1] = c.b;
    };
    double x[S][2], rhs[S][2];
    int gj = wrap_index(y0 + r0, h);
#pragma unroll
    for (int k = 0; k < S; ++k) {
        load(src + gj * w, x[k]);
        if (!DIFF) load(a.rhs + gj * w, rhs[k]);
        gj = gj + 1 == h ? 0 : gj + 1;
    }
#pragma unroll
    for (int k = 0; k < S; ++k)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            x[k][q] = own_register(x[k][q]);
            if (!DIFF) rhs[k][q] = own_register(rhs[k][q]);
        }

    const bool col = lane >= hx / 2 && lane < (kWaveRX - hx) / 2;
    auto store = [&](double *f) {
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const int r = r0 + k, j = y0 + r;
            if (r < H || r >= ry - H || j >= h || !col || xc >= w) continue;
            double *at = f + j * w + xc;
            if (xc + 1 < w)
                *reinterpret_cast<Pair<double> *>(at) = {x[k][0], x[k][1]};
            else
                *at = x[k][0];
        }
    };

    // c: the values as their neighbours add them; lr: the horizontal pairs.
    double c[S][2], lr[S][2];
    const int top_row = max(2 * wave - 1, 0) * 64 + lane;  // the outermost waves meet their own row
    const int bot_row = min(2 * wave + 2, 2 * nw - 1) * 64 + lane;
    auto publish = [&](int s) {  // for sweep s, which reads buffer s & 1
        double2 *X = lds + (s & 1) * XB;
#pragma unroll
        for (int k = 0; k < S; ++k)
#pragma unroll
            for (int q = 0; q < 2; ++q) c[k][q] = DIFF ? a.alpha * x[k][q] : x[k][q];
        X[2 * wave * 64 + lane] = {c[0][0], c[0][1]};
        X[(2 * wave + 1) * 64 + lane] = {c[S - 1][0], c[S - 1][1]};
#pragma unroll
        for (int k = 0; k < S; ++k) {
            lr[k][0] = from_left(c[k][1]) + c[k][1];
            lr[k][1] = c[k][0] + from_right(c[k][0]);
        }
        __syncthreads();
    };
    auto sweep = [&](int s) {
        const double2 *X = lds + (s & 1) * XB;
        const double2 above = X[top_row], below = X[bot_row];
        unsigned worst = 0;
#pragma unroll
        for (int k = 0; k < S; ++k)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const double T = k == 0 ? (q ? above.y : above.x) : c[k > 0 ? k - 1 : 0][q];
                const double B = k == S - 1 ? (q ? below.y : below.x) : c[k + 1 < S ? k + 1 : k][q];
                const double sum = lr[k][q] + T + B + 1.0 * (DIFF ? x[k][q] : rhs[k][q]);
                if (DIFF) {
                    x[k][q] = sum;  // the numerator
                    // |sum| in [2^-900, 2^900), read off the exponent
                    worst = max(worst, ((unsigned)__double2hiint(sum) & 0x7fffffffu) - (123u << 20));
                } else {
                    x[k][q] = sum * 0.25;  // / 4, exactly
                }
            }
        if (!DIFF) return;
        const bool fast = a.fast_div && __all(worst < (1800u << 20));
        if (fast) {
#pragma unroll
            for (int k = 0; k < S; ++k)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const double n = x[k][q];
                    double d = n * a.rcp_beta;
                    d = fma(fma(-d, a.beta, n), a.rcp_beta, d);
                    x[k][q] = fma(fma(-d, a.beta, n), a.rcp_beta, d);
                }
        } else {
#pragma unroll
            for (int k = 0; k < S; ++k)
#pragma unroll
                for (int q = 0; q < 2; ++q) x[k][q] = x[k][q] / a.beta;
        }
    };
    publish(1);
#pragma unroll 1
    for (int s = 1; s < a.ns; ++s) {
        sweep(s);
        publish(s + 1);
    }
    if (prev) store(prev);
    sweep(a.ns);
    store(dst);
}

// Workspace of the twin: four iterate planes (u and v, twice), b and three
// pressure planes.
size_t twin_ws_bytes(int w, int h) { return (size_t)w * h * 8 * sizeof(double); }

// K sweeps, at most kTwinSweeps a launch, as even as possible.  Iterates go
// from cur to next and back; the last one goes to `last`, and the one before
// it to `prev` (unless null), which may be neither cur nor next at that time.
template <bool DIFF>
void twin_sweeps(TwinArgs a, int K, double *const (&cur)[2], double *const (&next)[2],
                 double *const (&last)[2], double *const (&prev)[2], hipStream_t s) {
    const int nchunks = (K + kTwinSweeps - 1) / kTwinSweeps, planes = DIFF ? 2 : 1;
    double *const *from = cur, *const *to = next;
    for (int c = 0; c < nchunks; ++c) {
        a.ns = K / nchunks + (c < K % nchunks);
        const bool end = c + 1 == nchunks;
        for (int z = 0; z < 2; ++z) {
            a.src[z] = from[z];
            a.dst[z] = end ? last[z] : to[z];
            a.prev[z] = end ? prev[z] : nullptr;
        }
        a.tiles_x = wave_tiles_x(a.w, a.ns);
        const WaveShape sh = wave_shape(a.ns, device_cus(), [&](WaveShape x) {
            return planes * wave_tiles(a.w, a.h, a.ns, x);
        });
        const dim3 grid((unsigned)wave_tiles(a.w, a.h, a.ns, sh), planes), block(64 * sh.nw);
        if (sh.S == 2)
            hipLaunchKernelGGL((k_t_sweeps<2, DIFF>), grid, block, 0, s, a);
        else
            hipLaunchKernelGGL((k_t_sweeps<4, DIFF>), grid, block, 0, s, a);
        std::swap(from, to);
    }
}

int twin_step(double *P, double *Q, int w, int h, double dt, double visc, int kd, int kp, void *ws,
              hipStream_t s) {
    const size_t N = (size_t)w * h;
    double *pl[8];
    for (int k = 0; k < 8; ++k) pl[k] = static_cast<double *>(ws) + k * N;
    double *b = pl[4], *p0 = pl[5], *p1 = pl[6], *p2 = pl[7];
    const dim3 grid((w + kBX - 1) / kBX, (h + kBY * kRows - 1) / (kBY * kRows)), block(kBX, kBY);
    const double alpha = visc * dt;
    const double beta = 1.0 + 4.0 * alpha;  // src/fluid.cpp:145
    const double gamma = -1.0 / dt;         // src/fluid.cpp:218
    const bool even = kd % 2 == 0;

    // The chunks before the last alternate between planes {0, 1} and {2, 3};
    // the last reads one pair and leaves E in the other.  For odd Kd, E is
    // D^(Kd-1), and D^Kd lies in p1 and p2 until b is formed.
    double *const A[2] = {pl[0], pl[1]}, *const B[2] = {pl[2], pl[3]}, *const none[2] = {nullptr, nullptr};
    double *const pp[2] = {p1, p2};
    const bool odd_chunks = ((kd + kTwinSweeps - 1) / kTwinSweeps) & 1;
    double *const E[2] = {odd_chunks ? B[0] : A[0], odd_chunks ? B[1] : A[1]};
    hipLaunchKernelGGL(k_t_advect, grid, block, 0, s, P, A[0], A[1], w, h, dt, (double)w, (double)h,
                       1.0 / w, 1.0 / h, (w & (w - 1)) == 0, (h & (h - 1)) == 0);
    TwinArgs a{};
    a.w = w;
    a.h = h;
    a.alpha = alpha;
    a.beta = beta;
    a.rcp_beta = 1.0 / beta;
    a.fast_div = beta >= 0x1p-20 && beta <= 0x1p20;
    if (even)
        twin_sweeps<true>(a, kd, A, B, E, none, s);
    else
        twin_sweeps<true>(a, kd, A, B, pp, E, s);
    hipLaunchKernelGGL(k_t_divergence, grid, block, 0, s, even ? E[0] : p1, even ? E[1] : p2,
                       even ? Q : P, b, p0, w, h, gamma);
    // Pressure: chunks alternate between p0 and p1; the last reads one and
    // writes the other and p2.
    const bool podd = ((kp + kTwinSweeps - 1) / kTwinSweeps) & 1;
    double *pkm1 = podd ? p1 : p0;
    double *const c0[2] = {p0, nullptr}, *const c1[2] = {p1, nullptr}, *const end[2] = {p2, nullptr};
    double *const before[2] = {pkm1, nullptr};
    a.rhs = b;
    twin_sweeps<false>(a, kp, c0, c1, end, before, s);
    hipLaunchKernelGGL(k_t_finalize, grid, block, 0, s, P, Q, E[0], E[1], p2, pkm1, b, w, h, dt);
    return check_launch("FP64 twin step");
}

// ==================== FP32 precision form (temporally blocked) ===============
constexpr int kRowB2 = kMaxK + 1;      // rows 0..kMaxK: sum r(p^i)^2; this row: sum b^2
constexpr int kNRows = kMaxK + 2;
constexpr int kMaxLaunch = kMaxK + 2;  // pressure launches: chunks of >= 1 sweep, the fix-up

// Device-side state of one precision step (cleared by its first diffusion launch).
struct PCtl {
    unsigned count[kMaxLaunch];  // workgroups finished, per pressure launch
    int done;                    // 1: vp and tmp hold the result
    int stop;                    // first converged iterate a fold found, else -1
    int kp;                      // pressure sweeps of the result
    int pad;
    double total[kNRows];        // folded sums
};

struct PreciseArgs {
    float *P, *Q;               // vp, tmp: the outputs
    float *pl[3];               // pressure iterate planes; pl[0] holds the start
    const float *bpl;           // the divergence b
    const float2 *E;            // the diffused velocity the outputs keep
    double *part;               // per-tile FP64 sums, part[row * ntiles + tile]
    PCtl *ctl;
    int w, h, tiles_x, ntiles;
    float dt;
    int K, C, nchunks, launch;  // sweeps, sweeps per launch, chunks, this launch
    double tol2;
};

// Sum over the 64 lanes of a wave by a fixed butterfly: every lane ends
// with the same value, independent of scheduling.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// x plus the value DPP control CTRL moves into this lane (0 where it moves
// none), on the two 32-bit halves of a double.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const int mlo = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWS, 0xf, false);
    const int mhi = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROWS, 0xf, false);
    return x + __hiloint2double(mhi, mlo);
}

// Inclusive scan of x over the wave in a fixed pattern (row_shr 1, 2, 4, 8,
// then row_bcast 15 and 31): lane 63 ends with the wave's sum.  DPP moves
// only, no LDS round trip.
__device__ __forceinline__ double wave_scan_dpp(double x) {
    x = dpp_add<0x111, 0xf>(x);  // row_shr:1
    x = dpp_add<0x112, 0xf>(x);  // row_shr:2
    x = dpp_add<0x114, 0xf>(x);  // row_shr:4
    x = dpp_add<0x118, 0xf>(x);  // row_shr:8
    x = dpp_add<0x142, 0xa>(x);  // row_bcast:15
    x = dpp_add<0x143, 0xc>(x);  // row_bcast:31
    return x;
}

// ctl non-null (the step's first launch): workgroup 0 also clears the
// control block the pressure launches use.
__device__ __forceinline__ void clear_ctl(PCtl *ctl) {
    if (!ctl || blockIdx.x != 0) return;
    for (int k = threadIdx.x; k < kMaxLaunch; k += blockDim.x) ctl->count[k] = 0u;
    for (int k = threadIdx.x; k < kNRows; k += blockDim.x) ctl->total[k] = 0.0;
    if (threadIdx.x == 0) {
        ctl->done = 0;
        ctl->stop = -1;
        ctl->kp = 0;
    }
}

template <int H, bool LAST>
__global__ __launch_bounds__((Geo<H, 16>::NT)) void k_diffuse_precise(DiffuseArgs a, PCtl *ctl) {
    clear_ctl(ctl);
    diffuse_tile<H, LAST, 16, true>(a, xcd_tile(blockIdx.x, a.ntiles));
}

template <int H, bool FIRST, bool LAST, int S>
__global__ __launch_bounds__(kWaveMax * 64, S == 2 ? 8 : 6) void k_diffuse_wave_precise(DiffuseArgs a,
                                                                                      PCtl *ctl) {
    clear_ctl(ctl);
    diffuse_wave<H, FIRST ? From::Advect : From::Plane, LAST ? To::Step : To::Plane, S, true>(a, xcd_tile(blockIdx.x, a.ntiles));
}

// What a pressure launch does: the same in every workgroup, from the state the
// launches before it left.
struct PTask {
    bool run;     // false: nothing to do
    bool finish;  // re-run to the converged iterate
    bool fin;     // write the outputs
    int src, b0, ns;  // input plane, its iterate number, sweeps
};
__device__ __forceinline__ PTask pressure_task(const PreciseArgs &a) {
    const int done = a.ctl->done, stop = a.ctl->stop;
    PTask t{};
    if (done) return t;
    t.run = true;
    if (stop >= 0) {
        // The fold of launch k = launch - 1 (iterates kC .. kC + C - 1) found
        // iterate `stop`: re-run from launch k's input, or from launch k-1's
        // when `stop` is launch k's input itself (stop >= 1, so k >= 1 then).
        const int k = a.launch - 1, kb = k * a.C;
        t.finish = t.fin = true;
        if (stop > kb) {
            t.src = k % 3;
            t.b0 = kb;
        } else {
            t.src = (k + 2) % 3;
            t.b0 = kb - a.C;
        }
        t.ns = stop - t.b0;
    } else if (a.launch < a.nchunks) {
        t.src = a.launch % 3;
        t.b0 = a.launch * a.C;
        t.ns = min(a.C, a.K - t.b0);
        t.fin = a.launch == a.nchunks - 1;
    } else {
        t.run = false;  // the fix-up launch, with nothing to fix
    }
    return t;
}

// A launch's end: this workgroup's FP64 sums go to its slots, and the last
// workgroup to finish folds every row over the tiles and decides.
// wsum[m][wave]: the residual sums of sweep m + 1 (m < C); rK and b2 are this
// thread's shares of r(p^K)^2 and b^2; the workgroup has NT = blockDim.x
// threads.  (A release fence in place of count_finished's wait, at 2048^2
// and 16 sweeps: 369 us a step against 339.)
template <int NSLOT, int NWMAX>
__device__ __forceinline__ void end_launch(const PreciseArgs &a, const PTask &t, int tile, double rK,
                                           double b2, double (&wsum)[NSLOT][NWMAX],
                                           double (&rowsum)[NSLOT], int &last_group) {
    constexpr int C = NSLOT - 2;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, NW = blockDim.x >> 6;
    const bool fin = t.fin;
    const int b0 = t.b0, ns = t.ns;
    auto put = [&](int row, double v) {
        __hip_atomic_store(a.part + (size_t)row * a.ntiles + tile, v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    };
    if (!t.finish) {
        const double tk = wave_sum(rK), tb = wave_sum(b2);
        if (lane == 0) {
            wsum[C][wv] = tk;
            wsum[C + 1][wv] = tb;
        }
        __syncthreads();
        if ((int)threadIdx.x < NSLOT) {
            double t = 0.0;
            for (int w = 0; w < NW; ++w) t += wsum[threadIdx.x][w];
            rowsum[threadIdx.x] = t;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int m = 0; m < ns; ++m) put(b0 + m, rowsum[m]);
            if (fin) put(a.K, rowsum[C]);
            if (a.launch == 0) put(kRowB2, rowsum[C + 1]);
        }
    }
    // ---- the last workgroup of the launch folds and decides -----------------
    if (threadIdx.x == 0) {
        last_group = count_finished(&a.ctl->count[a.launch]) == (unsigned)a.ntiles - 1u;
    }
    __syncthreads();
    if (!last_group) return;
    if (t.finish) {
        if (threadIdx.x == 0) {
            a.ctl->kp = b0 + ns;
            a.ctl->done = 1;
        }
        return;
    }
    // Slot m of this launch is row b0 + m (m < ns), then row K (fin), then
    // b^2 (launch 0).  Wave w folds slots w, w + NW, ... over the tiles:
    // lane j sums tiles j, j + 64, ... with four accumulators in a fixed
    // pattern, then the butterfly; every total is the same on every run.
    const int nrow = ns + (fin ? 1 : 0) + (a.launch == 0 ? 1 : 0);
    for (int m = wv; m < nrow; m += NW) {
        const int row = m < ns ? b0 + m : (fin && m == ns ? a.K : kRowB2);
        const double *src = a.part + (size_t)row * a.ntiles;
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        int i = lane;
        for (; i + 192 < a.ntiles; i += 256) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                acc[q] += __hip_atomic_load(src + i + 64 * q, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        }
        for (int q = 0; i < a.ntiles; i += 64, ++q)
            acc[q] += __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const double tot = wave_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
        if (lane == 0) {
            a.ctl->total[row] = tot;
            rowsum[m] = tot;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const double b2 = a.launch == 0 ? rowsum[nrow - 1] : a.ctl->total[kRowB2];
        const double lim = a.tol2 * b2;
        int found = -1;
        for (int m = b0 >= 1 ? 0 : 1; m < ns; ++m)
            if (rowsum[m] <= lim) {
                found = b0 + m;
                break;
            }
        if (found >= 0) {
            a.ctl->stop = found;
        } else if (fin) {
            a.ctl->kp = a.K;
            a.ctl->done = 1;
        }
    }
}


// Up to C = H - 1 compensated pressure sweeps of one tile, the residual of
// every iterate they read, and (on the launch that ends the solve) the
// gradient subtraction and the outputs.  See the file comment for the
// launch sequence.
// NTMAX = 512: at most 128 VGPRs, so that two workgroups share a CU.
template <int H, int TS, int NTMAX>
__global__ __launch_bounds__((Geo<H, TS, NTMAX>::NT))
__attribute__((amdgpu_waves_per_eu(NTMAX == 512 ? 4 : 1))) void k_pressure_precise(PreciseArgs a) {
    using G = Geo<H, TS, NTMAX>;
    constexpr int S = G::S, RX = G::RX, RY = G::RY, PL = G::RYP * RX;
    constexpr int C = H - 1;      // most sweeps of one launch
    constexpr int NW = G::NT / 64;
    constexpr int NSLOT = C + 2;  // rows one launch adds: C residuals, r(p^K), b^2
    __shared__ float plane[2 * PL];
    __shared__ double wsum[NSLOT][NW];
    __shared__ double rowsum[NSLOT];
    __shared__ int last_group;

    const PTask task = pressure_task(a);
    if (!task.run) return;
    const bool fin = task.fin;
    const int ns = task.ns;
    const int tile = xcd_tile(blockIdx.x, a.ntiles);
    const Strip<G> st(threadIdx.x, tile, a.tiles_x, a.w, a.h);
    const float *__restrict__ in = a.pl[task.src];
    float p[S], rhs[S];
    double b2 = 0.0;
#pragma unroll
    for (int k = 0; k < S; ++k) {
        const int g = st.row_ok(k) ? st.gj[k] * a.w + st.gi : 0;
        p[k] = in[g];
        rhs[k] = a.bpl[g];
    }
    if (a.launch == 0) {
#pragma unroll
        for (int k = 0; k < S; ++k) b2 += st.mine(k, a.w, a.h) ? (double)rhs[k] * rhs[k] : 0.0;
    }
    // E, which only the outputs need: loaded before the sweeps so that its
    // latency hides behind them, except in 512-thread workgroups, whose
    // longer strips leave no registers for it.
    constexpr bool kEarlyE = NTMAX == 1024;
    float2 e[S];
    if (kEarlyE && fin) {
#pragma unroll
        for (int k = 0; k < S; ++k) e[k] = a.E[st.mine(k, a.w, a.h) ? st.cell(k, a.w) : 0];
    }

    // Sweeps (src/fluid.cpp:240-257), p' = RN(s - k) / 4 with (s, k) the
    // compensated L + R + T + B + b; the residual of the iterate read,
    // r = (s - 4p) - k in FP64, on the tile's own cells, summed over the
    // thread's rows, then over the wave (DPP) into wsum[s - 1][wave].
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int s = 1; s <= C; ++s) {
        if (s > ns) break;
        float *B = plane + (s & 1) * PL;
#pragma unroll
        for (int k = 0; k < S; ++k)
            if (st.active) B[(st.r0 + k) * RX + st.x] = p[k];
        __syncthreads();
        double racc = 0.0;
        if (st.active) {
            const float top = B[(st.r0 > 0 ? st.r0 - 1 : 0) * RX + st.x];
            const float bot = B[(st.r0 + S < RY ? st.r0 + S : RY - 1) * RX + st.x];
            const float *Bl = B + st.r0 * RX + st.xl, *Br = B + st.r0 * RX + st.xr;
            float prev = top;
#pragma unroll
            for (int k = 0; k < S; ++k) {
                const float cur = p[k];
                const float below = k == S - 1 ? bot : p[k + 1];
                float sv, kv;
                pressure_sum_comp(Bl[k * RX], Br[k * RX], prev, below, rhs[k], sv, kv);
                p[k] = (sv - kv) * 0.25f;
                const double r = fma(-4.0, (double)cur, (double)sv) - (double)kv;
                const double rm = st.mine(k, a.w, a.h) ? r : 0.0;
                racc = fma(rm, rm, racc);
                prev = cur;
            }
        }
        racc = wave_scan_dpp(racc);
        if (lane == 63) wsum[s - 1][wv] = racc;
    }

    double rK = 0.0;
    if (!fin) {
        float *__restrict__ out = a.pl[(a.launch + 1) % 3];
#pragma unroll
        for (int k = 0; k < S; ++k)
            if (st.mine(k, a.w, a.h)) out[st.cell(k, a.w)] = p[k];
    } else {
        // Gradient subtraction (src/fluid.cpp:273-295) and the outputs; the
        // plane written here was last read in sweep ns - 1.  The iterate
        // before the last sweep is what this thread published in it (its own
        // slots of plane ns & 1, which nothing has overwritten).
        float pp[S];
        {
            const float *Bl = plane + (ns & 1) * PL;
#pragma unroll
            for (int k = 0; k < S; ++k) pp[k] = st.active ? Bl[(st.r0 + k) * RX + st.x] : 0.0f;
        }
        float *B = plane + ((ns + 1) & 1) * PL;
        if (!kEarlyE) {
#pragma unroll
            for (int k = 0; k < S; ++k) e[k] = a.E[st.mine(k, a.w, a.h) ? st.cell(k, a.w) : 0];
        }
#pragma unroll
        for (int k = 0; k < S; ++k)
            if (st.active) B[(st.r0 + k) * RX + st.x] = p[k];
        __syncthreads();
        float4 *__restrict__ P4 = reinterpret_cast<float4 *>(a.P);
        float4 *__restrict__ Q4 = reinterpret_cast<float4 *>(a.Q);
#pragma unroll
        for (int k = 0; k < S; ++k) {
            if (!st.mine(k, a.w, a.h)) continue;
            const int o = (st.r0 + k) * RX + st.x;
            const float pL = B[o - 1], pR = B[o + 1], pT = B[o - RX], pB = B[o + RX];
            const float gradX = (pR - pL) * a.dt / 2.0f;
            const float gradY = (pB - pT) * a.dt / 2.0f;
            const int cell = st.cell(k, a.w);
            P4[cell] = make_float4(e[k].x - gradX, e[k].y - gradY, pp[k], rhs[k]);
            Q4[cell] = make_float4(e[k].x, e[k].y, p[k], rhs[k]);
            // Residual of p^K (the solve ran every sweep): FP64 from the floats.
            const double r = fma(-4.0, (double)p[k],
                                 (double)rhs[k] + (((double)pL + (double)pR) +
                                                   ((double)pT + (double)pB)));
            rK = fma(r, r, rK);
        }
    }

    end_launch<NSLOT, NW>(a, task, tile, rK, b2, wsum, rowsum, last_group);
}

// ---- host dispatch --------------------------------------------------------------
using DiffuseFn = void (*)(DiffuseArgs, PCtl *);
using PressureFn = void (*)(PreciseArgs);

// Diffusion launches: chunks of C = 4 or 8 sweeps (halo C), the last one
// of 1..C sweeps (halo 2..C+1).
DiffuseFn diffuse_precise_small(int H, bool last) {
    if (!last) return H == 4 ? k_diffuse_precise<4, false> : H == 8 ? k_diffuse_precise<8, false> : nullptr;
    switch (H) {
#define PFS_CASE(h) \
    case h:         \
        return k_diffuse_precise<h, true>;
        PFS_CASE(2) PFS_CASE(3) PFS_CASE(4) PFS_CASE(5) PFS_CASE(6) PFS_CASE(7) PFS_CASE(8)
        PFS_CASE(9)
#undef PFS_CASE
    }
    return nullptr;
}

template <int S>
DiffuseFn diffuse_precise_wave(int H, bool first, bool last) {
    if (!last) {
        if (H == 4) return first ? k_diffuse_wave_precise<4, true, false, S> : k_diffuse_wave_precise<4, false, false, S>;
        if (H == 8) return first ? k_diffuse_wave_precise<8, true, false, S> : k_diffuse_wave_precise<8, false, false, S>;
        return nullptr;
    }
    switch (H) {
#define PFS_CASE(h) \
    case h:         \
        return first ? k_diffuse_wave_precise<h, true, true, S> : k_diffuse_wave_precise<h, false, true, S>;
        PFS_CASE(2) PFS_CASE(3) PFS_CASE(4) PFS_CASE(5) PFS_CASE(6) PFS_CASE(7) PFS_CASE(8)
        PFS_CASE(9)
#undef PFS_CASE
    }
    return nullptr;
}

template <int H>
PressureFn pressure_precise_h(int ts, bool half) {
    switch (ts) {
#define PFS_CASE(t) \
    case t:         \
        return k_pressure_precise<H, t, 1024>;
        PFS_CASE(16) PFS_CASE(20) PFS_CASE(24) PFS_CASE(32) PFS_CASE(36) PFS_CASE(40) PFS_CASE(48)
        PFS_CASE(56)
#undef PFS_CASE
    }
    return half ? k_pressure_precise<H, 64, 512> : k_pressure_precise<H, 64, 1024>;
}

PressureFn pressure_precise_for(int C, int ts, bool half) {
    return C == 4 ? pressure_precise_h<5>(ts, half) : pressure_precise_h<9>(ts, half);
}

int threads_pressure_precise(int C, int ts, bool half) {
    if (ts == 64 && half) return C == 4 ? Geo<5, 64, 512>::NT : Geo<9, 64, 512>::NT;
    return threads_for(C + 1, ts);
}

// Sweeps per launch (4 or 8) and tile side (16, 32, 64; 0: the plain
// step's rule), process-wide.
std::atomic<int> g_precise_chunk{8};
std::atomic<int> g_precise_tile{0};
// 1: 512-thread pressure workgroups at tile side 64 (two per CU: one's
// loads and barriers overlap the other's sweeps; 0.30 against 0.33 ms per
// 2048^2 step with 1024).
std::atomic<int> g_precise_half{1};

// Workspace: the plain fused step's 8 planes (pressure start, b, two float2
// diffusion planes, two pressure planes), the control block, and the
// per-tile sums for the most tiles any side gives.
constexpr size_t kPCtlBytes = (sizeof(PCtl) + 255) / 256 * 256;
size_t precise_ws_bytes(int w, int h) {
    const size_t N = (size_t)w * h;
    const size_t planes = ((8 * N * sizeof(float)) + 255) / 256 * 256;
    return planes + kPCtlBytes + (size_t)kNRows * (size_t)tile_count(w, h, 16) * sizeof(double) +
           256;
}

// The pressure's side on a field whose side by the rule is ts: the smallest near
// it whose tiles the CUs hold at once, else ts (the workspace's slots hold what
// side 16 gives).  A step of 8 + 8 sweeps at 640x480, side 32 (300 tiles) 43.8 us,
// 36: 36.4; of 16 + 16 at 800x600, 64: 96.7, 48: 85.3; 320x240, 16: 49.7, 20: 46.2.  Past
// one tile a CU side 64's pairs of 512-thread workgroups are the faster
// (1200x1024: 144 us against 152 at side 56).
int pressure_side(int ts, int w, int h) {
    for (int side : {16, 20, 24, 32, 36, 40, 48, 56})
        if ((ts == 16) == (side < 32) && tile_count(w, h, side) <= device_cus()) return side;
    return ts;
}

int precise_step(float *P, float *Q, int w, int h, float dt, float visc, int K, double tol,
                 void *ws, hipStream_t s, PCtl **ctl_out) {
    const int C = g_precise_chunk.load();
    const int forced = g_precise_tile.load();
    const int ts = forced ? forced : tile_for_counts(tile_count(w, h, 64), tile_count(w, h, 32));
    const size_t N = (size_t)w * h;
    char *base = reinterpret_cast<char *>(((uintptr_t)ws + 255) & ~(uintptr_t)255);
    float *wsf = reinterpret_cast<float *>(base);
    PCtl *ctl = reinterpret_cast<PCtl *>(base + ((8 * N * sizeof(float)) + 255) / 256 * 256);
    double *part = reinterpret_cast<double *>(reinterpret_cast<char *>(ctl) + kPCtlBytes);
    *ctl_out = ctl;

    DiffuseArgs d = diffuse_args(P, Q, w, h, dt, visc, K, wsf, ts);
    Chunk plan[kMaxK];
    const int nd = chunk_plan(K, plan, kMaxK, C);
    for (int c = 0; c < nd; ++c) {
        diffuse_chunk(d, c, plan[c], wsf);
        const Chunk &k = plan[c];
        PCtl *clear = c == 0 ? ctl : nullptr;
        if (ts == 16) {
            hipLaunchKernelGGL(diffuse_precise_small(k.H, k.last), dim3(d.ntiles),
                               dim3(threads_for(k.H, ts)), 0, s, d, clear);
        } else {
            DiffuseArgs wd = d;
            const WaveShape sh =
                wave_shape(k.H, device_cus(), [&](WaveShape x) { return wave_tiles(w, h, k.H, x); }, 16);
            wd.tiles_x = wave_tiles_x(w, k.H);
            wd.ntiles = (int)wave_tiles(w, h, k.H, sh);
            hipLaunchKernelGGL(sh.S == 2 ? diffuse_precise_wave<2>(k.H, k.first, k.last)
                                         : diffuse_precise_wave<4>(k.H, k.first, k.last),
                               dim3(wd.ntiles), dim3(64 * sh.nw), 0, s, wd, clear);
        }
        PFS_TRY(check_launch("precise diffuse"));
    }
    PreciseArgs pa{};
    pa.P = P;
    pa.Q = Q;
    pa.pl[0] = wsf;  // d.pw: the pressure start
    pa.pl[1] = wsf + 6 * N;
    pa.pl[2] = wsf + 7 * N;
    pa.bpl = wsf + N;
    pa.E = reinterpret_cast<const float2 *>(wsf + 2 * N + 2 * N * ((nd - 1) & 1));
    pa.part = part;
    pa.ctl = ctl;
    pa.w = w;
    pa.h = h;
    const int side = forced ? forced : pressure_side(ts, w, h);
    pa.tiles_x = (w + side - 1) / side;
    pa.ntiles = (int)tile_count(w, h, side);
    pa.dt = dt;
    pa.K = K;
    pa.C = C;
    pa.nchunks = (K + C - 1) / C;
    pa.tol2 = tol * tol;
    const bool half = g_precise_half.load() != 0;
    const PressureFn pf = pressure_precise_for(C, side, half);
    const int nt = threads_pressure_precise(C, side, half);
    for (int l = 0; l <= pa.nchunks; ++l) {  // the chunks, then the fix-up
        pa.launch = l;
        hipLaunchKernelGGL(pf, dim3(pa.ntiles), dim3(nt), 0, s, pa);
        PFS_TRY(check_launch("precise pressure"));
    }
    return PFS_OK;
}

}  // namespace
}  // namespace pfs

using namespace pfs;

extern "C" {

size_t pfs_precise_workspace_bytes(int vx, int vy, int fp64) {
    if (vx < 1 || vy < 1) return 0;
    return fp64 ? twin_ws_bytes(vx, vy) : precise_ws_bytes(vx, vy);
}

int pfs_set_precise_schedule(int sweeps_per_launch, int tile, int pressure_threads) {
    if (sweeps_per_launch != 0 && sweeps_per_launch != 4 && sweeps_per_launch != 8)
        return set_error(PFS_ERR_INVALID, "sweeps per launch must be 0 (default), 4 or 8");
    if (tile != 0 && !valid_tile_side(tile))
        return set_error(PFS_ERR_INVALID, "tile side must be 0 (automatic), 16, 32 or 64");
    if (pressure_threads != 0 && pressure_threads != 512 && pressure_threads != 1024)
        return set_error(PFS_ERR_INVALID, "pressure threads must be 0 (default), 512 or 1024");
    g_precise_chunk = sweeps_per_launch ? sweeps_per_launch : 8;
    g_precise_tile = tile;
    g_precise_half = pressure_threads != 1024 ? 1 : 0;
    return PFS_OK;
}

int pfs_simulate_fluid_step_precise(pfs_field *vp, pfs_field *tmp, float dt, float viscosity,
                                    int max_iters, double tol, void *workspace,
                                    size_t workspace_bytes, void *stream,
                                    pfs_precise_report *report) {
    PFS_TRY(check_field(vp, "vp", 4));
    PFS_TRY(check_field(tmp, "tmp", 4));
    if (vp->x != tmp->x || vp->y != tmp->y || vp->z != 4 || tmp->z != 4)
        return set_error(PFS_ERR_INVALID, "vp and tmp must both be W x H x 4");
    if (vp->data == tmp->data) return set_error(PFS_ERR_INVALID, "vp and tmp alias");
    if ((uintptr_t)vp->data % 16 || (uintptr_t)tmp->data % 16)
        return set_error(PFS_ERR_UNSUPPORTED, "vp and tmp must be 16-byte aligned");
    if (max_iters < 1 || max_iters > kMaxK)
        return set_error(PFS_ERR_INVALID, "max_iters must be in [1, PFS_PRECISE_MAX_ITERS]");
    if (!(tol >= 0.0)) return set_error(PFS_ERR_INVALID, "tol must be >= 0");
    if (!workspace || workspace_bytes < precise_ws_bytes(vp->x, vp->y))
        return set_error(PFS_ERR_INVALID, "workspace smaller than pfs_precise_workspace_bytes()");
    hipStream_t s = (hipStream_t)stream;
    PCtl *ctl = nullptr;
    PFS_TRY(precise_step(vp->data, tmp->data, vp->x, vp->y, dt, viscosity, max_iters, tol,
                         workspace, s, &ctl));
    if (report) {
        PCtl h;
        PFS_HIP_TRY(hipMemcpyAsync(&h, ctl, sizeof(h), hipMemcpyDeviceToHost, s));
        PFS_HIP_TRY(hipStreamSynchronize(s));
        std::memset(report, 0, sizeof(*report));
        report->iters_used = h.kp;
        report->b_norm = std::sqrt(h.total[kRowB2]);
        report->residual_norm = std::sqrt(h.total[h.kp]);
        for (int k = 0; k <= kMaxK; ++k) report->residual_history[k] = std::sqrt(h.total[k]);
    }
    return PFS_OK;
}

int pfs_simulate_fluid_step_f64(double *vp, double *tmp, int vx, int vy, double dt,
                                double viscosity, int iters_diffuse, int iters_pressure,
                                void *workspace, size_t workspace_bytes, void *stream) {
    if (!vp || !tmp || vp == tmp) return set_error(PFS_ERR_INVALID, "vp/tmp NULL or aliased");
    if (vx < 1 || vy < 1 || (long long)vx * vy * 4 > (long long)INT32_MAX)
        return set_error(PFS_ERR_INVALID, "bad field size");
    if (iters_diffuse < 1 || iters_pressure < 1 || iters_pressure > iters_diffuse ||
        iters_diffuse > kMaxK)
        return set_error(PFS_ERR_INVALID, "need 1 <= iters_pressure <= iters_diffuse <= max");
    if (!workspace || workspace_bytes < twin_ws_bytes(vx, vy))
        return set_error(PFS_ERR_INVALID, "workspace smaller than pfs_precise_workspace_bytes()");
    return twin_step(vp, tmp, vx, vy, dt, viscosity, iters_diffuse, iters_pressure, workspace,
                     (hipStream_t)stream);
}

}  // extern "C"
