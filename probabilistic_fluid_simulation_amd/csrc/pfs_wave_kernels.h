// Wave-tiled bodies of the fused step (gfx950): the large-field form of the
// diffusion body in pfs_step_kernels.h, with the same arithmetic in the same
// order.
//
// A wavefront owns S whole rows of a 128-cell wide region, lane l the cells
// 2l and 2l + 1 of each, all in registers.  A cell's horizontal neighbours
// are its lane's other cell and a neighbouring lane's, which the DPP wave
// shifts deliver as an operand of the addition itself; its vertical
// neighbours are in the same lane, except at the first and last of the
// wave's rows, which the waves of a workgroup exchange through LDS (two rows
// written and two read per wave and sweep, one barrier).
//
// What bounds it, and why this shape.  The sweeps are bound by VALU issue and
// by the exchange's latency.  gfx950 issues plain FP32 additions, products
// and FMAs of two wavefronts together (2.4 cycles per instruction and SIMD
// measured, 4.5 alone), but an operation with a DPP operand keeps those around
// it from pairing, and two operations with an SGPR operand do not pair with
// each other: so a sweep issues its DPP additions in one group and reads its
// constants from VGPRs, and two or more workgroups share a CU.  Per value and
// sweep: one product (alpha), the four additions of the reference, the
// division in two operations, half a min3 for its range test.
// Measured (1024^2 / 2048^2 at 8 sweeps, 3840x2160 at 30, all launches of the
// diffusion): square tiles 25.9 / 96.9 / 511 us; this form 18.6 / 51 / 241 us.
// Of that, before the back-trace lost its wraps (near_trace), the ring of one
// cell around the staged velocities (without it the region's outermost cells
// trace out of it in every wave and gather from memory) took 23.9 / 63.9 / 285 to
// 21.1 / 54.2 / 261 at 12 waves of 4 rows.
#pragma once

#include <type_traits>

#include "pfs_step_kernels.h"

namespace pfs {

constexpr int kWaveRX = 128;  // cells across a wave's region: two per lane
constexpr int kWaveMax = 16;  // wavefronts of a workgroup, at most

template <int H_>
struct WaveGeo {
    static constexpr int H = H_;
    static constexpr int HX = H_ + (H_ & 1);  // halo columns: even, so that a lane's two cells share a side
    static constexpr int TX = kWaveRX - 2 * HX;
};

// The value of the lane to the left (right); 0 for the first (last) lane,
// whose cells are halo that no result depends on.
__device__ __forceinline__ float from_left(float x) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));  // wave_shr:1
}
__device__ __forceinline__ float from_right(float x) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));  // wave_shl:1
}

// A wave's place in its tile: region column 0 is global column x0, the
// wave's rows are region rows [r0, r0 + S).
template <int H, int S>
struct WaveTile {
    using G = WaveGeo<H>;
    int lane, wave, nw, ry, r0, x0, y0, xc;
    int gi[2];
    bool inside;  // the region does not wrap in x
    __device__ WaveTile(int tile, int tiles_x, int w, int h) {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        nw = blockDim.x >> 6;
        ry = nw * S;
        r0 = wave * S;
        x0 = (tile % tiles_x) * G::TX - G::HX;
        y0 = (tile / tiles_x) * (ry - 2 * H) - H;
        xc = x0 + 2 * lane;
        inside = x0 >= 0 && x0 + kWaveRX <= w;
        gi[0] = column(2 * lane, w);
        gi[1] = column(2 * lane + 1, w);
    }
    // Global column of region column c.
    __device__ int column(int c, int w) const {
        int g = x0 + c;
        if (w >= kWaveRX) {
            g = g < 0 ? g + w : g;
            return g >= w ? g - w : g;
        }
        return wrap_index(g, w);
    }
    __device__ int first_row(int h) const { return wrap_index(y0 + r0, h); }
    static __device__ int next_row(int g, int h) { return g + 1 == h ? 0 : g + 1; }
    // Region row r0 + k holds tile cells inside the field.
    __device__ bool row_mine(int k, int h) const {
        const int r = r0 + k;
        return r >= H && r < ry - H && y0 + r < h;
    }
    // Column 2 * lane + c holds tile cells inside the field.
    __device__ bool col_mine(int c, int w) const {
        return lane >= G::HX / 2 && lane < (kWaveRX - G::HX) / 2 && xc + c < w;
    }
};

// Two neighbouring values at an address with the alignment of one.
template <typename T>
struct Pair {
    T a, b;
};
__device__ __forceinline__ void store_pair(float *p, float a, float b, bool two) {
    if (two)
        *reinterpret_cast<Pair<float> *>(p) = {a, b};
    else
        *p = a;
}
__device__ __forceinline__ void store_pair(float2 *p, float2 a, float2 b, bool two) {
    if (two)
        *reinterpret_cast<Pair<float2> *>(p) = {a, b};
    else
        *p = a;
}

// x in a VGPR of its own.  Two uses: constants that the sweep's instructions
// read as VGPRs; and the sweep loop's values, which are loaded and stored as
// vectors: left as parts of those vectors across the loop, the register
// allocator of ROCm 7.2 gave one of them and a temporary the same register
// (seen in the assembly, and in the results).  So what a sweep loop carries or
// reads and what was loaded as part of a vector takes a register of its own
// before the loop, and u, v and the pressure again before they are stored as one.
// The source does not tell which of them would fare badly without: every
// instance of these kernels is compared bit for bit (tests/test_gpu_every_kernel.py).
__device__ __forceinline__ float own_register(float x) {
    float y;
    asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
    return y;
}

// Where a launch's cells come from and go to.
enum class From {
    Plane,   // the iterate plane of the chunk before
    Advect,  // the step's first chunk: vp, advected
    Field    // an operator's first chunk: the field itself
};
enum class To {
    Plane,  // the iterate plane
    Step,   // the step's last chunk: E, the divergence and the pressure start
    Field   // an operator's last chunk: the last two iterates into the two fields
};

template <int H, From FROM, To TO, int S, bool COMP = false>
__device__ __forceinline__ void diffuse_wave(const DiffuseArgs &a, int tile) {
    constexpr bool FIRST = FROM == From::Advect, LAST = TO == To::Step;
    constexpr int NS = H - (LAST ? 1 : 0);
    constexpr int NWMAX = kWaveMax;
    constexpr int XB = NWMAX * 2 * 64;  // one exchange buffer: two rows per wave
    // The staged velocities: the region and a ring of one cell around it, so
    // that no back-trace of less than a cell leaves them.
    constexpr int VP = kWaveRX + 2;  // row pitch
    constexpr int VN = FIRST ? ((NWMAX * S + 2) * VP + 1) / 2 : 0;
    __shared__ float4 lds[VN > 2 * XB ? VN : 2 * XB];

    const WaveTile<H, S> t(tile, a.tiles_x, a.w, a.h);
    float u[S][2], v[S][2];
    if (FIRST) {
        const float2 *__restrict__ P2 = reinterpret_cast<const float2 *>(a.P);
        float2 *V = reinterpret_cast<float2 *>(lds) + VP + 1;  // region cell (0, 0)
        {
            // Coalesced: the wave's rows, cells lane and lane + 64 of each;
            // then the ring.
            const int c0 = t.column(t.lane, a.w), c1 = t.column(t.lane + 64, a.w);
            int gj = t.first_row(a.h);
            float2 f[S][2];
#pragma unroll
            for (int k = 0; k < S; ++k) {
                f[k][0] = P2[2 * (gj * a.w + c0)];
                f[k][1] = P2[2 * (gj * a.w + c1)];
                gj = t.next_row(gj, a.h);
            }
            const int ring = 2 * (VP + t.ry);
            for (int e = threadIdx.x; e < ring; e += blockDim.x) {
                const int m = e - 2 * VP;
                const int ry = m >= 0 ? (m >> 1) : (e < VP ? -1 : t.ry);
                const int rx = m >= 0 ? ((m & 1) ? kWaveRX : -1) : (e < VP ? e : e - VP) - 1;
                V[ry * VP + rx] = P2[2 * (wrap_index(t.y0 + ry, a.h) * a.w + wrap_index(t.x0 + rx, a.w))];
            }
#pragma unroll
            for (int k = 0; k < S; ++k) {
                V[(t.r0 + k) * VP + t.lane] = f[k][0];
                V[(t.r0 + k) * VP + t.lane + 64] = f[k][1];
            }
        }
        __syncthreads();
        // Every cell's back-trace (src/fluid.cpp:36-67), its corners from the
        // staged velocities.  A trace that near_trace does not take is redone
        // below, so that this loop has no branch.
        const float fi[2] = {(float)t.gi[0], (float)t.gi[1]};
        const int kx[2] = {a.w + t.gi[0] - (2 * t.lane + 1), a.w + t.gi[1] - (2 * t.lane + 2)};
        auto trace_of = [&](int k, int q, int gj, float2 c) {
            return near_trace(a, fi[q], (float)gj, c, kx[q], a.h + gj - (t.r0 + k + 1), VP, t.ry + 2);
        };
        unsigned long long off = 0;
        int gj = t.first_row(a.h);
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const float2 c2[2] = {V[(t.r0 + k) * VP + 2 * t.lane], V[(t.r0 + k) * VP + 2 * t.lane + 1]};
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const Near r = trace_of(k, q, gj, c2[q]);
                off |= __ballot(!r.on);
                const float2 *F = reinterpret_cast<const float2 *>(lds) + (r.on ? r.ry * VP + r.rx : 0u);
                const float2 f00 = F[0], f10 = F[1], f01 = F[VP], f11 = F[VP + 1];
                u[k][q] = bilerp(r.sx, r.sy, f00.x, f10.x, f01.x, f11.x);
                v[k][q] = bilerp(r.sx, r.sy, f00.y, f10.y, f01.y, f11.y);
            }
            gj = t.next_row(gj, a.h);
            __builtin_amdgcn_sched_barrier(0);  // one row's corners in registers at a time
        }
        if (off != 0) {
#pragma unroll 1
            for (int m = 0; m < 2 * S; ++m) {
                const int k = m >> 1, q = m & 1;
                const float2 c = V[(t.r0 + k) * VP + 2 * t.lane + q];
                const int row = wrap_index(t.y0 + t.r0 + k, a.h);
                if ((q ? trace_of(k, 1, row, c) : trace_of(k, 0, row, c)).on) continue;
                const float2 n = far_advect(a, q ? t.gi[1] : t.gi[0], row, c);
#pragma unroll
                for (int kk = 0; kk < S; ++kk)
#pragma unroll
                    for (int qq = 0; qq < 2; ++qq)
                        if (2 * kk + qq == m) {
                            u[kk][qq] = n.x;
                            v[kk][qq] = n.y;
                        }
            }
        }
        __syncthreads();  // the exchange buffers lie over the staged velocities
    } else if (FROM == From::Field) {
        const float2 *__restrict__ F2 = reinterpret_cast<const float2 *>(a.P);
        int gj = t.first_row(a.h);
#pragma unroll
        for (int k = 0; k < S; ++k) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float2 c = F2[2 * (gj * a.w + t.gi[q])];
                u[k][q] = c.x;
                v[k][q] = c.y;
            }
            gj = t.next_row(gj, a.h);
        }
    } else {
        int gj = t.first_row(a.h);
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const float2 *row = a.dsrc + gj * a.w;
            Pair<float2> c;
            if (t.inside) {
                c = *reinterpret_cast<const Pair<float2> *>(row + t.xc);
            } else {
                c.a = row[t.gi[0]];
                c.b = row[t.gi[1]];
            }
            u[k][0] = c.a.x;
            v[k][0] = c.a.y;
            u[k][1] = c.b.x;
            v[k][1] = c.b.y;
            gj = t.next_row(gj, a.h);
        }
    }

    const bool col0 = t.col_mine(0, a.w), col1 = t.col_mine(1, a.w);
    const int cell0 = (t.y0 + t.r0) * a.w + t.xc;  // of row 0; rows are a.w apart

    // The tile cells' pressure start (last chunk): copied to its plane, the
    // loads (a whole 16-byte cell for 4 bytes when they come from tmp)
    // streaming in under the sweeps.
    float warm[S][2];
    auto warm_ok = [&](int k, int z) {
        const int c = t.lane + 64 * z;
        return t.row_mine(k, a.h) && c >= WaveGeo<H>::HX && c < kWaveRX - WaveGeo<H>::HX && t.x0 + c < a.w;
    };
    const int wcell = (t.y0 + t.r0) * a.w + t.x0 + t.lane;
    if (LAST) {
        const float *__restrict__ W = a.k_even ? a.Q : a.P;
#pragma unroll
        for (int k = 0; k < S; ++k)  // other cells load cell 0, unused
#pragma unroll
            for (int z = 0; z < 2; ++z)
                warm[k][z] = W[4 * (warm_ok(k, z) ? wcell + k * a.w + 64 * z : 0) + 2];
    }

    auto store_field = [&](float *f) {  // channels 0 and 1 of an operator's field
        float2 *F2 = reinterpret_cast<float2 *>(f);
#pragma unroll
        for (int k = 0; k < S; ++k)
            if (t.row_mine(k, a.h) && col0) {
                F2[2 * (cell0 + k * a.w)] = make_float2(u[k][0], v[k][0]);
                if (col1) F2[2 * (cell0 + k * a.w + 1)] = make_float2(u[k][1], v[k][1]);
            }
    };
    auto store_uv = [&]() {  // the iterate, or E
#pragma unroll
        for (int k = 0; k < S; ++k)
            if (t.row_mine(k, a.h) && col0)
                store_pair(a.ddst + cell0 + k * a.w, make_float2(u[k][0], v[k][0]),
                           make_float2(u[k][1], v[k][1]), col1);
    };

    const int top_row = max(2 * t.wave - 1, 0) * 64 + t.lane;  // the outermost waves meet their own row
    const int bot_row = min(2 * t.wave + 2, 2 * t.nw - 1) * 64 + t.lane;
    const float scale = own_register(COMP ? 1.0f : a.alpha);
    const FixedDiv db{own_register(a.db.hi), own_register(a.db.lo), 1};
    auto each = [&](auto &&f) {
#pragma unroll
        for (int k = 0; k < S; ++k) {
            f(u[k][0]);
            f(v[k][0]);
            f(u[k][1]);
            f(v[k][1]);
        }
    };
    each([](float &x) { x = own_register(x); });
    // One sweep reads c, the rows as their neighbours add them (alpha-scaled,
    // or raw for COMP), and lr, the sum of every cell's two horizontal
    // neighbours.
    float4 c[S], lr[S];
    auto scaled = [&](int k) {
        return COMP ? make_float4(u[k][0], v[k][0], u[k][1], v[k][1])
                    : make_float4(scale * u[k][0], scale * v[k][0], scale * u[k][1], scale * v[k][1]);
    };
    auto publish = [&](int s) {  // the wave's outer rows, for sweep s
        float4 *X = lds + (s & 1) * XB;
        c[0] = scaled(0);
        c[S - 1] = scaled(S - 1);
        X[2 * t.wave * 64 + t.lane] = c[0];
        X[(2 * t.wave + 1) * 64 + t.lane] = c[S - 1];
    };
    // The other rows, then all the DPP operations together: each one keeps
    // the operations around it from pairing with another wave's.
    auto sides = [&]() {
#pragma unroll
        for (int k = 1; k < S - 1; ++k) c[k] = scaled(k);
        if constexpr (!COMP) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < S; ++k)
                lr[k] = make_float4(from_left(c[k].z) + c[k].z, from_left(c[k].w) + c[k].w,
                                    from_right(c[k].x) + c[k].x, from_right(c[k].y) + c[k].y);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Row k's numerators, left in (u, v); lo: their least magnitude.
    auto numerators = [&](int k, const float4 &T, const float4 &B, float &lo) {
        if constexpr (COMP) {
            const float4 C = c[k];
            u[k][0] = diffuse_num_comp(from_left(C.z), C.z, T.x, B.x, C.x, a.alpha);
            v[k][0] = diffuse_num_comp(from_left(C.w), C.w, T.y, B.y, C.y, a.alpha);
            u[k][1] = diffuse_num_comp(C.x, from_right(C.x), T.z, B.z, C.z, a.alpha);
            v[k][1] = diffuse_num_comp(C.y, from_right(C.y), T.w, B.w, C.w, a.alpha);
        } else {
            u[k][0] = lr[k].x + T.x + B.x + 1.0f * u[k][0];
            v[k][0] = lr[k].y + T.y + B.y + 1.0f * v[k][0];
            u[k][1] = lr[k].z + T.z + B.z + 1.0f * u[k][1];
            v[k][1] = lr[k].w + T.w + B.w + 1.0f * v[k][1];
        }
        lo = fminf(lo, fminf(fabsf(u[k][0]), fabsf(v[k][0])));
        lo = fminf(lo, fminf(fabsf(u[k][1]), fabsf(v[k][1])));
    };
    // Exactly rounded division of rows by beta, tested for the whole wave:
    // two operations where the host has proven them, else five, else (a
    // numerator out of their range) element by element.
    auto divide = [&](bool outer, float lo) {
        auto rows = [&](auto &&f) {
#pragma unroll
            for (int k = 0; k < S; ++k)
                if ((k == 0 || k == S - 1) == outer) {
                    f(u[k][0]);
                    f(v[k][0]);
                    f(u[k][1]);
                    f(v[k][1]);
                }
        };
        const bool above_lo = __all(lo >= 0x1p-96f);
        if (above_lo && a.fast_div == 2) {
            rows([&](float &x) { x = div_fast2(x, db); });
        } else {
            float hi = 0.0f;
            rows([&](float &x) { hi = fmaxf(hi, fabsf(x)); });
            if (above_lo && a.fast_div != 0 && __all(hi < 0x1p96f))
                rows([&](float &x) { x = div_fast(x, a.beta, a.rcp_beta); });
            else
                rows([&](float &x) { x = div_fixed(x, a.beta, a.rcp_beta, a.fast_div != 0); });
        }
    };
    // A sweep is ordered so that the exchange hides behind arithmetic: the
    // inner rows' numerators while the outer rows' neighbours are read, and
    // the inner rows' division after the outer rows are published for the
    // next sweep, before the barrier.
    auto sweep = [&](int s, auto more) {
        const float4 *X = lds + (s & 1) * XB;
        const float4 above = X[top_row], below = X[bot_row];
        float lo = 0x1p127f, lo_outer = 0x1p127f;
#pragma unroll
        for (int k = 1; k < S - 1; ++k) numerators(k, c[k - 1], c[k + 1 < S ? k + 1 : k], lo);
        numerators(0, above, S > 1 ? c[S > 1 ? 1 : 0] : below, lo_outer);
        if (S > 1) numerators(S - 1, c[S > 1 ? S - 2 : 0], below, lo_outer);
        divide(true, lo_outer);
        if (decltype(more)::value) publish(s + 1);
        if (S > 2) divide(false, lo);
        if (decltype(more)::value) {
            sides();
            __syncthreads();
        }
    };
    publish(1);
    sides();
    __syncthreads();
#pragma unroll 1
    for (int s = 1; s < NS; ++s) sweep(s, std::true_type{});
    if (LAST && !a.k_even) store_uv();  // E = D^(K-1)
    if (TO == To::Field) store_field(a.field[1]);
    sweep(NS, std::false_type{});
    each([](float &x) { x = own_register(x); });

    if (TO == To::Field) {
        store_field(a.field[0]);
        return;
    }
    if (!LAST) {
        store_uv();
        return;
    }
    if (a.k_even) store_uv();
#pragma unroll
    for (int k = 0; k < S; ++k)
#pragma unroll
        for (int z = 0; z < 2; ++z)
            if (warm_ok(k, z)) a.pw[wcell + k * a.w + 64 * z] = warm[k][z];

    // Divergence of D^K on the tile (src/fluid.cpp:221-237).  The buffer
    // written here was last read in sweep NS - 1, which every thread has left.
    float2 *X = reinterpret_cast<float2 *>(lds + ((NS + 1) & 1) * XB);
    X[2 * t.wave * 64 + t.lane] = make_float2(v[0][0], v[0][1]);
    X[(2 * t.wave + 1) * 64 + t.lane] = make_float2(v[S - 1][0], v[S - 1][1]);
    __syncthreads();
    const float2 above = X[top_row], under = X[bot_row];
#pragma unroll
    for (int k = 0; k < S; ++k) {
        const float t0 = k == 0 ? above.x : v[k > 0 ? k - 1 : 0][0];
        const float t1 = k == 0 ? above.y : v[k > 0 ? k - 1 : 0][1];
        const float b0 = k == S - 1 ? under.x : v[k + 1 < S ? k + 1 : k][0];
        const float b1 = k == S - 1 ? under.y : v[k + 1 < S ? k + 1 : k][1];
        const float d0 = a.gamma * ((u[k][1] - from_left(u[k][1])) + (b0 - t0));
        const float d1 = a.gamma * ((from_right(u[k][0]) - u[k][0]) + (b1 - t1));
        if (t.row_mine(k, a.h) && col0) {
            const int cell = cell0 + k * a.w;
            store_pair(a.bpl + cell, d0, d1, col1);
        }
    }
}

// H pressure sweeps (src/fluid.cpp:240-257) in the same layout: a chunk of the
// step that is not its last (Plane to Plane), or of the operator
// computePressure, whose first chunk also forms the divergence
// (src/fluid.cpp:221-237) of the field it reads and whose last writes the
// last two iterates and the divergence into both fields.
// Bound, like the diffusion's sweeps, by VALU issue; one value a cell and no
// division.  3840x2160, 8 sweeps: 33 us against 39 us for the square tiles
// (whose LDS traffic is 7 rows written and 16 read a wave and sweep).
template <int H, From FROM, To TO, int S>
__device__ __forceinline__ void pressure_wave(const PressureArgs &a, int tile) {
    constexpr int NS = H;
    constexpr int XB = kWaveMax * 2 * 64;
    __shared__ float2 lds[2 * XB];

    const WaveTile<H, S> t(tile, a.tiles_x, a.w, a.h);
    const int top_row = max(2 * t.wave - 1, 0) * 64 + t.lane;
    const int bot_row = min(2 * t.wave + 2, 2 * t.nw - 1) * 64 + t.lane;
    const bool col0 = t.col_mine(0, a.w), col1 = t.col_mine(1, a.w);
    const int cell0 = (t.y0 + t.r0) * a.w + t.xc;
    float2 c[S], rhs[S], lr[S];
    if (FROM == From::Field) {
        const float4 *__restrict__ F4 = reinterpret_cast<const float4 *>(a.P);
        float4 f[S][2];
        int gj = t.first_row(a.h);
#pragma unroll
        for (int k = 0; k < S; ++k) {
            f[k][0] = F4[gj * a.w + t.gi[0]];
            f[k][1] = F4[gj * a.w + t.gi[1]];
            gj = t.next_row(gj, a.h);
        }
        lds[2 * t.wave * 64 + t.lane] = make_float2(f[0][0].y, f[0][1].y);
        lds[(2 * t.wave + 1) * 64 + t.lane] = make_float2(f[S - 1][0].y, f[S - 1][1].y);
        __syncthreads();
        const float2 above = lds[top_row], below = lds[bot_row];
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const int up = k > 0 ? k - 1 : 0, down = k + 1 < S ? k + 1 : k;
            const float2 T = k == 0 ? above : make_float2(f[up][0].y, f[up][1].y);
            const float2 B = k == S - 1 ? below : make_float2(f[down][0].y, f[down][1].y);
            c[k] = make_float2(f[k][0].z, f[k][1].z);
            rhs[k] = make_float2(a.gamma * ((f[k][1].x - from_left(f[k][1].x)) + (B.x - T.x)),
                                 a.gamma * ((from_right(f[k][0].x) - f[k][0].x) + (B.y - T.y)));
        }
    } else {
        const float *__restrict__ src = a.first ? a.pw : a.psrc;
        int gj = t.first_row(a.h);
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const float *sr = src + gj * a.w, *br = a.bpl + gj * a.w;
            if (t.inside) {
                const Pair<float> x = *reinterpret_cast<const Pair<float> *>(sr + t.xc);
                const Pair<float> y = *reinterpret_cast<const Pair<float> *>(br + t.xc);
                c[k] = make_float2(x.a, x.b);
                rhs[k] = make_float2(y.a, y.b);
            } else {
                c[k] = make_float2(sr[t.gi[0]], sr[t.gi[1]]);
                rhs[k] = make_float2(br[t.gi[0]], br[t.gi[1]]);
            }
            gj = t.next_row(gj, a.h);
        }
    }
    const float quarter = own_register(0.25f);
#pragma unroll
    for (int k = 0; k < S; ++k) {
        c[k] = make_float2(own_register(c[k].x), own_register(c[k].y));
        rhs[k] = make_float2(own_register(rhs[k].x), own_register(rhs[k].y));
    }
    // Sweep s reads buffer s & 1 (the divergence's exchange used buffer 0).
    auto publish = [&](int s) {
        float2 *X = lds + (s & 1) * XB;
        X[2 * t.wave * 64 + t.lane] = c[0];
        X[(2 * t.wave + 1) * 64 + t.lane] = c[S - 1];
    };
    auto sides = [&]() {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < S; ++k)
            lr[k] = make_float2(from_left(c[k].y) + c[k].y, from_right(c[k].x) + c[k].x);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto cell = [&](int k, const float2 &T, const float2 &B) {  // / 4 as the exact product by a quarter
        return make_float2((lr[k].x + T.x + B.x + 1.0f * rhs[k].x) * quarter,
                           (lr[k].y + T.y + B.y + 1.0f * rhs[k].y) * quarter);
    };
    auto sweep = [&](int s, auto more) {
        const float2 *X = lds + (s & 1) * XB;
        const float2 above = X[top_row], below = X[bot_row];
        float2 n[S];
#pragma unroll
        for (int k = 1; k < S - 1; ++k) n[k] = cell(k, c[k - 1], c[k + 1 < S ? k + 1 : k]);
        n[0] = cell(0, above, c[1]);
        n[S - 1] = cell(S - 1, c[S - 2], below);
#pragma unroll
        for (int k = 0; k < S; ++k) c[k] = n[k];
        if (decltype(more)::value) {
            publish(s + 1);
            sides();
            __syncthreads();
        }
    };
    auto store_field = [&](float *f) {  // channels 2 and 3 of an operator's field
        float2 *F2 = reinterpret_cast<float2 *>(f);
#pragma unroll
        for (int k = 0; k < S; ++k)
            if (t.row_mine(k, a.h) && col0) {
                F2[2 * (cell0 + k * a.w) + 1] = make_float2(c[k].x, rhs[k].x);
                if (col1) F2[2 * (cell0 + k * a.w + 1) + 1] = make_float2(c[k].y, rhs[k].y);
            }
    };
    publish(1);
    sides();
    __syncthreads();
#pragma unroll 2
    for (int s = 1; s < NS; ++s) sweep(s, std::true_type{});
    if (TO == To::Field) store_field(a.field[1]);
    sweep(NS, std::false_type{});
    if (TO == To::Field) {
        store_field(a.field[0]);
        return;
    }
#pragma unroll
    for (int k = 0; k < S; ++k)
        if (t.row_mine(k, a.h) && col0) {
            store_pair(a.pdst + cell0 + k * a.w, own_register(c[k].x), own_register(c[k].y), col1);
            if (FROM == From::Field) store_pair(a.bdst + cell0 + k * a.w, rhs[k].x, rhs[k].y, col1);
        }
}

// ---- host side: the shape of a launch ---------------------------------------

// S rows per wavefront (2 or 4), nw wavefronts per workgroup.
struct WaveShape {
    int S, nw;
};
inline int wave_tiles_x(int w, int H) {
    const int tx = kWaveRX - 2 * (H + (H & 1));
    return (w + tx - 1) / tx;
}
inline long long wave_tiles(int w, int h, int H, WaveShape s) {
    const int ty = s.S * s.nw - 2 * H;
    return (long long)wave_tiles_x(w, H) * ((h + ty - 1) / ty);
}

// The shape for a launch whose tile count is count(shape):
//   - 2 rows per wave and the fewest waves with which every tile has a CU of
//     its own, if 16 waves do: the sweeps of one tile are a chain of
//     exchanges, and short strips keep it short (512^2, 8 sweeps: 9.3 us with
//     16 waves of 2 rows, 10.8 with 8 of 4; 611x397, 30 sweeps: 29 us against 34);
//   - else 4 rows per wave, likewise (1024^2, 8 sweeps: 20.2 us with 15 waves,
//     250 tiles; 21.1 with 12, 350 tiles);
//   - else `many` waves of 4 rows: 12 make two workgroups per CU, one's memory
//     phases under the other's sweeps (2048^2, 8 sweeps: 54 us; 67 with 16 waves,
//     which leave no room for a second workgroup); the compensated sums, with
//     twice the arithmetic, gain more from 16 waves' narrower share of halo
//     rows (a precise step of 16 + 16 sweeps at 3840x2160 569 -> 539 us, at
//     2048^2 304 -> 303).
template <typename Count>
WaveShape wave_shape(int H, int cus, Count &&count, int many = 12) {
    for (int S = 2; S <= 4; S += 2)
        for (int nw = (2 * H + 4 + S - 1) / S; nw <= kWaveMax; ++nw)
            if (count(WaveShape{S, nw}) <= cus) return {S, nw};
    return {4, many};
}

}  // namespace pfs
