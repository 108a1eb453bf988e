// Particle layer over the grid fluid (gfx950).  No counterpart in the
// reference, which has no particles: these are tracers carried by the grid's
// velocity field, with a uniform neighbour grid over them.
//
//   pfs_particles_advect     x += (dt*u(x))/W, y likewise (the reference's
//                            back-trace, src/fluid.cpp:39-41, run forward),
//                            u bilinear at the position with the reference's
//                            corner keys and blend order (:55-66); positions
//                            wrap back into [0, W) exactly;
//   pfs_ngrid_build          cell keys; a stable LSD radix sort of
//                            (key, particle) pairs, 8- or 10-bit digits: per-block
//                            LDS histograms, a DPP prefix scan, and a scatter
//                            whose in-block ranks come from wavefront ballots;
//                            cell start/end tables (every cell, empty or
//                            not, gets its lower bound, found by searches of
//                            the sorted keys); positions in sorted order;
//   pfs_ngrid_neighbors      neighbour counts, their exclusive scan, and the
//                            lists (CSR) of every particle within radius r,
//                            visiting the 3x3 cells in a fixed order;
//   pfs_ngrid_density        SPH density from the lists' traversal with the
//                            poly6 kernel, FP32 sums in traversal order.
//
// Every integer output (keys, sort order, tables, lists) is deterministic
// and equals the CPU restatement in oracle/pfs_particles.c bit for bit.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>

#include "pfs.h"
#include "pfs_device.h"
#include "pfs_grid.h"
#include "pfs_internal.h"

namespace pfs {
namespace {

constexpr int kThreads = 1024;              // scan kernels, and the sort's large tiles
constexpr int kItems = 4;                   // values or keys per thread
constexpr int kTile = kThreads * kItems;    // values per block
constexpr int kWaves = kThreads / 64;
constexpr int kMaxRadixBits = 10;           // digits of 8 or 10 bits

// ---- wavefront and block scans ------------------------------------------
// Inclusive scan across the 64 lanes: four row shifts (1, 2, 4, 8) give
// every 16-lane row its prefix, then the row totals are carried by the
// row_bcast:15 (into rows 1, 3) and row_bcast:31 (into rows 2, 3) DPP forms.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
    x += __builtin_amdgcn_update_dpp(0u, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0u, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0u, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0u, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0u, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0u, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

// Exclusive scan over a block of NT threads; *total gets the sum.  Uses `sh`
// (NT / 64 + 1 words of LDS).
template <int NT>
__device__ __forceinline__ uint32_t excl_scan(uint32_t x, uint32_t *sh, uint32_t *total) {
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(x);
    if (lane == 63) sh[wave] = inc;
    __syncthreads();
    if (wave == 0) {
        const uint32_t w = lane < NW ? sh[lane] : 0u;
        const uint32_t wi = wave_incl_scan(w);
        if (lane < NW) sh[lane] = wi - w;  // exclusive over waves
        if (lane == NW - 1) sh[NW] = wi;
    }
    __syncthreads();
    const uint32_t out = sh[wave] + inc - x;
    *total = sh[NW];
    __syncthreads();  // sh may be reused by the caller
    return out;
}

// ---- generic exclusive scan (three kernels) --------------------------------
__global__ __launch_bounds__(kThreads) void k_scan_reduce(const uint32_t *__restrict__ in, int n,
                                                          uint32_t *__restrict__ sums) {
    __shared__ uint32_t sh[kWaves + 1];
    const size_t base = (size_t)blockIdx.x * kTile + (size_t)threadIdx.x * kItems;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if (base + k < (size_t)n) s += in[base + k];
    uint32_t total;
    (void)excl_scan<kThreads>(s, sh, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Block b adds up the totals of blocks [0, b) itself (a few hundred at
// most), then scans its tile; the last block also writes the grand total.  sums
// null (few blocks): it adds up their values instead, which out then may not
// overlap.
__global__ __launch_bounds__(kThreads) void k_scan_down(const uint32_t *in, uint32_t *out, int n,
                                                        const uint32_t *__restrict__ sums,
                                                        uint32_t *__restrict__ grand) {
    __shared__ uint32_t sh[kWaves + 1];
    uint32_t before = 0;
    if (sums) {
        for (int j = threadIdx.x; j < (int)blockIdx.x; j += kThreads) before += sums[j];
    } else {
        for (int b = 0; b < (int)blockIdx.x; ++b)
#pragma unroll
            for (int k = 0; k < kItems; ++k) before += in[(size_t)b * kTile + k * kThreads + threadIdx.x];
    }
    uint32_t offset;
    (void)excl_scan<kThreads>(before, sh, &offset);
    const size_t base = (size_t)blockIdx.x * kTile + (size_t)threadIdx.x * kItems;
    uint32_t v[kItems], s = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        v[k] = base + k < (size_t)n ? in[base + k] : 0u;
        s += v[k];
    }
    uint32_t total;
    uint32_t run = offset + excl_scan<kThreads>(s, sh, &total);
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        if (base + k < (size_t)n) out[base + k] = run;
        run += v[k];
    }
    if (grand && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *grand = offset + total;
}

int nblocks_for(size_t n) { return (int)((n + kTile - 1) / kTile); }

// Blocks up to which the scan is one launch, each block reading what precedes
// it: 16,384 values 4.0 us against 6.1 in two launches, 32,768 4.7
// against 6.5.
constexpr int kOneScan = 8;

// Exclusive scan of n values in two kernels (block totals, then blocks
// scanned from the totals before them), or one for few blocks; grand (device, may be null) gets the
// total.  ws: nblocks_for(n) words.  out may be in: the totals then come from a
// launch of their own at any count, since blocks that read what precedes their
// tile would meet what others have written there.
int scan_exclusive(const uint32_t *in, uint32_t *out, int n, uint32_t *grand, uint32_t *ws,
                   hipStream_t s) {
    const int nb = nblocks_for((size_t)n);
    if (nb == 0) return PFS_OK;
    const uintptr_t i0 = (uintptr_t)in, o0 = (uintptr_t)out, bytes = (uintptr_t)n * sizeof *in;
    const bool apart = i0 + bytes <= o0 || o0 + bytes <= i0;
    const bool totals = nb > kOneScan || (nb > 1 && !apart);
    if (totals) hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kThreads), 0, s, in, n, ws);
    hipLaunchKernelGGL(k_scan_down, dim3(nb), dim3(kThreads), 0, s, in, out, n,
                       totals ? ws : nullptr, grand);
    return check_launch("exclusive scan");
}

// ---- stable LSD radix sort of (key, value) pairs ---------------------------
// Digits of RB bits (8 or 10).  The histogram of block b is stored digit
// major, hist[d * nb + b]; each digit's row is then scanned on its own
// (k_digit_rows; up to kFewTiles tiles every scatter block adds its columns
// up itself), and the scatter adds the digit's base, the exclusive scan of the
// row totals, which every scatter block forms for itself.

// Cell of a position in [0, W): (int)(x * kx) with kx = gx / W (float),
// clamped into the grid.
__device__ __forceinline__ int cell_of(float x, float k, int g) {
    const int c = (int)(x * k);
    return c < 0 ? 0 : (c >= g ? g - 1 : c);
}

struct CellKeyArgs {  // the first pass computes the keys from the positions
    const float *x, *y;
    float kx, ky;
    int gx, gy;
};

// The sort's tiles: NT threads of kItems keys each.
template <int NT>
constexpr int sort_tile() {
    return NT * kItems;
}

// Block histograms of one digit.  With FROM_XY the keys are made here from
// the positions, cy * gx + cx, and written to `keys`.
template <int RB, int NT, bool FROM_XY>
__global__ __launch_bounds__(NT) void k_radix_hist(const uint32_t *__restrict__ kin, CellKeyArgs ck,
                                                   uint32_t *__restrict__ keys, int n, int shift,
                                                   uint32_t *__restrict__ hist, int nb) {
    constexpr int R = 1 << RB;
    __shared__ uint32_t h[R];
    for (int d = threadIdx.x; d < R; d += NT) h[d] = 0;
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * sort_tile<NT>();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const size_t i = base + (size_t)r * NT + threadIdx.x;
        if (i < (size_t)n) {
            uint32_t k;
            if (FROM_XY) {
                k = (uint32_t)(cell_of(ck.y[i], ck.ky, ck.gy) * ck.gx + cell_of(ck.x[i], ck.kx, ck.gx));
                keys[i] = k;
            } else {
                k = kin[i];
            }
            atomicAdd(&h[(k >> shift) & (R - 1)], 1u);
        }
    }
    __syncthreads();
    for (int d = threadIdx.x; d < R; d += NT) hist[(size_t)d * nb + blockIdx.x] = h[d];
}

// Block d scans row d of the digit-major histogram (nb tile counts)
// exclusively in place, and writes the row's total to tot[d].
template <int NT>
__global__ __launch_bounds__(NT) void k_digit_rows(uint32_t *__restrict__ hist,
                                                   uint32_t *__restrict__ tot, int nb) {
    __shared__ uint32_t sh[NT / 64 + 1];
    uint32_t *row = hist + (size_t)blockIdx.x * nb;
    uint32_t carry = 0;
    for (int b0 = 0; b0 < nb; b0 += sort_tile<NT>()) {
        const int j = b0 + threadIdx.x * kItems;
        uint32_t v[kItems], s = 0;
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            v[k] = j + k < nb ? row[j + k] : 0u;
            s += v[k];
        }
        uint32_t total;
        uint32_t run = carry + excl_scan<NT>(s, sh, &total);
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            if (j + k < nb) row[j + k] = run;
            run += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

// Workgroups are dispatched to the 8 XCDs in turn (workgroup i to XCD i % 8);
// this numbers tiles so that each XCD takes a contiguous run of them.  Tiles
// next to each other write the two ends of the same output cache lines, which
// then meet in one L2.  A bijection on [0, nb) for any nb.
__device__ __forceinline__ int xcd_block(int i, int nb) {
    const int q = nb >> 3, r = nb & 7, x = i & 7;
    return x * q + min(x, r) + (i >> 3);
}

// Scatter of one pass.  Wave w of a tile takes its kItems * 64 keys from w *
// 256 on in kItems rounds of 64, so the tile's order is (wave, round, lane).
// The rank of an item among equal digits is: the digit's base (scan of the
// digit totals) plus the earlier tiles' count, plus the equal digits of earlier
// waves (per-wave LDS counts, scanned across waves once), plus those of this
// wave's earlier rounds (the wave's running count) and of the lanes below it
// (RB ballots, one per digit bit, intersected).  vin null: the values are the
// key indices.  xs non-null (the last pass): the positions are gathered into
// sorted order as well.  FEW: `rows` is the histogram itself, and each tile
// adds up its few columns (one launch less).
constexpr int kFewTiles = 16;
template <int RB, int NT, bool FEW>
__global__ __launch_bounds__(NT) void k_radix_scatter(
    const uint32_t *__restrict__ kin, const uint32_t *__restrict__ vin, uint32_t *__restrict__ kout,
    uint32_t *__restrict__ vout, int n, int shift, const uint32_t *__restrict__ rows,
    const uint32_t *__restrict__ tot, int nb, const float *__restrict__ x,
    const float *__restrict__ y, float *__restrict__ xs, float *__restrict__ ys) {
    constexpr int R = 1 << RB, NW = NT / 64, TILE = sort_tile<NT>();
    constexpr int DPT = R > NT ? R / NT : 1;  // digits per thread, consecutive
    // The tile in digit order lies over the waves' counts, which it replaces: two
    // large tiles then share a CU.
    constexpr int WORDS = NW * R > 2 * TILE ? NW * R : 2 * TILE;
    __shared__ uint32_t words[WORDS];
    uint32_t(*wcount)[R] = reinterpret_cast<uint32_t(*)[R]>(words);
    uint32_t *lkey = words, *lval = words + TILE;
    __shared__ uint32_t gofs[R], loff[R];
    __shared__ uint32_t sh[NW + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tb = xcd_block(blockIdx.x, nb);  // the tile of this workgroup
    const int d0 = (int)threadIdx.x * DPT;     // this thread's digits (none: d0 >= R)
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const size_t base = (size_t)tb * TILE + (size_t)wave * (kItems * 64) + lane;
    uint32_t key[kItems], val[kItems], dig[kItems], local[kItems];
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const size_t i = base + (size_t)r * 64;
        const bool valid = i < (size_t)n;
        key[r] = valid ? kin[i] : 0u;
        val[r] = valid ? (vin ? vin[i] : (uint32_t)i) : 0u;
    }
    for (int e = threadIdx.x; e < NW * R; e += NT) words[e] = 0;
    {
        uint32_t t[DPT], before[DPT], s = 0;
#pragma unroll
        for (int m = 0; m < DPT; ++m) {
            t[m] = before[m] = 0;
            if (d0 + m < R) {
                const size_t row = (size_t)(d0 + m) * nb;
                if (FEW) {
#pragma unroll
                    for (int b = 0; b < kFewTiles; ++b) {
                        const uint32_t c = b < nb ? rows[row + b] : 0u;
                        t[m] += c;
                        before[m] += b < tb ? c : 0u;
                    }
                } else {
                    t[m] = tot[d0 + m];
                    before[m] = rows[row + tb];
                }
            }
            s += t[m];
        }
        uint32_t all;
        uint32_t dbase = excl_scan<NT>(s, sh, &all);  // its barriers also order the clear
#pragma unroll
        for (int m = 0; m < DPT; ++m)
            if (d0 + m < R) {
                gofs[d0 + m] = dbase + before[m];
                dbase += t[m];
            }
    }
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const bool valid = base + (size_t)r * 64 < (size_t)n;
        const uint32_t d = (key[r] >> shift) & (R - 1);
        dig[r] = d;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t m = __ballot(valid && bit);
            peers &= bit ? m : ~m;
        }
        if (!valid) peers = 0;
        const uint32_t rank = (uint32_t)__popcll(peers & below);
        // The wave's own running count of digit d: read by every lane of
        // the digit, advanced by its lowest lane.  A wave's LDS accesses
        // complete in order, and the wave barrier keeps the compiler from
        // moving the next round's read above this write.
        const uint32_t before = valid ? wcount[wave][d] : 0u;
        local[r] = before + rank;
        if (valid && rank == 0) wcount[wave][d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // Digit counts of the waves -> exclusive across waves; then the tile's
    // first slot of each digit (loff).  The tile is put in digit order in LDS
    // and written out by consecutive threads, so that each store instruction
    // covers a few runs of consecutive positions.
    {
        uint32_t dt[DPT], s = 0;
#pragma unroll
        for (int m = 0; m < DPT; ++m) {
            dt[m] = 0;
            if (d0 + m < R)
                for (int w = 0; w < NW; ++w) {
                    const uint32_t c = wcount[w][d0 + m];
                    wcount[w][d0 + m] = dt[m];
                    dt[m] += c;
                }
            s += dt[m];
        }
        uint32_t all;
        uint32_t lo = excl_scan<NT>(s, sh, &all);
#pragma unroll
        for (int m = 0; m < DPT; ++m)
            if (d0 + m < R) {
                loff[d0 + m] = lo;
                lo += dt[m];
            }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < kItems; ++r)
        local[r] = base + (size_t)r * 64 < (size_t)n ? loff[dig[r]] + wcount[wave][dig[r]] + local[r]
                                                     : (uint32_t)TILE;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r)
        if (local[r] < (uint32_t)TILE) {
            lkey[local[r]] = key[r];
            lval[local[r]] = val[r];
        }
    __syncthreads();
    const int count = (int)min((size_t)TILE, (size_t)n - (size_t)tb * TILE);
    for (int j = threadIdx.x; j < count; j += NT) {
        const uint32_t k = lkey[j], v = lval[j];
        const uint32_t d = (k >> shift) & (R - 1);
        const uint32_t pos = gofs[d] + ((uint32_t)j - loff[d]);
        if (pos < (uint32_t)n) {  // always, when the scans are right: kept as a bound
            kout[pos] = k;
            vout[pos] = v;
            if (xs && v < (uint32_t)n) {
                xs[pos] = x[v];
                ys[pos] = y[v];
            }
        }
    }
}

// ---- grid ------------------------------------------------------------------
// start[c] = the lower bound of cell c in the sorted keys, which is also
// end[c - 1]; the last cell ends at n.  Chains of dependent loads bound this,
// 20 for a binary search of 2^20 keys: two waves of a block of cells find the
// bounds of its first cell and of the next block's, 64 probes at a time (4
// loads), and each cell is then searched between them, in L1.  1,000,000 cells
// and particles: 8.3 -> 6.8 us.
__global__ __launch_bounds__(256) void k_cell_tables(const uint32_t *__restrict__ sk, int n,
                                                     uint32_t *__restrict__ start,
                                                     uint32_t *__restrict__ end, uint32_t ncells) {
    __shared__ uint32_t bracket[2];
    const uint32_t c0 = blockIdx.x * 256, c = c0 + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave < 2) {
        const uint32_t want = c0 + wave * 256;
        uint32_t lo = 0, hi = (uint32_t)n;
        while (lo < hi) {  // the answer stays in [lo, hi]; hi - lo falls below a 64th
            const uint32_t step = (hi - lo + 63) >> 6, p = lo + lane * step;
            const uint32_t less = (uint32_t)__popcll(__ballot(p < hi && sk[p] < want));
            const uint32_t top = lo + less * step;  // the first probe not below, if in range
            if (less) lo = top - step + 1;
            hi = less ? min(hi, top) : lo;
        }
        if (lane == 0) bracket[wave] = lo;
    }
    __syncthreads();
    if (c >= ncells) return;
    uint32_t lo = bracket[0], hi = bracket[1];
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sk[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    start[c] = lo;
    if (c > 0) end[c - 1] = lo;
    if (c + 1 == ncells) end[c] = (uint32_t)n;
}

__global__ void k_gather_u32(const uint32_t *__restrict__ index, const uint32_t *__restrict__ in,
                             uint32_t *__restrict__ out, int n) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t i = index[p];
    out[p] = i < (uint32_t)n ? in[i] : 0u;
}

// x_q - x_p on a periodic axis of length L (half = L/2), positions in
// [0, L): the nearer image.  Across the wrap the far operand is moved by L
// first, exactly (it lies in (L/2, L), so x - L is exact by Sterbenz), and
// the two nearby values are then subtracted with one rounding at their own
// scale; subtracting first would round at L's scale.
__device__ __forceinline__ float periodic_diff(float xq, float xp, float L, float half) {
    const float d = xq - xp;
    const float over = (xq - L) - xp, under = xq - (xp - L);  // both formed: selects, no branches
    return d > half ? over : (d < -half ? under : d);
}

struct NArgs {
    const float *xs, *ys;
    const uint32_t *order;  // null: outputs indexed by sorted position
    const uint32_t *sk, *start, *end;
    int n, gx, gy;
    float W, H, half_w, half_h, r2;
    __device__ uint32_t id(uint32_t p) const { return order ? order[p] : p; }
};

// ---- four (or 16) lanes per particle ----------------------------------------
// The neighbour passes give a particle a quad of lanes: four candidates (or
// listed neighbours) are loaded and evaluated side by side, and order-bound
// sums are then added up one after another, each term broadcast over the quad
// by a DPP operand of its addition, so that every value equals the serial
// walk's.  Against one lane per particle the chain of dependent loads is a
// quarter as long, a wavefront's loads cover consecutive addresses, and a
// small set fills four times as many wavefronts; the sums cost one addition a
// term on every lane.  All four lanes of a quad always run together.
__device__ __forceinline__ int quad_lane() { return (int)(threadIdx.x & 3u); }

template <int J>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t x) {  // lane J's value
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x55 * J, 0xf, 0xf, true);
}
template <int J>
__device__ __forceinline__ float quad_bcast(float x) {
    return __uint_as_float(quad_bcast<J>(__float_as_uint(x)));
}
// s + the quad's four terms in lane order.
__device__ __forceinline__ float quad_add(float s, float t) {
    s += quad_bcast<0>(t);
    s += quad_bcast<1>(t);
    s += quad_bcast<2>(t);
    s += quad_bcast<3>(t);
    return s;
}
__device__ __forceinline__ uint32_t quad_total(uint32_t c) {
    return quad_bcast<0>(c) + quad_bcast<1>(c) + quad_bcast<2>(c) + quad_bcast<3>(c);
}
// Groups of L lanes (4 or 16) a particle: the lane's place in its group, and
// the group's bits of a wave-wide vote.
template <int L>
__device__ __forceinline__ int group_lane() {
    return (int)(threadIdx.x & (L - 1u));
}
template <int L>
__device__ __forceinline__ uint32_t group_vote(bool b) {
    return (uint32_t)(__ballot(b) >> (threadIdx.x & (64u - L))) & ((1u << L) - 1u);
}

// The sorted positions of one row of the 3x3 cells around cell (cx, cy): [s1,
// e1) the row's cells in order up to a wrap, [s2, e2) those after it.  The
// cells of one row are consecutive keys, so without a wrap the three are one
// range, [start of the left cell, end of the right cell).
struct RowRanges {
    uint32_t s1, e1, s2, e2;
};
__device__ __forceinline__ RowRanges row_ranges(const NArgs &a, int cx, int cy, int oy) {
    const int ny = cy + oy < 0 ? cy + oy + a.gy : (cy + oy >= a.gy ? cy + oy - a.gy : cy + oy);
    const uint32_t row = (uint32_t)(ny * a.gx);
    RowRanges r{0, 0, 0, 0};
    if (cx == 0) {  // cells gx-1 | 0, 1
        r.s1 = a.start[row + a.gx - 1];
        r.e1 = a.end[row + a.gx - 1];
        r.s2 = a.start[row];
        r.e2 = a.end[row + 1];
    } else if (cx == a.gx - 1) {  // cells gx-2, gx-1 | 0
        r.s1 = a.start[row + cx - 1];
        r.e1 = a.end[row + cx];
        r.s2 = a.start[row];
        r.e2 = a.end[row];
    } else {
        r.s1 = a.start[row + cx - 1];
        r.e1 = a.end[row + cx + 1];
    }
    r.e1 = min(r.e1, (uint32_t)a.n);
    r.e2 = min(r.e2, (uint32_t)a.n);
    return r;
}

// The three rows' ranges (lo, hi: [k][0] up to a wrap, [k][1] after) of p's
// cell, visited in order: near(q, end, d2_of) for the whole row of a cell away
// from the domain's edges, else any(q, end, d2_of) for each range; d2_of the
// squared periodic distance of a candidate at (x, y) from p.
template <typename Near, typename Any>
__device__ __forceinline__ void visit_rows(const NArgs &a, int p, int cx, int cy,
                                           const uint32_t (&lo)[3][2], const uint32_t (&hi)[3][2],
                                           Near &&near, Any &&any) {
    const float px = a.xs[p], py = a.ys[p];
    const bool big = a.gx >= 7 && a.gy >= 7;
    if (big && cx >= 1 && cx <= a.gx - 2 && cy >= 1 && cy <= a.gy - 2) {
        // No candidate is more than 3 cells away, less than half the domain
        // when it spans 7 or more cells: the periodic correction is the
        // identity.
        near([&](float ox, float oy) {
            const float dx = ox - px, dy = oy - py;
            return dx * dx + dy * dy;
        });
    } else if (big) {
        // Near an edge of a grid of 7 or more cells a side, whether a
        // candidate lies across the wrap is known per range: cell gx-1
        // seen from cell 0 (its candidates lie in (W/2, W): shifted by -W),
        // cell 0 seen from cell gx-1 (p lies there: p shifted by -W), and
        // the same for rows.  Every other candidate is within 2W/7 of p and
        // every shifted one at least 5W/7 away before the shift, so these
        // are exactly the cases periodic_diff corrects, with its values:
        // (x_q + -W) - x_p and (x_q + -0) - (x_p - W).
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float qsy = (cy == 0 && k == 0) ? -a.H : -0.0f;
            const float pyu = (cy == a.gy - 1 && k == 2) ? py - a.H : py;
            auto shifted = [&](float qsx, float pxu) {
                return [=](float ox, float oy_) {
                    const float dx = (ox + qsx) - pxu, dy = (oy_ + qsy) - pyu;
                    return dx * dx + dy * dy;
                };
            };
            any(lo[k][0], hi[k][0], shifted(cx == 0 ? -a.W : -0.0f, px));
            any(lo[k][1], hi[k][1], shifted(-0.0f, cx == a.gx - 1 ? px - a.W : px));
        }
    } else {
        auto d2_of = [&](float ox, float oy) {
            const float dx = periodic_diff(ox, px, a.W, a.half_w);
            const float dy = periodic_diff(oy, py, a.H, a.half_h);
            return dx * dx + dy * dy;
        };
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            any(lo[k][0], hi[k][0], d2_of);
            any(lo[k][1], hi[k][1], d2_of);
        }
    }
}

// Visits every particle q of the 3x3 cells around p's cell, p included (rows
// then columns, -1..1, then q ascending), L at a time: f(q, ok, d2) on the
// group's lanes for consecutive q, ok false past a range's end.
template <int L, typename F>
__device__ __forceinline__ void for_neighbors(const NArgs &a, int p, F &&f) {
    const uint32_t c = a.sk[p];
    if (c >= (uint32_t)a.gx * (uint32_t)a.gy) return;  // a cell by construction: kept as a bound
    const int cx = (int)(c % (uint32_t)a.gx), cy = (int)(c / (uint32_t)a.gx);
    const int l = group_lane<L>();
    // Lane j of a quad finds row j's ranges (lane 3 repeats row 2), all at once.
    const RowRanges r = row_ranges(a, cx, cy, min(quad_lane(), 2) - 1);
    const uint32_t lo[3][2] = {{quad_bcast<0>(r.s1), quad_bcast<0>(r.s2)},
                               {quad_bcast<1>(r.s1), quad_bcast<1>(r.s2)},
                               {quad_bcast<2>(r.s1), quad_bcast<2>(r.s2)}};
    const uint32_t hi[3][2] = {{quad_bcast<0>(r.e1), quad_bcast<0>(r.e2)},
                               {quad_bcast<1>(r.e1), quad_bcast<1>(r.e2)},
                               {quad_bcast<2>(r.e1), quad_bcast<2>(r.e2)}};
    // Positions of candidate q + l of a range ending at end (p's past it).
    auto at = [&](uint32_t q, uint32_t end, float &x, float &y) {
        const uint32_t k = q + l < end ? q + l : (uint32_t)p;
        x = a.xs[k];
        y = a.ys[k];
    };
    auto scan = [&](uint32_t q, uint32_t end, auto &&d2_of) {
        for (; q < end; q += L) {
            float x, y;
            at(q, end, x, y);
            f(q + l, q + l < end, d2_of(x, y));
        }
    };
    visit_rows(
        a, p, cx, cy, lo, hi,
        [&](auto &&d2_of) {  // the first candidates of the three rows loaded together
            float x[3], y[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) at(lo[k][0], hi[k][0], x[k], y[k]);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (lo[k][0] < hi[k][0])
                    f(lo[k][0] + l, lo[k][0] + l < hi[k][0], d2_of(x[k], y[k]));
                scan(lo[k][0] + L, hi[k][0], d2_of);
            }
        },
        scan);
}

// The same visit by one lane per particle, for order-bound sums over sets
// large enough to fill the GPU that way: f(d2) for every candidate.
template <typename F>
__device__ __forceinline__ void for_neighbors_serial(const NArgs &a, int p, F &&f) {
    const uint32_t c = a.sk[p];
    if (c >= (uint32_t)a.gx * (uint32_t)a.gy) return;
    const int cx = (int)(c % (uint32_t)a.gx), cy = (int)(c / (uint32_t)a.gx);
    uint32_t lo[3][2], hi[3][2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {  // every row's loads before the first is used
        const RowRanges r = row_ranges(a, cx, cy, k - 1);
        lo[k][0] = r.s1;
        lo[k][1] = r.s2;
        hi[k][0] = r.e1;
        hi[k][1] = r.e2;
    }
    auto scan = [&](uint32_t q, uint32_t end, auto &&d2_of) {
        const float *xp = a.xs + q, *yp = a.ys + q;
        for (; q + 4 <= end; q += 4, xp += 4, yp += 4) {
            const float x0 = xp[0], x1 = xp[1], x2 = xp[2], x3 = xp[3];
            const float y0 = yp[0], y1 = yp[1], y2 = yp[2], y3 = yp[3];
            const float e0 = d2_of(x0, y0), e1 = d2_of(x1, y1), e2 = d2_of(x2, y2),
                        e3 = d2_of(x3, y3);
            f(e0);
            f(e1);
            f(e2);
            f(e3);
        }
        for (; q < end; ++q, ++xp, ++yp) f(d2_of(*xp, *yp));
    };
    visit_rows(
        a, p, cx, cy, lo, hi,
        [&](auto &&d2_of) {
#pragma unroll
            for (int k = 0; k < 3; ++k) scan(lo[k][0], hi[k][0], d2_of);
        },
        scan);
}

// 256 threads: 256 / L particles; blocks in rows (pfs_grid.h).
template <int L>
__device__ __forceinline__ unsigned group_first() {
    return (blockIdx.y * gridDim.x + blockIdx.x) * (256 / L);
}
template <int L>
__device__ __forceinline__ int group_particle() {
    return (int)(group_first<L>() + threadIdx.x / L);
}

template <int L>
__global__ __launch_bounds__(256) void k_nbr_count(NArgs a, uint32_t *__restrict__ counts) {
    const int p = group_particle<L>();
    if (p >= a.n) return;
    uint32_t c = 0;
    for_neighbors<L>(a, p, [&](uint32_t q, bool ok, float d2) {
        c += (uint32_t)__popc(group_vote<L>(ok && d2 < a.r2 && (int)q != p));
    });
    const uint32_t i = a.id((uint32_t)p);
    if (group_lane<L>() == 0 && i < (uint32_t)a.n) counts[i] = c;
}

__global__ __launch_bounds__(256) void k_nbr_count_serial(NArgs a, uint32_t *__restrict__ counts) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.n) return;
    uint32_t c = 0;
    for_neighbors_serial(a, p, [&](float d2) { c += d2 < a.r2 ? 1u : 0u; });
    const uint32_t i = a.id((uint32_t)p);
    if (i < (uint32_t)a.n) counts[i] = c ? c - 1u : 0u;  // without p itself, as k_density
}

template <int L>
__global__ __launch_bounds__(256) void k_nbr_fill(NArgs a, const uint32_t *__restrict__ offsets,
                                                  uint32_t *__restrict__ nbr, size_t capacity) {
    const int p = group_particle<L>();
    if (p >= a.n) return;
    const uint32_t i = a.id((uint32_t)p);
    if (i >= (uint32_t)a.n) return;
    const uint32_t below = (1u << group_lane<L>()) - 1u;
    size_t o = offsets[i];
    for_neighbors<L>(a, p, [&](uint32_t q, bool ok, float d2) {
        const bool keep = ok && d2 < a.r2 && (int)q != p;
        const uint32_t vote = group_vote<L>(keep);
        const size_t to = o + __popc(vote & below);
        if (keep && to < capacity) nbr[to] = a.id(q);
        o += __popc(vote);
    });
}

// The same lists by sorted position (order null), written through LDS: the
// lists of a wave's 16 consecutive particles are one contiguous block of the
// output, so each wave gathers its entries in an LDS window of kFillWin
// slots and then writes the window out with consecutive lanes.  A block larger
// than the window takes further traversals, one per window.  Waves work
// independently: the LDS handoff is within one wave, whose LDS accesses
// complete in order.  1024 slots hold a wave's lists at 64 neighbours per
// particle in one traversal (16 KB per workgroup).
constexpr int kFillWin = 1024;
template <int L>
__global__ __launch_bounds__(256) void k_nbr_fill_lds(NArgs a, const uint32_t *__restrict__ offsets,
                                                      const uint32_t *__restrict__ counts,
                                                      uint32_t *__restrict__ nbr, size_t capacity) {
    __shared__ uint32_t win[4][kFillWin];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int PW = 64 / L;  // particles of a wave
    const int p = group_particle<L>();
    const int pw = (int)group_first<L>() + wave * PW;  // the wave's first particle
    if (pw >= a.n) return;                             // the whole wave is past the end
    const int plast = min(pw + PW - 1, a.n - 1);
    const uint32_t below = (1u << group_lane<L>()) - 1u;
    const size_t base = offsets[pw], end = (size_t)offsets[plast] + counts[plast];
    uint32_t *buf = win[wave];
    for (size_t w0 = base; w0 < end; w0 += kFillWin) {
        if (p < a.n) {
            size_t o = offsets[p];
            for_neighbors<L>(a, p, [&](uint32_t q, bool ok, float d2) {
                const bool keep = ok && d2 < a.r2 && (int)q != p;
                const uint32_t vote = group_vote<L>(keep);
                const size_t to = o + __popc(vote & below);
                if (keep && to >= w0 && to < w0 + kFillWin) buf[to - w0] = q;
                o += __popc(vote);
            });
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const size_t stop = end - w0 < (size_t)kFillWin ? end - w0 : (size_t)kFillWin;
        for (size_t j = lane; j < stop; j += 64)
            if (w0 + j < capacity) nbr[w0 + j] = buf[j];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// SPH density with the 2D poly6 kernel, W(d) = c (r^2 - d^2)^3; with counts,
// the neighbour counts of the same traversal.
// rho = mc * S with mc = mass * 4/(pi r^8) and S the FP32 sum, in traversal
// order and p included where it falls, of (r^2 - d2)^3 over the candidates
// with d2 < r^2.  A rejected candidate adds +0 (t clamped at 0), which leaves
// S unchanged, so the loop does not branch.  All terms are positive: S is
// within (m - 1) u of the exact sum of its m rounded terms.
__device__ __forceinline__ void store_density(const NArgs &a, int p, float rho_p, uint32_t cnt,
                                              float *rho, uint32_t *counts) {
    const uint32_t i = a.id((uint32_t)p);
    if (i >= (uint32_t)a.n) return;
    rho[i] = rho_p;
    // A finite p met itself (d2 = 0) and counted it; a non-finite p counted
    // nothing (every d2 it forms is NaN or Inf), as k_nbr_count.
    if (counts) counts[i] = cnt ? cnt - 1u : 0u;
}

__global__ __launch_bounds__(256) void k_density(NArgs a, float mc, float *__restrict__ rho,
                                                 uint32_t *__restrict__ counts) {
    const int p = group_particle<4>();
    if (p >= a.n) return;
    float sum = 0.0f;
    uint32_t cnt = 0;
    for_neighbors<4>(a, p, [&](uint32_t, bool ok, float d2) {
        const float t = ok ? fmaxf(a.r2 - d2, 0.0f) : 0.0f;
        sum = quad_add(sum, t * t * t);
        cnt += ok && d2 < a.r2 ? 1u : 0u;
    });
    cnt = quad_total(cnt);
    if (quad_lane() == 0) store_density(a, p, mc * sum, cnt, rho, counts);
}

__global__ __launch_bounds__(256) void k_density_serial(NArgs a, float mc, float *__restrict__ rho,
                                                        uint32_t *__restrict__ counts) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.n) return;
    float sum = 0.0f;
    uint32_t cnt = 0;
    for_neighbors_serial(a, p, [&](float d2) {
        const float t = fmaxf(a.r2 - d2, 0.0f);
        sum += t * t * t;
        cnt += d2 < a.r2 ? 1u : 0u;
    });
    store_density(a, p, mc * sum, cnt, rho, counts);
}

// A position wrapped into [0, n): unchanged when already inside (the
// reference's fmod(fmod(x,n)+n,n) would re-round it), else by the exact
// fmod; a tiny negative x whose x + n rounds to n becomes 0.
__device__ __forceinline__ float wrap_pos(float x, float n) {
    if (x >= 0.0f && x < n) return x;
    x = fmodf(x, n);
    if (x < 0.0f) x += n;
    return x >= n ? 0.0f : x;
}

// Tracers: one forward step through the velocity field, sampled bilinearly
// at the position: corners i0 = (int)x, i1 = (i0 + 1) mod W, weights and
// blend as src/fluid.cpp:55-66.
__global__ void k_tracer_advect(float *__restrict__ x, float *__restrict__ y, int n,
                                const float *__restrict__ vp, int w, int h, int vc, float dt,
                                float fw, float fh, float inv_w, float inv_h, int pow2_w,
                                int pow2_h) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float px = x[i], py = y[i];
    const int i0 = min(max((int)px, 0), w - 1), j0 = min(max((int)py, 0), h - 1);
    const int i1 = i0 + 1 == w ? 0 : i0 + 1, j1 = j0 + 1 == h ? 0 : j0 + 1;
    const float sx = px - (float)i0, sy = py - (float)j0;
    const float *f00 = vp + ((size_t)j0 * w + i0) * vc, *f10 = vp + ((size_t)j0 * w + i1) * vc;
    const float *f01 = vp + ((size_t)j1 * w + i0) * vc, *f11 = vp + ((size_t)j1 * w + i1) * vc;
    const float u = bilerp(sx, sy, f00[0], f10[0], f01[0], f11[0]);
    const float v = bilerp(sx, sy, f00[1], f10[1], f01[1], f11[1]);
    x[i] = wrap_pos(px + div_n(dt * u, fw, inv_w, pow2_w), fw);
    y[i] = wrap_pos(py + div_n(dt * v, fh, inv_h, pow2_h), fh);
}

// ---- position-based fluids: the density constraint, Jacobi iterations ------
// Macklin & Mueller, "Position Based Fluids" (ACM TOG 32(4), 2013), in 2D,
// on the sorted positions, with the neighbour lists found at the start of
// the solve (as the paper does once per step), kernels evaluated at the
// current iterate:
//   C_i = rho_i / rho0 - 1,  rho_i = m * W_poly6 summed over i and its list
//   lambda_i = -C_i / (sum_k |grad_k C_i|^2 + eps)
//   dx_i = (1 / rho0) * sum_{j in list} (lambda_i + lambda_j) grad W_spiky(x_i - x_j)
// with W_poly6 = 4/(pi h^8) (h^2 - r^2)^3 and grad W_spiky(d) =
// -30/(pi h^5) (h - r)^2 d / r for 0 < r < h (zero outside).  All updates
// of an iteration read the same iterate (Jacobi); positions wrap.
struct PbfCtl {
    int done;  // 0, or 1 + the iterate the solve converged on
};

struct PbfArgs {
    const float *xs, *ys;  // the current iterate (sorted positions)
    const uint32_t *noff, *ncnt, *nbr;  // neighbour lists by sorted position
    const uint32_t *sk, *cstart, *cend;  // the start's sorted keys and cell tables
    int gx, gy;
    int n;
    float W, H, half_w, half_h;
    float h, h2, mc, gc, rho0, r0sq, eps;
    int fast_w;      // spiky_w's short root and division
    float *lambda;   // [n] by sorted position
    float *nx, *ny;  // the next iterate
    double *part;    // [max_iters + 1][nblocks]: per-block sums of C^2
    double *res;     // [max_iters + 1]: sum of C^2 of each iterate
    PbfCtl *ctl;
    int it, nblocks;
    double tol2n;    // convergence: sum C^2 <= tol^2 * n
};

// The positions a workgroup's 256 particles gather, staged in LDS (one lane
// per particle only; with four, the gathers of a quad lie together and memory
// is as fast: 262,144 particles of 7 / 37 neighbours, 4 iterations 158 / 350 us
// against 169 / 361 staged).  Their lists lie in the three row windows of their
// cells' 3x3 blocks: when the particles share one cell row away from the
// domain's edges, row cy + oy contributes the sorted positions
// [start(cy + oy, cx_first - 1), end(cy + oy, cx_last + 1)), a few hundred in
// all.  `on` is uniform over the workgroup; otherwise (several rows, an edge,
// more than kStage positions, or lists too short to repay the staging) the
// gathers go to memory.  1,048,576 particles, 4 iterations, staged against not:
// 7 neighbours 438 / 402 us, 20 731 / 729, 37 1126 / 1269.
constexpr uint32_t kStageFrom = 20 * 256;  // list entries of the workgroup
constexpr int kStage = 2048;
struct Staged {
    float x[kStage], y[kStage], l[kStage];
    uint32_t w0, w1, w2, len0, len01, len012;  // window starts; cumulative lengths
    int on;
};

// The passes take 256 particles a workgroup, QUAD lanes (1 or 4) each.
constexpr int kPbfParticles = 256;
template <int QUAD>
__device__ __forceinline__ int pbf_particle() {
    return (int)(blockIdx.x * kPbfParticles + threadIdx.x / QUAD);
}

template <bool WITH_LAMBDA>
__device__ __forceinline__ void stage_windows(const PbfArgs &b, Staged &st) {
    if (threadIdx.x < 64) {  // one wavefront; lane k finds row k's window (lanes past 2 repeat row 2)
        const int p0 = blockIdx.x * kPbfParticles;
        const int pl = min(p0 + kPbfParticles, b.n) - 1;
        const uint32_t c0 = b.sk[p0], c1 = b.sk[pl];
        const int cy = (int)(c0 / (uint32_t)b.gx), cx0 = (int)(c0 % (uint32_t)b.gx),
                  cx1 = (int)(c1 % (uint32_t)b.gx);
        const uint32_t entries = b.noff[pl] + b.ncnt[pl] - b.noff[p0];
        const bool on = entries >= kStageFrom && (int)(c1 / (uint32_t)b.gx) == cy && cy >= 1 && cy <= b.gy - 2 && cx0 >= 1 &&
                        cx1 <= b.gx - 2 && c0 < (uint32_t)b.gx * (uint32_t)b.gy &&
                        c1 < (uint32_t)b.gx * (uint32_t)b.gy;
        uint32_t w = 0, len = 0;
        if (on) {
            const uint32_t row = (uint32_t)((cy - 1 + min((int)threadIdx.x, 2)) * b.gx);
            w = b.cstart[row + cx0 - 1];
            const uint32_t we = b.cend[row + cx1 + 1];
            len = we > w ? we - w : 0u;
        }
        const uint32_t len0 = quad_bcast<0>(len), len1 = quad_bcast<1>(len), len2 = quad_bcast<2>(len);
        const uint32_t w1 = quad_bcast<1>(w), w2 = quad_bcast<2>(w);
        if (threadIdx.x == 0) {
            st.w0 = w;
            st.w1 = w1;
            st.w2 = w2;
            st.len0 = len0;
            st.len01 = len0 + len1;
            st.len012 = len0 + len1 + len2;
            st.on = on && len0 + len1 + len2 <= (uint32_t)kStage;
        }
    }
    __syncthreads();
    if (!st.on) return;
    // Window k's positions go to slots [len_0 + .. + len_(k-1), + len_k).
    for (uint32_t j = threadIdx.x; j < st.len012; j += blockDim.x) {
        uint32_t q;
        if (j < st.len0) q = st.w0 + j;
        else if (j < st.len01) q = st.w1 + (j - st.len0);
        else q = st.w2 + (j - st.len01);
        if (q < (uint32_t)b.n) {
            st.x[j] = b.xs[q];
            st.y[j] = b.ys[q];
            if (WITH_LAMBDA) st.l[j] = b.lambda[q];
        }
    }
    __syncthreads();
}

// The LDS slot of sorted position q, or kStage when q is in no window (the
// lists then did not come from these cells; such entries read memory).
__device__ __forceinline__ uint32_t staged_slot(const Staged &st, uint32_t q) {
    if (q >= st.w0 && q - st.w0 < st.len0) return q - st.w0;
    if (q >= st.w1 && q - st.w1 < st.len01 - st.len0) return q - st.w1 + st.len0;
    if (q >= st.w2 && q - st.w2 < st.len012 - st.len01) return q - st.w2 + st.len01;
    return (uint32_t)kStage;
}

// A particle's position and list, loaded at a pass's entry (particle n - 1's
// past the end), under the look at the control block and what follows it.
struct PbfOwn {
    float x, y;
    uint32_t o, c;
};
__device__ __forceinline__ PbfOwn load_own(const PbfArgs &b, int p) {
    p = min(p, b.n - 1);
    return {b.xs[p], b.ys[p], b.noff[p], b.ncnt[p]};
}

// Every listed neighbour of p, in list order: f(q, slot, ok, dx, dy, d2) with
// (dx, dy) = x_q - x_p, periodic (the lists were found at the start; the
// positions have moved since), slot q's LDS slot (kStage: not staged), ok false
// past the list's end (q is then p).  QUAD = 4: four at a time on the quad's
// lanes, the entries of two steps loaded together.  QUAD = 1: eight loaded
// together, and the list's last few in fours.
template <int QUAD, typename F>
__device__ __forceinline__ void for_listed(const PbfArgs &b, const Staged *st, int p,
                                           const PbfOwn &own, F &&f) {
    const float px = own.x, py = own.y;
    const uint32_t o = own.o, c = own.c;
    const bool on = QUAD == 1 && st->on;
    const uint32_t l = QUAD == 4 ? (uint32_t)quad_lane() : 0u;
    // n steps from entry k on; all of them listed unless masked.
    auto batch = [&](uint32_t k, auto n, auto masked) {
        constexpr int N = decltype(n)::value;
        uint32_t q[N], sl[N];
        float x[N], y[N];
        auto listed = [&](int j) { return !decltype(masked)::value || k + QUAD * j + l < c; };
#pragma unroll
        for (int j = 0; j < N; ++j) q[j] = listed(j) ? b.nbr[o + k + QUAD * j + l] : (uint32_t)p;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            sl[j] = (uint32_t)kStage;
            if constexpr (QUAD == 1) {
                if (on) sl[j] = staged_slot(*st, q[j]);
                const bool lds = sl[j] < (uint32_t)kStage;
                x[j] = lds ? st->x[lds ? sl[j] : 0] : b.xs[q[j]];
                y[j] = lds ? st->y[lds ? sl[j] : 0] : b.ys[q[j]];
            } else {
                x[j] = b.xs[q[j]];
                y[j] = b.ys[q[j]];
            }
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            // periodic_diff's selects run only in a wavefront that has a pair
            // across the wrap: they are 12 of an entry's 70 operations.
            float dx = x[j] - px, dy = y[j] - py;
            if (__any(fabsf(dx) > b.half_w || fabsf(dy) > b.half_h)) {
                dx = periodic_diff(x[j], px, b.W, b.half_w);
                dy = periodic_diff(y[j], py, b.H, b.half_h);
            }
            f(q[j], sl[j], listed(j), dx, dy, dx * dx + dy * dy);
        }
    };
    uint32_t k = 0;
    if constexpr (QUAD == 4) {
        for (; k + 4 < c; k += 8) batch(k, std::integral_constant<int, 2>{}, std::true_type{});
        if (k < c) batch(k, std::integral_constant<int, 1>{}, std::true_type{});
    } else {
        for (; k + 8 <= c; k += 8) batch(k, std::integral_constant<int, 8>{}, std::false_type{});
        for (; k < c; k += 4) batch(k, std::integral_constant<int, 4>{}, std::true_type{});
    }
}

// w with grad W_spiky(x_p - x_q) = -w * (dx, dy): ((gc * t) * t) / r,
// t = h - r, r = sqrt(d2), for 0 < d2 < h^2; else 0 (selected, so that the
// loops do not branch; adding +-0 leaves the sums unchanged).
// Root and division correctly rounded without their range handling: r and an
// approximation of 1/r from one reciprocal root by Goldschmidt's iteration and
// a last residual step (exact for every d2 in [2^-100, 2^100), all 1.7e9 tried once
// on the GPU; the tests hold samples and the significands excluded below),
// the division by Markstein's steps as in div_fast.  Their theorem needs 1/r
// correctly rounded, which it is but for 5 significands of d2 in two binades,
// all x tried for those: only r = 2 - 2^-23 (times a power of two) divides some
// x wrongly, d2's significand then being all ones, the last bit aside.  Such a
// d2 anywhere in the wavefront, one below 2^-100, or a radius that lets the
// quotients' remainders underflow (b.fast_w, host) takes the plain forms.
__device__ __forceinline__ float spiky_w(const PbfArgs &b, float d2) {
    const bool in = d2 > 0.0f && d2 < b.h2;
    const float d = in ? d2 : 1.0f;
    if (b.fast_w && !__any(d < 0x1p-100f || (__float_as_uint(d) | 0xff800001u) == 0xffffffffu)) {
        const float y0 = __builtin_amdgcn_rsqf(d);
        float g = d * y0, y = 0.5f * y0;
        const float e = fmaf(-y, g, 0.5f);
        g = fmaf(g, e, g);
        y = fmaf(y, e, y);
        const float r = fmaf(fmaf(-g, g, d), y, g);
        y = y + y;
        y = fmaf(fmaf(-r, y, 1.0f), y, y);
        const float t = b.h - r;
        const float w = div_fast((b.gc * t) * t, r, y);
        return in ? w : 0.0f;
    }
    const float r = sqrtf(d2);
    const float t = b.h - r;
    const float w = ((b.gc * t) * t) / r;
    return in ? w : 0.0f;
}

// A term of an order-bound sum: the quad's four in lane order, or this lane's.
template <int QUAD>
__device__ __forceinline__ float add_terms(float s, float t) {
    return QUAD == 4 ? quad_add(s, t) : s + t;
}

// Block-wide FP64 sum over NW wavefronts (thread 0 gets it): wave shuffles,
// then the waves in order.
template <int NW>
__device__ __forceinline__ double block_sum(double v) {
    __shared__ double part[NW];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    double w[NW], s = 0.0;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NW; ++k) w[k] = part[k];
#pragma unroll
        for (int k = 0; k < NW; ++k) s += w[k];
    }
    return s;
}

// The total of iterate b.it's block sums, for thread 0 of a block of 1024:
// strided sums in block order, then the waves in order.
__device__ __forceinline__ double fold_sums(const PbfArgs &b) {
    double v = 0.0;
    for (int k = threadIdx.x; k < b.nblocks; k += 1024) v += b.part[(size_t)b.it * b.nblocks + k];
    return block_sum<16>(v);
}
// Writes iterate b.it's total and, at convergence, the verdict.
__device__ __forceinline__ void record(const PbfArgs &b, double total) {
    b.res[b.it] = total;
    if (total <= b.tol2n) b.ctl->done = 1 + b.it;
}

// lambda of iterate b.it, and the block sums of C^2.  Short
// lists are bound by the chain of loads (list, entries, positions), long ones by
// VALU issue, about 45 operations an entry.  250,001 particles of 7 / 37
// neighbours, 4 iterations of both passes: 145 / 327 us with the plain root and
// division and every entry's wrap selects, 139 / 304 without; 135 / 297 with a
// particle's own data loaded at entry and the sums folded in the update.
template <int QUAD>
__global__ __launch_bounds__(kPbfParticles *QUAD) void k_pbf_lambda(PbfArgs b) {
    const int p = pbf_particle<QUAD>();
    const PbfOwn own = load_own(b, p);
    if (b.ctl->done) return;  // the same verdict for every thread
    Staged *st = nullptr;
    if constexpr (QUAD == 1) {
        __shared__ Staged shared;
        st = &shared;
    }
    if constexpr (QUAD == 1) stage_windows<false>(b, *st);
    double c2 = 0.0;
    if (p < b.n) {
        float S = b.h2 * b.h2 * b.h2;  // p itself
        float gx = 0.0f, gy = 0.0f, g2 = 0.0f;
        for_listed<QUAD>(b, st, p, own, [&](uint32_t, uint32_t, bool ok, float dx, float dy, float d2) {
            const float t2 = ok ? fmaxf(b.h2 - d2, 0.0f) : 0.0f;
            S = add_terms<QUAD>(S, t2 * t2 * t2);
            const float w = spiky_w(b, d2);  // 0 past the list's end, where d2 = 0
            const float vx = w * dx, vy = w * dy;
            gx = add_terms<QUAD>(gx, vx);
            gy = add_terms<QUAD>(gy, vy);
            g2 = add_terms<QUAD>(g2, vx * vx + vy * vy);
        });
        const float rho = b.mc * S;
        const float C = rho / b.rho0 - 1.0f;
        const float denom = (gx * gx + gy * gy + g2) / b.r0sq + b.eps;
        if (QUAD == 1 || quad_lane() == 0) {
            b.lambda[p] = -C / denom;
            c2 = (double)C * (double)C;
        }
    }
    const double s = block_sum<kPbfParticles * QUAD / 64>(c2);
    if (threadIdx.x == 0) b.part[(size_t)b.it * b.nblocks + blockIdx.x] = s;
}

// Decides, between the passes, whether iterate b.it has converged, where the
// update's workgroups don't do it themselves.  (A fold by the last workgroup of
// k_pbf_lambda measured slower, with a release fence and without: every
// workgroup then stays for its sum's way to memory; 262,144 particles of 7
// neighbours, 4 iterations 158 us against 139.)
__global__ __launch_bounds__(1024) void k_pbf_check(PbfArgs b) {
    if (b.ctl->done) return;
    const double total = fold_sums(b);
    if (threadIdx.x == 0) record(b, total);
}

// The update of iterate b.it into the next iterate (nx, ny).
template <int QUAD>
__global__ __launch_bounds__(kPbfParticles *QUAD) void k_pbf_delta(PbfArgs b) {
    const int p = pbf_particle<QUAD>();
    const PbfOwn own = load_own(b, p);
    const float lp = b.lambda[min(p, b.n - 1)];
    const int done = b.ctl->done;
    Staged *st = nullptr;
    if constexpr (QUAD == 1) {
        if (done) return;  // as k_pbf_check left it
        __shared__ Staged shared;
        st = &shared;
        stage_windows<true>(b, *st);
    } else {
        // Every workgroup folds the block sums for itself, a load or two a
        // thread, and comes to the same verdict; the first one records it.  A
        // thread that already reads this iterate's record goes on like those that
        // read none, so that a workgroup meets the fold's barriers as a whole:
        // only an earlier iterate's ends it here.
        if (done != 0 && done <= b.it) return;
        __shared__ int over;
        const double total = fold_sums(b);
        if (threadIdx.x == 0) {
            over = total <= b.tol2n;
            if (blockIdx.x == 0) record(b, total);
        }
        __syncthreads();
        if (over) return;
    }
    if (p >= b.n) return;
    float ax = 0.0f, ay = 0.0f;
    for_listed<QUAD>(b, st, p, own, [&](uint32_t q, uint32_t slot, bool, float dx, float dy, float d2) {
        const float w = spiky_w(b, d2);
        float lq;
        if constexpr (QUAD == 1) {
            const bool lds = slot < (uint32_t)kStage;
            lq = lds ? st->l[lds ? slot : 0] : b.lambda[q];
        } else {
            lq = b.lambda[q];
        }
        const float s = lp + lq;
        ax = add_terms<QUAD>(ax, s * (w * dx));
        ay = add_terms<QUAD>(ay, s * (w * dy));
    });
    if (QUAD == 4 && quad_lane() != 0) return;
    b.nx[p] = wrap_pos(own.x + -(ax / b.rho0), b.W);
    b.ny[p] = wrap_pos(own.y + -(ay / b.rho0), b.H);
}

// Ends the solve on the caller's buffers: the final iterate f lives in the
// scratch pair when f is odd.
__global__ void k_pbf_finish(const PbfCtl *ctl, int iters, const float *sx, const float *sy,
                             float *xs, float *ys, int *iters_used, int n) {
    const int f = ctl->done ? ctl->done - 1 : iters;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p == 0 && iters_used) *iters_used = f;
    if (p < n && (f & 1)) {
        xs[p] = sx[p];
        ys[p] = sy[p];
    }
}

__global__ void k_pbf_init(PbfCtl *ctl, double *res, int nres) {
    if (threadIdx.x == 0) ctl->done = 0;
    for (int k = threadIdx.x; k < nres; k += blockDim.x) res[k] = -1.0;  // not computed
}

int grid_for(int n) { return blocks_for(n, 256); }
// Particles from which the density and the counts take one lane each instead
// of four: 4 wavefronts for every SIMD then.  Density with counts, one lane
// against four, us: 65,536 particles of 20 neighbours 14.2 / 9.9, 131,072
// 14.9 / 12.0, 262,144 17.8 / 17.9, 1,048,576 41.3 / 60.8.
constexpr int kSerialFrom = 1 << 18;
// The same line for the constraint solve's passes, by the count alone: sets of
// long lists above it would still gain from four lanes.  4 iterations, one lane
// against four, us: 65,536 particles of 7 / 37 neighbours 108 / 248 against
// 68 / 119, 262,144 145 / 372 against 137 / 312, 393,216 171 / 498 against 183 /
// 420, 1,048,576 360 / 1054 against 452 / 1027.
constexpr int kPbfSerialFrom = 3 << 17;
dim3 group_grid(int n, int L) {  // 256 threads, L a particle
    const Blocks b = block_rows(blocks_for(n, 256 / L));
    return dim3(b.x, b.y);
}
// Lanes a particle of the counts and lists (which no order binds): 16 where four
// leave the GPU short of wavefronts and a row's candidates are several loads one
// after another.  Grid's counts, scan, fill, four lanes against 16, us: 16,384
// particles of 7 / 20 / 37 neighbours 41 / 50 / 62 against 39 / 39 / 42, 65,536
// 44 / 55 / 67 against 45 / 49 / 55, 131,072 47 / 62 / 81 against 57 / 65 / 77.
int list_lanes(int n) { return n <= 1 << 16 ? 16 : 4; }

// The digit plan for keys below ncells: the fewest passes, 8-bit digits
// where they suffice for that many passes, else 10-bit.
struct RadixPlan {
    int passes, bits;
};
RadixPlan radix_plan(uint32_t ncells) {
    int kb = 0;
    while (kb < 32 && (ncells - 1) >> kb) ++kb;
    if (kb <= 8) return {1, 8};
    if (kb <= 16) return {2, 8};
    if (kb <= 20) return {2, 10};
    if (kb <= 24) return {3, 8};
    return {3, 10};
}

// Workspace layout (words): sorted keys (2 buffers), values spare buffer,
// digit histogram (2^11 words for each 4096 keys: four 8-bit rows of 1024-key
// tiles, or two 10-bit rows of 2048-key ones), digit row totals (2^10), scan
// block sums.
struct SortWs {
    uint32_t *k0, *k1, *v1, *hist, *tot, *sums;
};
size_t hist_words(int n) {
    const size_t nb = (size_t)nblocks_for((size_t)n);
    return ((size_t)2 << kMaxRadixBits) * (nb ? nb : 1);
}
size_t sort_ws_words(int n, size_t ncells) {
    const size_t hist = hist_words(n);
    size_t sums = std::max<size_t>(nblocks_for(hist / 2), nblocks_for((size_t)n));
    sums = std::max<size_t>(sums, nblocks_for(ncells));
    return 3 * (size_t)n + hist + ((size_t)1 << kMaxRadixBits) + sums + 64;
}
SortWs sort_ws(void *ws, int n) {  // ws: 4-byte aligned
    uint32_t *p = static_cast<uint32_t *>(ws);
    SortWs s;
    s.k0 = p;
    s.k1 = p + n;
    s.v1 = p + 2 * (size_t)n;
    s.hist = p + 3 * (size_t)n;
    s.tot = s.hist + hist_words(n);
    s.sums = s.tot + ((size_t)1 << kMaxRadixBits);
    return s;
}

bool valid_grid(const pfs_ngrid *g) {
    return g && g->n >= 1 && g->gx >= 3 && g->gy >= 3 && g->domain_w > 0 && g->domain_h > 0 &&
           g->radius > 0 && (int64_t)g->gx * g->gy <= ((int64_t)1 << 30) &&
           g->radius <= g->domain_w / g->gx && g->radius <= g->domain_h / g->gy;
}

// Up to kSmallSort particles the sort's tiles are 1024 keys (8-bit digits)
// or 2048 (10-bit): 4096-key tiles leave most CUs idle there, and a tile is one
// long chain.  Both kinds' counts fit the same workspace.  Building the grid
// of 10,000 / 60,000 / 1,000,000 cells, large -> small tiles: 16,384 particles
// 29.7 / 31.9 / 41.5 -> 25.5 / 26.2 / 41.3 us; 131,072: 37.7 / 39.3 / 55.2 ->
// 28.9 / 29.8 / 46.9; 524,288: 46.9 / 47.6 / 65.5 -> 39.8 / 41.2 / 59.4;
// 786,432: 50.9 / 50.9 / 70.2 -> 50.5 / 52.6 / 77.2, where the large ones stay.
constexpr int kSmallSort = 1 << 19;

struct SortArgs {
    int n;
    const float *x, *y;
    uint32_t *keys;
    float *xs, *ys;
    uint32_t *const *kb, *const *vb;
    SortWs w;
    CellKeyArgs ck;
    hipStream_t s;
};

template <int RB, int NT>
void sort_passes(const SortArgs &a, int passes) {
    const int nb = blocks_for(a.n, sort_tile<NT>());
    const bool few = NT < kThreads && nb <= kFewTiles;  // past kSmallSort never
    const uint32_t *kin = a.keys;
    for (int p = 0; p < passes; ++p) {
        const int shift = RB * p;
        const bool last = p + 1 == passes;
        const uint32_t *vin = p == 0 ? nullptr : a.vb[p & 1];
        float *oxs = last ? a.xs : nullptr, *oys = last ? a.ys : nullptr;
        if (p == 0)
            hipLaunchKernelGGL((k_radix_hist<RB, NT, true>), dim3(nb), dim3(NT), 0, a.s, nullptr, a.ck,
                               a.keys, a.n, shift, a.w.hist, nb);
        else
            hipLaunchKernelGGL((k_radix_hist<RB, NT, false>), dim3(nb), dim3(NT), 0, a.s, kin, a.ck,
                               nullptr, a.n, shift, a.w.hist, nb);
        if constexpr (NT < kThreads)
            if (few)
                hipLaunchKernelGGL((k_radix_scatter<RB, NT, true>), dim3(nb), dim3(NT), 0, a.s, kin, vin,
                                   a.kb[(p + 1) & 1], a.vb[(p + 1) & 1], a.n, shift, a.w.hist, a.w.tot,
                                   nb, a.x, a.y, oxs, oys);
        if (!few) {
            if (nb <= sort_tile<256>())
                hipLaunchKernelGGL(k_digit_rows<256>, dim3(1 << RB), dim3(256), 0, a.s, a.w.hist,
                                   a.w.tot, nb);
            else
                hipLaunchKernelGGL(k_digit_rows<kThreads>, dim3(1 << RB), dim3(kThreads), 0, a.s,
                                   a.w.hist, a.w.tot, nb);
            hipLaunchKernelGGL((k_radix_scatter<RB, NT, false>), dim3(nb), dim3(NT), 0, a.s, kin, vin,
                               a.kb[(p + 1) & 1], a.vb[(p + 1) & 1], a.n, shift, a.w.hist, a.w.tot, nb,
                               a.x, a.y, oxs, oys);
        }
        kin = a.kb[(p + 1) & 1];
    }
}

NArgs nargs(const pfs_ngrid *g, const float *xs, const float *ys,
            const uint32_t *order, const uint32_t *sk, const uint32_t *start, const uint32_t *end) {
    NArgs a{};
    a.xs = xs;
    a.ys = ys;
    a.order = order;
    a.sk = sk;
    a.start = start;
    a.end = end;
    a.n = g->n;
    a.gx = g->gx;
    a.gy = g->gy;
    a.W = g->domain_w;
    a.H = g->domain_h;
    a.half_w = g->domain_w * 0.5f;
    a.half_h = g->domain_h * 0.5f;
    a.r2 = g->radius * g->radius;
    return a;
}

// PBF workspace: the control block, the block sums of C^2 of every iterate,
// and the scratch position pair.
struct PbfWs {
    PbfCtl *ctl;
    double *part;
    float *sx, *sy;
};
size_t pbf_part_bytes(int n, int max_iters) {
    return ((size_t)(max_iters + 1) * grid_for(n) * sizeof(double) + 255) & ~(size_t)255;
}
size_t pbf_ws_bytes(int n, int max_iters) {
    return 256 + pbf_part_bytes(n, max_iters) + 2 * (((size_t)n * sizeof(float) + 255) & ~(size_t)255);
}
PbfWs pbf_ws(void *ws, int n, int max_iters) {
    char *p = static_cast<char *>(ws);
    PbfWs w;
    w.ctl = reinterpret_cast<PbfCtl *>(p);
    w.part = reinterpret_cast<double *>(p + 256);
    w.sx = reinterpret_cast<float *>(p + 256 + pbf_part_bytes(n, max_iters));
    w.sy = w.sx + ((((size_t)n * sizeof(float) + 255) & ~(size_t)255) / sizeof(float));
    return w;
}

thread_local size_t t_list_total = 0;  // of this thread's last call of the next

// Offsets and *total from counts, then the lists (checked against the
// capacity first, which waits for *total).
int lists_from_counts(const pfs_ngrid *g, const NArgs &a, const uint32_t *counts,
                      uint32_t *offsets, uint32_t *nbr, size_t nbr_capacity, uint32_t *total,
                      const SortWs &w, hipStream_t s) {
    PFS_TRY(scan_exclusive(counts, offsets, g->n, total, w.sums, s));
    uint32_t h_total = 0;
    PFS_HIP_TRY(hipMemcpyAsync(&h_total, total, sizeof h_total, hipMemcpyDeviceToHost, s));
    PFS_HIP_TRY(hipStreamSynchronize(s));
    t_list_total = h_total;
    if (h_total > nbr_capacity)
        return set_error(PFS_ERR_INVALID, "ngrid: neighbour list capacity " +
                                              std::to_string(nbr_capacity) + " < " +
                                              std::to_string(h_total));
    const int L = list_lanes(g->n);
    const dim3 grid = group_grid(g->n, L);
    if (a.order)
        hipLaunchKernelGGL(L == 16 ? k_nbr_fill<16> : k_nbr_fill<4>, grid, dim3(256), 0, s, a,
                           offsets, nbr, nbr_capacity);
    else
        hipLaunchKernelGGL(L == 16 ? k_nbr_fill_lds<16> : k_nbr_fill_lds<4>, grid, dim3(256), 0, s, a,
                           offsets, counts, nbr, nbr_capacity);
    return check_launch("neighbour lists");
}

}  // namespace
}  // namespace pfs

using namespace pfs;

extern "C" {

int pfs_ngrid_init(pfs_ngrid *g, int n, float domain_w, float domain_h, float radius) {
    if (!g || n < 1 || !(domain_w > 0) || !(domain_h > 0) || !(radius > 0))
        return set_error(PFS_ERR_INVALID, "ngrid: need n >= 1 and positive sizes");
    g->n = n;
    g->domain_w = domain_w;
    g->domain_h = domain_h;
    g->radius = radius;
    const double gx = std::floor((double)domain_w / radius), gy = std::floor((double)domain_h / radius);
    if (gx < 3 || gy < 3 || gx * gy > (double)(1 << 30))
        return set_error(PFS_ERR_INVALID, "ngrid: the domain must span 3 to 2^30 cells of the radius");
    g->gx = (int)gx;
    g->gy = (int)gy;
    // Cells at least `radius` wide, so neighbours within it are in the 3x3 block.
    while (g->radius > g->domain_w / g->gx) --g->gx;
    while (g->radius > g->domain_h / g->gy) --g->gy;
    if (g->gx < 3 || g->gy < 3) return set_error(PFS_ERR_INVALID, "ngrid: fewer than 3 cells");
    g->kx = (float)g->gx / domain_w;
    g->ky = (float)g->gy / domain_h;
    return PFS_OK;
}

size_t pfs_ngrid_workspace_bytes(const pfs_ngrid *g) {
    if (!g || g->n < 1) return 0;
    return sort_ws_words(g->n, (size_t)g->gx * g->gy) * sizeof(uint32_t);
}

int pfs_scan_exclusive_u32(const uint32_t *in, uint32_t *out, int n, uint32_t *total, void *ws,
                           size_t ws_bytes, void *stream) {
    if (n < 0 || (n > 0 && (!in || !out))) return set_error(PFS_ERR_INVALID, "scan: bad arguments");
    if (!ws || ws_bytes < (size_t)(nblocks_for((size_t)n) + 1) * sizeof(uint32_t))
        return set_error(PFS_ERR_INVALID, "scan: workspace too small");
    return scan_exclusive(in, out, n, total, static_cast<uint32_t *>(ws), (hipStream_t)stream);
}

int pfs_gather_u32(const uint32_t *index, const uint32_t *in, uint32_t *out, int n, void *stream) {
    if (n < 0 || (n > 0 && (!index || !in || !out)) || in == out)
        return set_error(PFS_ERR_INVALID, "gather: bad arguments");
    if (n == 0) return PFS_OK;
    hipLaunchKernelGGL(k_gather_u32, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, index, in,
                       out, n);
    return check_launch("gather");
}

int pfs_particles_advect(float *x, float *y, int n, const pfs_field *vp, float dt, void *stream) {
    PFS_TRY(check_field(vp, "vp", 2));
    if (n < 0 || (n > 0 && (!x || !y))) return set_error(PFS_ERR_INVALID, "advect: bad particles");
    if (n == 0) return PFS_OK;
    hipLaunchKernelGGL(k_tracer_advect, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, x, y,
                       n, vp->data, vp->x, vp->y, vp->z, dt, (float)vp->x, (float)vp->y,
                       1.0f / (float)vp->x, 1.0f / (float)vp->y, (vp->x & (vp->x - 1)) == 0,
                       (vp->y & (vp->y - 1)) == 0);
    return check_launch("particle advect");
}

int pfs_ngrid_build(const pfs_ngrid *g, const float *x, const float *y, uint32_t *keys,
                    uint32_t *order, uint32_t *cell_start, uint32_t *cell_end, float *xs, float *ys,
                    void *ws, size_t ws_bytes, void *stream) {
    if (!valid_grid(g)) return set_error(PFS_ERR_INVALID, "ngrid: not initialised by pfs_ngrid_init");
    if (!x || !y || !keys || !order || !cell_start || !cell_end || !xs || !ys)
        return set_error(PFS_ERR_INVALID, "ngrid: NULL buffer");
    if (!ws || ws_bytes < pfs_ngrid_workspace_bytes(g) || ((uintptr_t)ws & 3))
        return set_error(PFS_ERR_INVALID,
                         "ngrid: workspace not 4-byte aligned or smaller than pfs_ngrid_workspace_bytes()");
    hipStream_t s = (hipStream_t)stream;
    const int n = g->n;
    const uint32_t ncells = (uint32_t)g->gx * (uint32_t)g->gy;
    SortWs w = sort_ws(ws, n);

    // Buffers alternate so that the last pass writes the keys to k0 (kept for
    // the neighbour passes) and the particle ids to `order`.  The first pass
    // makes the keys (into `keys`) and takes the particle ids as its values;
    // the last gathers the positions into sorted order.
    const RadixPlan plan = radix_plan(ncells);
    const int passes = plan.passes;
    uint32_t *kb[2] = {passes % 2 == 0 ? w.k0 : w.k1, passes % 2 == 0 ? w.k1 : w.k0};
    uint32_t *vb[2] = {passes % 2 == 0 ? order : w.v1, passes % 2 == 0 ? w.v1 : order};
    const CellKeyArgs ck{x, y, g->kx, g->ky, g->gx, g->gy};
    const SortArgs sa{n, x, y, keys, xs, ys, kb, vb, w, ck, s};
    if (plan.bits == 8)
        n <= kSmallSort ? sort_passes<8, 256>(sa, passes) : sort_passes<8, 1024>(sa, passes);
    else
        n <= kSmallSort ? sort_passes<10, 512>(sa, passes) : sort_passes<10, 1024>(sa, passes);
    // Cell tables: the lower bound of every cell (empty ones included) in the
    // sorted keys, left in k0 by the last pass.
    const unsigned cblocks = (unsigned)(((size_t)ncells + 255) / 256);
    hipLaunchKernelGGL(k_cell_tables, dim3(cblocks), dim3(256), 0, s, w.k0, n, cell_start, cell_end,
                       ncells);
    return check_launch("neighbour grid");
}

int pfs_ngrid_neighbors(const pfs_ngrid *g, const float *xs, const float *ys, const uint32_t *order,
                        const uint32_t *cell_start, const uint32_t *cell_end, uint32_t *counts,
                        uint32_t *offsets, uint32_t *nbr, size_t nbr_capacity, uint32_t *total,
                        void *ws, size_t ws_bytes, void *stream) {
    if (!valid_grid(g)) return set_error(PFS_ERR_INVALID, "ngrid: not initialised by pfs_ngrid_init");
    if (!xs || !ys || !cell_start || !cell_end || !counts || !offsets || !total)
        return set_error(PFS_ERR_INVALID, "ngrid: NULL buffer");
    if (!ws || ws_bytes < pfs_ngrid_workspace_bytes(g) || ((uintptr_t)ws & 3))
        return set_error(PFS_ERR_INVALID,
                         "ngrid: workspace not 4-byte aligned or smaller than pfs_ngrid_workspace_bytes()");
    hipStream_t s = (hipStream_t)stream;
    SortWs w = sort_ws(ws, g->n);
    const NArgs a = nargs(g, xs, ys, order, w.k0, cell_start, cell_end);
    if (g->n < kSerialFrom)
        hipLaunchKernelGGL(list_lanes(g->n) == 16 ? k_nbr_count<16> : k_nbr_count<4>,
                           group_grid(g->n, list_lanes(g->n)), dim3(256), 0, s, a, counts);
    else
        hipLaunchKernelGGL(k_nbr_count_serial, dim3(grid_for(g->n)), dim3(256), 0, s, a, counts);
    if (!nbr) return scan_exclusive(counts, offsets, g->n, total, w.sums, s);  // no lists
    return lists_from_counts(g, a, counts, offsets, nbr, nbr_capacity, total, w, s);
}

size_t pfs_ngrid_list_total(void) { return t_list_total; }

int pfs_ngrid_lists(const pfs_ngrid *g, const float *xs, const float *ys, const uint32_t *order,
                    const uint32_t *cell_start, const uint32_t *cell_end, const uint32_t *counts,
                    uint32_t *offsets, uint32_t *nbr, size_t nbr_capacity, uint32_t *total,
                    void *ws, size_t ws_bytes, void *stream) {
    if (!valid_grid(g)) return set_error(PFS_ERR_INVALID, "ngrid: not initialised by pfs_ngrid_init");
    if (!xs || !ys || !cell_start || !cell_end || !counts || !offsets || !nbr || !total)
        return set_error(PFS_ERR_INVALID, "ngrid: NULL buffer");
    if (!ws || ws_bytes < pfs_ngrid_workspace_bytes(g) || ((uintptr_t)ws & 3))
        return set_error(PFS_ERR_INVALID,
                         "ngrid: workspace not 4-byte aligned or smaller than pfs_ngrid_workspace_bytes()");
    SortWs w = sort_ws(ws, g->n);
    const NArgs a = nargs(g, xs, ys, order, w.k0, cell_start, cell_end);
    return lists_from_counts(g, a, counts, offsets, nbr, nbr_capacity, total, w,
                             (hipStream_t)stream);
}


size_t pfs_pbf_workspace_bytes(const pfs_ngrid *g, int max_iters) {
    if (!g || g->n < 1 || max_iters < 0 || max_iters > PFS_PBF_MAX_ITERS) return 0;
    return pbf_ws_bytes(g->n, max_iters);
}

int pfs_pbf_solve(const pfs_ngrid *g, float *xs, float *ys, const uint32_t *cell_start,
                  const uint32_t *cell_end, const uint32_t *nbr_offsets, const uint32_t *nbr_counts,
                  const uint32_t *nbr, float mass, float rho0, float eps, int max_iters, double tol,
                  float *lambda, double *residuals, int *iters_used, void *ngrid_ws,
                  size_t ngrid_ws_bytes, void *ws, size_t ws_bytes, void *stream) {
    if (!valid_grid(g)) return set_error(PFS_ERR_INVALID, "ngrid: not initialised by pfs_ngrid_init");
    if (!xs || !ys || !cell_start || !cell_end || !nbr_offsets || !nbr_counts || !nbr || !lambda ||
        !residuals)
        return set_error(PFS_ERR_INVALID, "pbf: NULL buffer");
    if (!ngrid_ws || ngrid_ws_bytes < pfs_ngrid_workspace_bytes(g) || ((uintptr_t)ngrid_ws & 3))
        return set_error(PFS_ERR_INVALID, "pbf: neighbour-grid workspace too small or misaligned");
    if (!(rho0 > 0.0f) || !(eps > 0.0f) || !(mass > 0.0f) || !(tol >= 0.0) || max_iters < 0 ||
        max_iters > PFS_PBF_MAX_ITERS)
        return set_error(PFS_ERR_INVALID, "pbf: need mass, rho0, eps > 0, tol >= 0, 0 <= max_iters <= " +
                                              std::to_string(PFS_PBF_MAX_ITERS));
    if (!ws || ws_bytes < pbf_ws_bytes(g->n, max_iters) || ((uintptr_t)ws & 255))
        return set_error(PFS_ERR_INVALID,
                         "pbf: workspace not 256-byte aligned or smaller than pfs_pbf_workspace_bytes()");
    hipStream_t s = (hipStream_t)stream;
    const int n = g->n, nb = grid_for(n);
    const PbfWs w = pbf_ws(ws, n, max_iters);
    const double h = g->radius;
    PbfArgs b{};
    b.noff = nbr_offsets;
    b.ncnt = nbr_counts;
    b.nbr = nbr;
    b.sk = sort_ws(ngrid_ws, n).k0;
    b.cstart = cell_start;
    b.cend = cell_end;
    b.gx = g->gx;
    b.gy = g->gy;
    b.n = n;
    b.W = g->domain_w;
    b.H = g->domain_h;
    b.half_w = g->domain_w * 0.5f;
    b.half_h = g->domain_h * 0.5f;
    b.h = g->radius;
    b.h2 = g->radius * g->radius;
    const float coef = (float)(4.0 / (3.14159265358979323846 * h * h * h * h * h * h * h * h));
    b.mc = mass * coef;
    b.gc = (float)(-30.0 / (3.14159265358979323846 * h * h * h * h * h));
    // Remainders of (gc * t) * t over r, t from an ulp of h to h, stay normal.
    const float w_max = std::fabs(b.gc) * b.h2;
    b.fast_w = b.h2 >= 0x1p-60f && b.h2 <= 0x1p60f && w_max >= 0x1p-30f && w_max <= 0x1p60f;
    b.rho0 = rho0;
    b.r0sq = rho0 * rho0;
    b.eps = eps;
    b.lambda = lambda;
    b.part = w.part;
    b.res = residuals;
    b.ctl = w.ctl;
    b.nblocks = nb;
    b.tol2n = tol * tol * (double)n;
    float *bx[2] = {xs, w.sx}, *by[2] = {ys, w.sy};
    const bool quad = n < kPbfSerialFrom;
    hipLaunchKernelGGL(k_pbf_init, dim3(1), dim3(256), 0, s, w.ctl, residuals, max_iters + 1);
    for (int it = 0; it <= max_iters; ++it) {
        b.it = it;
        b.xs = bx[it & 1];
        b.ys = by[it & 1];
        b.nx = bx[(it + 1) & 1];
        b.ny = by[(it + 1) & 1];
        hipLaunchKernelGGL(quad ? k_pbf_lambda<4> : k_pbf_lambda<1>, dim3(nb),
                           dim3(kPbfParticles * (quad ? 4 : 1)), 0, s, b);
        if (!quad || it == max_iters) hipLaunchKernelGGL(k_pbf_check, dim3(1), dim3(1024), 0, s, b);
        if (it < max_iters)
            hipLaunchKernelGGL(quad ? k_pbf_delta<4> : k_pbf_delta<1>, dim3(nb),
                               dim3(kPbfParticles * (quad ? 4 : 1)), 0, s, b);
    }
    hipLaunchKernelGGL(k_pbf_finish, dim3(nb), dim3(256), 0, s, w.ctl, max_iters, w.sx, w.sy, xs, ys,
                       iters_used, n);
    return check_launch("pbf solve");
}

int pfs_ngrid_density(const pfs_ngrid *g, const float *xs, const float *ys, const uint32_t *order,
                      const uint32_t *cell_start, const uint32_t *cell_end, float mass, float *rho,
                      uint32_t *counts, void *ws, size_t ws_bytes, void *stream) {
    if (!valid_grid(g)) return set_error(PFS_ERR_INVALID, "ngrid: not initialised by pfs_ngrid_init");
    if (!xs || !ys || !cell_start || !cell_end || !rho)
        return set_error(PFS_ERR_INVALID, "ngrid: NULL buffer");
    if (!ws || ws_bytes < pfs_ngrid_workspace_bytes(g) || ((uintptr_t)ws & 3))
        return set_error(PFS_ERR_INVALID,
                         "ngrid: workspace not 4-byte aligned or smaller than pfs_ngrid_workspace_bytes()");
    SortWs w = sort_ws(ws, g->n);
    hipStream_t s = (hipStream_t)stream;
    const NArgs a = nargs(g, xs, ys, order, w.k0, cell_start, cell_end);
    // 2D poly6: 4 / (pi r^8), in float from the double constant, times the mass.
    const double r = g->radius;
    const float coef = (float)(4.0 / (3.14159265358979323846 * r * r * r * r * r * r * r * r));
    const float mc = mass * coef;
    if (g->n < kSerialFrom)
        hipLaunchKernelGGL(k_density, group_grid(g->n, 4), dim3(256), 0, s, a, mc, rho, counts);
    else
        hipLaunchKernelGGL(k_density_serial, dim3(grid_for(g->n)), dim3(256), 0, s, a, mc, rho, counts);
    return check_launch("density");
}

}  // extern "C"
