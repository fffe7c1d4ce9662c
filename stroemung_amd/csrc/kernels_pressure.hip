// gfx950 kernels for the pressure Poisson solve (POISSON of NaSt2D):
//  * the reference-compatible lexicographic SOR of tall channels, run as a
//    diagonal wavefront inside one workgroup per channel -- bit-exact with the
//    reference's x-outer / y-inner in-place sweep, including its unmasked
//    sequential residual fold and stopping rule (src/simulation.rs:216-285);
//  * the set-up of the red-black solve (its sweeps live in kernels_rbtb.hip)
//    and the ghost refresh used by the stage entry points.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "stm_internal.h"

namespace stm {

__device__ __forceinline__ double ghost_value(const double* __restrict__ p, int64_t i,
                                              int64_t P, uint8_t edge) {
    // src/grid/mod.rs:343-412; (a + b) / 2.0 equals (a + b) * 0.5 exactly.
    switch (edge) {
    case E_N: return p[i - 1];
    case E_NE: return (p[i - 1] + p[i + P]) * 0.5;
    case E_E: return p[i + P];
    case E_SE: return (p[i + 1] + p[i + P]) * 0.5;
    case E_S: return p[i + 1];
    case E_SW: return (p[i + 1] + p[i - P]) * 0.5;
    case E_W: return p[i - P];
    case E_NW: return (p[i - 1] + p[i - P]) * 0.5;
    default: return p[i];
    }
}

// Ghost pressure of boundary cells (all colours, or one).  Reads fluid cells
// only and writes boundary cells only, so it is order-free.
__global__ void __launch_bounds__(256)
k_ghost(int nbtot, const BEntry* __restrict__ be, const ChanState* __restrict__ cs,
        double* __restrict__ p, int colour, int only_active)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nbtot) return;
    const BEntry e = be[k];
    if (e.edge == E_NONE) return;
    if (colour >= 0 && e.colour != colour) return;
    if (only_active && !cs[e.chan].active) return;
    p[e.gidx] = ghost_value(p, e.gidx, e.pitch, e.edge);
}

// Sum slot `slot` of the partials of one channel's tiles in a fixed order.
__device__ double chan_sum(const ChanDesc& d, const double* __restrict__ part, int slot,
                           double* sh) {
    const int tid = threadIdx.x;
    double acc = 0.0;
    for (int k = d.tile0 + tid; k < d.tile0 + d.ntiles; k += blockDim.x)
        acc = acc + part[(int64_t)k * NPART + slot];
    sh[tid] = acc;
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if (tid < st) sh[tid] = sh[tid] + sh[tid + st];
        __syncthreads();
    }
    return sh[0];
}

// Per-tile sums over interior fluid cells: pass 0 sum of rhs (slot 0),
// pass 1 sum of (rhs - mean)^2 (slot 1).
__global__ void __launch_bounds__(TILE_THREADS)
k_rhs_sums(const ChanDesc* __restrict__ cd, const ChanState* __restrict__ cs,
           const Tile* __restrict__ tiles, const uint8_t* __restrict__ flags,
           const double* __restrict__ rhs, double* __restrict__ part, int pass)
{
    __shared__ double sh[TILE_THREADS];
    const Tile t = tiles[blockIdx.x];
    const ChanDesc& d = cd[t.chan];
    const int x = t.x0 + threadIdx.y, y = t.y0 + threadIdx.x;
    const int tid = threadIdx.y * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (x >= 1 && x <= d.nx - 2 && y >= 1 && y <= d.ny - 2) {
        const int64_t i = d.off + x * (int64_t)d.pitch + y;
        if (flag_fluid(flags[i])) {
            const double r = pass ? rhs[i] - cs[t.chan].rhs_mean : rhs[i];
            v = pass ? r * r : r;
        }
    }
    sh[tid] = v;
    __syncthreads();
    for (int st = TILE_THREADS / 2; st > 0; st >>= 1) {
        if (tid < st) sh[tid] = sh[tid] + sh[tid + st];
        __syncthreads();
    }
    if (tid == 0) part[blockIdx.x * NPART + pass] = sh[0];
}

// The mean of rhs over interior fluid cells.  The pressure problem has
// Neumann conditions all round (every boundary's ghost copies its fluid
// neighbour), so it is solvable only for rhs of zero mean; with inflow and
// outflow the mean is not zero and no iteration can push the residual below
// it.  The red-black solver solves for rhs - mean.
__global__ void __launch_bounds__(256)
k_rhs_mean(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
           const double* __restrict__ part)
{
    __shared__ double sh[256];
    const ChanDesc& d = cd[blockIdx.x];
    const double sum = chan_sum(d, part, 0, sh);
    if (threadIdx.x == 0) cs[blockIdx.x].rhs_mean = d.n_inner > 0.0 ? sum / d.n_inner : 0.0;
}

// Start of a solve: tol2 = eps^2 * sum((rhs - mean)^2) over interior fluid
// cells, and what runs.
__device__ __forceinline__ void begin_solve(const ChanDesc& d, ChanState& s, double rsum2,
                                            int32_t* active_out) {
    const bool rb = d.solver == SOLVER_RB;
    s.rhs2 = rsum2;
    s.tol2 = d.eps2 * rsum2;
    if (rb) {   // (a lexicographic solve looks at how its last one ended)
        s.sor_iters = 0;
        s.exhausted = 0;
    }
    s.active = (rb && d.itermax > 0) ? 1 : 0;
    s.stop_launch = s.active ? -1 : 0;
    s.pbuf = 0;
    s.budget = 0;
    *active_out = s.active;
}

__global__ void __launch_bounds__(256)
k_solve_begin(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
              const double* __restrict__ part, int32_t* __restrict__ active_out)
{
    __shared__ double sh[256];
    const ChanDesc& d = cd[blockIdx.x];
    const double rsum2 = chan_sum(d, part, 1, sh);
    if (threadIdx.x == 0) begin_solve(d, cs[blockIdx.x], rsum2, active_out + blockIdx.x);
}

// The sum of v over a wave as the tree of offsets 32, 16, .. 1 gives it (lane 0).
__device__ __forceinline__ double wave_tree(double v) {
    for (int off = 32; off > 0; off >>= 1) v = v + __shfl_down(v, off, 64);
    return v;
}

// k_rhs_sums, k_rhs_mean, k_rhs_sums and k_solve_begin of one channel in one
// workgroup, in the same order: a wave sums a tile, a lane taking its column's
// four cells as the first two steps of the tile's tree pair them, and the first
// wave folds the tiles likewise.  For small channels, whose four launches took
// 12 us of kernels and the gaps between them (a one-sweep solve of 102 x 22 cells:
// 102 us with them, 92 so).
__global__ void __launch_bounds__(1024)
k_solve_stats(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
              const Tile* __restrict__ tiles, const uint8_t* __restrict__ flags,
              const double* __restrict__ rhs, int32_t* __restrict__ active_out)
{
    static_assert(TILE_X == 4 && TILE_Y == 64, "a lane's four cells");
    static_assert(STATS_TILES <= 64, "a tile a lane in the fold");
    __shared__ double part[STATS_TILES], total;
    const ChanDesc& d = cd[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double mean = 0.0;
    for (int pass = 0; pass < 2; pass++) {
        for (int k = wave; k < d.ntiles; k += 16) {
            const Tile t = tiles[d.tile0 + k];
            const int y = t.y0 + lane;
            double v[TILE_X];
#pragma unroll
            for (int r = 0; r < TILE_X; r++) {
                const int x = t.x0 + r;
                const bool in = x >= 1 && x <= d.nx - 2 && y >= 1 && y <= d.ny - 2;
                const int64_t i = d.off + (in ? x * (int64_t)d.pitch + y : 0);
                const double a = rhs[i] - mean;   // (pass 0: the value itself)
                v[r] = in && flag_fluid(flags[i]) ? (pass ? a * a : rhs[i]) : 0.0;
            }
            const double s = wave_tree((v[0] + v[2]) + (v[1] + v[3]));
            if (lane == 0) part[k] = s;
        }
        __syncthreads();
        if (wave == 0) {
            auto at = [&](int k) { return k < d.ntiles ? 0.0 + part[k] : 0.0; };
            const double s = wave_tree(at(lane));
            if (lane == 0) total = s;
        }
        __syncthreads();
        if (pass == 0) mean = d.n_inner > 0.0 ? total / d.n_inner : 0.0;
        else if (threadIdx.x == 0) begin_solve(d, cs[blockIdx.x], total, active_out + blockIdx.x);
        if (pass == 0 && threadIdx.x == 0) cs[blockIdx.x].rhs_mean = mean;
    }
}

// ------------------------------------------------ lexicographic (reference)

// src/math.rs:176-186, squared -- one term of the reference's norm fold.
__device__ __forceinline__ double ref_residual_sq(const double* __restrict__ p,
                                                  const double* __restrict__ rhs, int64_t i,
                                                  int64_t P, double dx2, double dy2) {
    const double pc = p[i];
    const double part1 = ((p[i + P] - pc) - (pc - p[i - P])) / dx2;
    const double part2 = ((p[i + 1] - pc) - (pc - p[i - 1])) / dy2;
    const double r = (part1 + part2) - rhs[i];
    return r * r;
}

// acc + s[0] + s[1] + ... + s[n - 1], added left to right, from LDS: every
// lane of the wave reads the same address (a broadcast, no bank conflict),
// sixteen reads in flight, then their additions, one dependent add per term.
__device__ __forceinline__ double lds_ordered_sum(double acc, const double* s, int n) {
    int k = 0;
    for (; k + 16 <= n; k += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = s[k + u];
#pragma unroll
        for (int u = 0; u < 16; u++) acc = acc + v[u];
    }
    for (; k < n; k++) acc = acc + s[k];
    return acc;
}

// The sequential sum from 0.0 of the interior terms t[(x, y)] >= 0, x-major
// (x outer, y inner), by the first wave of the workgroup: the wave loads 64
// consecutive terms of a row at once, eight such chunks per batch, puts the
// batch in `stage` (512 doubles of LDS) in that order and adds it term by
// term, so the additions are the sequential ones in the same order, bit for
// bit.  Lanes past the end of a row add +0.0, which leaves the sum unchanged:
// it starts at +0.0 and adds squares, so it is never -0.0 (a NaN or infinity
// stays what it is).  A wave's LDS accesses complete in order, so the batch
// it stored is what it reads back (the wavefront-scope fences keep the
// compiler from moving them).
__device__ __forceinline__ double ordered_row_sum(const double* __restrict__ t, int64_t base,
                                                  int64_t P, int nxi, int nyi, double* stage) {
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    if (nxi <= 0 || nyi <= 0) return acc;
    const int64_t chunks = (int64_t)nxi * ((nyi + 63) / 64);
    int x = 1, y0 = 0;   // the next chunk to load: row x, terms 1 + y0 ..
    // that chunk: every lane loads (an address clamped into the channel, so
    // the loads are unconditional and all of a batch are in flight together),
    // and `in` says whether the lane's term is part of the sum (not past the
    // row or the last row)
    auto take = [&](bool& in) -> double {
        in = x <= nxi && y0 + lane < nyi;
        const double v = t[base + (int64_t)min(x, nxi) * P + 1 + min(y0 + lane, nyi - 1)];
        y0 += 64;
        if (y0 >= nyi) {
            y0 = 0;
            x++;
        }
        return v;
    };
    constexpr int U = 8;
    for (int64_t k = 0; k < chunks; k += U) {
        double v[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = take(in[u]);
#pragma unroll
        for (int u = 0; u < U; u++) stage[u * 64 + lane] = in[u] ? v[u] : 0.0;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        acc = lds_ordered_sum(acc, stage, U * 64);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    return acc;
}

// src/simulation.rs:216-227: sum r^2 over every interior cell, x-major,
// sequentially from 0.0, divided by the fluid count.  The squares are formed
// in parallel; the first wave then folds them in the reference's order.
__device__ double ref_norm_squared(const ChanDesc& d, const double* __restrict__ p,
                                   const double* __restrict__ rhs, double* __restrict__ sq,
                                   double* sh_out) {
    const int nxi = d.nx - 2, nyi = d.ny - 2;
    const int64_t P = d.pitch;
    for (int k = threadIdx.x; k < nxi * nyi; k += blockDim.x) {
        const int x = 1 + k / nyi, y = 1 + k % nyi;
        const int64_t i = d.off + x * P + y;
        sq[i] = ref_residual_sq(p, rhs, i, P, d.delx2, d.dely2);
    }
    __syncthreads();
    __shared__ double stage[512];
    if (threadIdx.x < 64) {
        const double acc = ordered_row_sum(sq, d.off, P, nxi, nyi, stage);
        if (threadIdx.x == 0) *sh_out = acc / d.fluid_cells;
    }
    __syncthreads();
    return *sh_out;
}

// Construction (src/simulation.rs:94-96 -> 229-237): initial_norm_squared
// when the state carries none.  The squares first, by the whole chip, dense in
// the norm's order (x-major) ...
__global__ void __launch_bounds__(256)
k_norm_squares(const ChanDesc* __restrict__ cd, const ChanState* __restrict__ cs,
               const double* __restrict__ rhs, const double* __restrict__ p,
               double* __restrict__ sq, uint32_t per)   // per: workgroups of a channel
{
    const uint32_t c = blockIdx.x / per, part = blockIdx.x - c * per;
    if (cs[c].has_init) return;
    const ChanDesc& d = cd[c];
    const int nxi = d.nx - 2, nyi = d.ny - 2;
    const int64_t n = (int64_t)nxi * nyi, P = d.pitch;
    for (int64_t k = part * 256 + threadIdx.x; k < n; k += (int64_t)per * 256) {
        const int64_t i = d.off + (1 + k / nyi) * P + 1 + k % nyi;
        sq[d.off + k] = ref_residual_sq(p, rhs, i, P, d.delx2, d.dely2);
    }
}

// ... then their sum, one after another.  That chain is what bounds the call:
// a dependent FP64 add takes 4.6 cycles, so nothing may come between two of
// them.  The terms are read as scalars (an add takes one operand from there),
// sixteen (two cache lines) at a time and a block ahead; a scalar cache miss is far longer than
// a block, so the other waves read the next segment of the terms into
// that cache while the first adds this one.  Construction of 1002 x 503 cells:
// 3.24 -> 1.49 ms, 7.1 cycles a term (a scalar cache hit is still a little
// longer than a block; blocks of twenty, which straddle lines, took 8.5), and
// 17 with the terms broadcast from LDS as before.
constexpr int NORM_WAVES = 12;
constexpr int NORM_SEG = 512;   // terms of a segment, 4 KB: two of them fit the 16 KB cache
__global__ void __launch_bounds__(64 * NORM_WAVES)
k_initial_norm(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
               const double* __restrict__ sq)
{
    const ChanDesc& d = cd[blockIdx.x];
    ChanState& s = cs[blockIdx.x];
    if (s.has_init) return;
    using Scalars = const double __attribute__((address_space(4)))*;
    const Scalars t = (Scalars)(uintptr_t)(sq + d.off);
    const int n = (d.nx - 2) * (d.ny - 2);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // a wave's share of the segment at s0, all its lines (8 terms) in flight
    auto touch = [&](int s0) {
        constexpr int SHARE = (NORM_SEG / 8 + NORM_WAVES - 2) / (NORM_WAVES - 1);
        double v[SHARE];
#pragma unroll
        for (int j = 0; j < SHARE; j++)
            v[j] = t[min(s0 + 8 * ((wave - 1) * SHARE + j), n - 1)];
        static_assert(SHARE == 6, "one statement takes all of them, so that they are in flight together");
        asm volatile("" :: "s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]), "s"(v[4]), "s"(v[5]));
    };
    double acc = 0.0;
    if (wave > 0) touch(0);
    __syncthreads();
    for (int s0 = 0; s0 < n; s0 += NORM_SEG) {
        if (wave > 0) {
            touch(s0 + NORM_SEG);
        } else {
            constexpr int B = 16;
            const int end = min(s0 + NORM_SEG, n), whole = s0 + (end - s0) / (2 * B) * (2 * B);
            double v[B], w[B];
            // adds a, whose loads were issued a block ago, while b's are on
            // their way (issued once a has come: scalar loads return in no
            // order, so a wait is for all of them)
            auto block = [&](const double (&a)[B], double (&b)[B], int next) {
                acc = acc + a[0];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < B; u++) b[u] = t[next + u];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 1; u < B; u++) acc = acc + a[u];
                __builtin_amdgcn_sched_barrier(0);
            };
            // (a block past the last one may be read, not added: the channel's
            // slice is longer than its interior by two rows)
#pragma unroll
            for (int u = 0; u < B; u++) v[u] = t[s0 + u];
            for (int k = s0; k < whole; k += 2 * B) {
                block(v, w, k + B);
                block(w, v, k + 2 * B);
            }
            for (int k = whole; k < end; k++) acc = acc + t[k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        s.init_norm2 = acc / d.fluid_cells;
        s.has_init = 1;
    }
}

// src/simulation.rs:266-270: the SOR update of one fluid cell from its x + 1,
// x - 1, y + 1 and y - 1 neighbours, in the reference's association.
__device__ __forceinline__ double lex_update(const ChanDesc& d, double pc, double pxp, double pxm,
                                             double pyp, double pym, double r) {
    return (d.omw * pc) + (d.mid * ((((pxp + pxm) / d.delx2) + ((pyp + pym) / d.dely2)) - r));
}

// The most sweeps that k_lex_solve does of a solve that the pipeline can go on with.
constexpr int LEX_FEW = 2;

// src/simulation.rs:239-285 for the channels with solver == SOLVER_LEX that no
// instance of the pipelined solve takes (kernels_lex.hip: more than 512 rows, or no
// scratch for them), and the first LEX_FEW sweeps of solves that are expected to be
// short (lex_few, lex_begin): the pipeline's set-up (its diagonal-major copies) and
// its longer step pay from the second or third sweep on.  A solve (statistics
// included) of 102 x 22 cells in one sweep: 73 us here, 87 there; in two 113 and 88,
// in four 196 and 90.
// Lexicographic Gauss-Seidel order (x outer, y inner, in place) makes cell
// (x, y) read the new W and N values and the old E and S values; sweeping the
// anti-diagonals x + y = const in increasing order, with a barrier between
// them, reproduces exactly those reads, so the result is bit-identical.
//
// A channel that fits LEX_LDS_CELLS is staged in LDS once (p, rhs, the flags and the
// norm's terms, 115 KB), iterated there and written back: the same operations on the same values in the same order.  The
// first wave sweeps alone, a lane per cell of a diagonal: a wave's LDS accesses
// complete in order, so it needs no workgroup barrier between diagonals (the
// wavefront-scope fence keeps the compiler from reordering).  Three sizes (67 x
// 67, 67 x 68, 68 x 67) have a diagonal of 65 cells and a loop over it, which in
// the others' sweeps cost 7% of a solve of one sweep (102 x 22 cells).
__global__ void __launch_bounds__(1024)
k_lex_solve(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
            const BEntry* __restrict__ be, const uint8_t* __restrict__ flags,
            const double* __restrict__ rhs, double* __restrict__ p, double* __restrict__ scratch)
{
    __shared__ double sh_norm;
    __shared__ double sp[LEX_LDS_CELLS], srhs[LEX_LDS_CELLS], ssq[LEX_LDS_CELLS];
    __shared__ uint8_t sfl[LEX_LDS_CELLS];
    const ChanDesc d = cd[blockIdx.x];
    if (d.solver != SOLVER_LEX) return;
    ChanState& s = cs[blockIdx.x];
    const bool few = d.lex_class >= 0;
    if (few && !lex_few(d.lex_begin, d.itermax, s)) return;
    const int limit = few ? min(d.itermax, LEX_FEW) : d.itermax;
    const int nxi = d.nx - 2, nyi = d.ny - 2;
    const int64_t P = d.pitch;
    const double init = s.init_norm2;
    const int tid = threadIdx.x;
    double norm2 = 0.0;
    int iters = d.itermax, exhausted = 1;
    const int ny = d.ny, ncell = d.nx * d.ny;
    if (ncell <= LEX_LDS_CELLS) {
        for (int l = tid; l < ncell; l += blockDim.x) {
            const int x = l / ny, y = l - (l / ny) * ny;
            const int64_t g = d.off + x * P + y;
            sp[l] = p[g];
            srhs[l] = rhs[g];
            sfl[l] = flags[g];
        }
        __syncthreads();
        for (int it = 0; it < limit; it++) {
            // copy_pressure_to_boundaries, src/grid/mod.rs:343-412
            for (int k = tid; k < d.nb; k += blockDim.x) {
                const BEntry e = be[d.boff + k];
                if (e.edge != E_NONE) {
                    const int64_t o = e.gidx - d.off;
                    const int l = (int)(o / P) * ny + (int)(o % P);
                    sp[l] = ghost_value(sp, l, ny, e.edge);
                }
            }
            __syncthreads();
            if (tid < 64) {
                // the flag and the values are read together (an interior
                // cell's neighbours are all in the channel); only a fluid
                // cell stores its update
                auto cell = [&](int x, int dd) {
                    const int l = x * ny + (dd - x);
                    const uint8_t f = sfl[l];
                    const double nv = lex_update(d, sp[l], sp[l + ny], sp[l - ny],
                                                 sp[l + 1], sp[l - 1], srhs[l]);
                    if (flag_fluid(f)) sp[l] = nv;
                };
                auto diagonals = [&](auto wide) {
                    for (int dd = 2; dd <= nxi + nyi; dd++) {
                        const int xlo = dd - nyi > 1 ? dd - nyi : 1;
                        const int xhi = dd - 1 < nxi ? dd - 1 : nxi;
                        if constexpr (wide.value) {
                            for (int x = xlo + tid; x <= xhi; x += 64) cell(x, dd);
                        } else if (xlo + tid <= xhi) {
                            cell(xlo + tid, dd);
                        }
                        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    }
                };
                if (min(nxi, nyi) <= 64) diagonals(std::false_type{});
                else diagonals(std::true_type{});
            }
            __syncthreads();
            // src/simulation.rs:216-227, as ref_norm_squared, on the LDS copy:
            // the terms in the reference's order (x-major over the interior),
            // then added in that order
            for (int k = tid; k < nxi * nyi; k += blockDim.x) {
                const int l = (1 + k / nyi) * ny + 1 + k % nyi;
                ssq[k] = ref_residual_sq(sp, srhs, l, ny, d.delx2, d.dely2);
            }
            __syncthreads();
            if (tid < 64) {
                const double acc = lds_ordered_sum(0.0, ssq, nxi * nyi);
                if (tid == 0) sh_norm = acc / d.fluid_cells;
            }
            __syncthreads();
            norm2 = sh_norm;
            if ((norm2 < init) || (norm2 < d.eps2)) {
                iters = it + 1;
                exhausted = 0;
                break;
            }
        }
        for (int l = tid; l < ncell; l += blockDim.x) {
            const int x = l / ny, y = l - (l / ny) * ny;
            p[d.off + x * P + y] = sp[l];
        }
        if (few && exhausted && limit < d.itermax) {   // the pipeline goes on from here
            if (tid == 0) s.budget = limit;
            return;
        }
        if (tid == 0) {
            s.budget = -1;
            s.lex_exact -= s.lex_exact > 0;
            s.sor_iters = (uint32_t)iters;
            s.norm2 = norm2;
            s.exhausted = exhausted;
            s.active = 0;
        }
        return;
    }
    for (int it = 0; it < limit; it++) {
        // copy_pressure_to_boundaries, src/grid/mod.rs:343-412
        for (int k = threadIdx.x; k < d.nb; k += blockDim.x) {
            const BEntry e = be[d.boff + k];
            if (e.edge != E_NONE) p[e.gidx] = ghost_value(p, e.gidx, e.pitch, e.edge);
        }
        __syncthreads();
        for (int dd = 2; dd <= nxi + nyi; dd++) {
            const int xlo = dd - nyi > 1 ? dd - nyi : 1;
            const int xhi = dd - 1 < nxi ? dd - 1 : nxi;
            for (int x = xlo + (int)threadIdx.x; x <= xhi; x += blockDim.x) {
                const int y = dd - x;
                const int64_t i = d.off + x * P + y;
                // the flag and the values are read together; only a fluid
                // cell stores its update
                const uint8_t f = flags[i];
                const double nv = lex_update(d, p[i], p[i + P], p[i - P], p[i + 1], p[i - 1],
                                             rhs[i]);
                if (flag_fluid(f)) p[i] = nv;
            }
            __syncthreads();
        }
        norm2 = ref_norm_squared(d, p, rhs, scratch, &sh_norm);
        if ((norm2 < init) || (norm2 < d.eps2)) {
            iters = it + 1;
            exhausted = 0;
            break;
        }
    }
    if (few && exhausted && limit < d.itermax) {
        if (threadIdx.x == 0) s.budget = limit;
        return;
    }
    if (threadIdx.x == 0) {
        s.budget = -1;
        s.lex_exact -= s.lex_exact > 0;
        s.sor_iters = (uint32_t)iters;
        s.norm2 = norm2;
        s.exhausted = exhausted;
        s.active = 0;
    }
}

// ---------------------------------------------------------------- launchers

#define TB dim3(TILE_Y, TILE_X)

void launch_ghost(hipStream_t st, int nbtot, const BEntry* be, const ChanState* cs, double* p,
                  int colour, int only_active) {
    if (nbtot > 0)
        k_ghost<<<(nbtot + 255) / 256, 256, 0, st>>>(nbtot, be, cs, p, colour, only_active);
}
void launch_rhs_stats(hipStream_t st, int ntiles, int nchan, const ChanDesc* cd, ChanState* cs,
                      const Tile* tiles, const uint8_t* flags, const double* rhs, double* part) {
    k_rhs_sums<<<ntiles, dim3(TILE_Y, TILE_X), 0, st>>>(cd, cs, tiles, flags, rhs, part, 0);
    k_rhs_mean<<<nchan, 256, 0, st>>>(cd, cs, part);
    k_rhs_sums<<<ntiles, dim3(TILE_Y, TILE_X), 0, st>>>(cd, cs, tiles, flags, rhs, part, 1);
}
void launch_solve_stats(hipStream_t st, int nchan, const ChanDesc* cd, ChanState* cs,
                        const Tile* tiles, const uint8_t* flags, const double* rhs,
                        int32_t* active) {
    k_solve_stats<<<nchan, 1024, 0, st>>>(cd, cs, tiles, flags, rhs, active);
}
void launch_solve_begin(hipStream_t st, int nchan, const ChanDesc* cd, ChanState* cs,
                        const double* part, int32_t* active) {
    k_solve_begin<<<nchan, 256, 0, st>>>(cd, cs, part, active);
}
void launch_initial_norm(hipStream_t st, int nchan, const ChanDesc* cd, ChanState* cs,
                         const double* rhs, const double* p, double* scratch) {
    // four workgroups a CU over all channels, each with a few cells a thread
    // (in x, whose grids are not limited to 65536)
    const uint32_t per = (uint32_t)std::max(1, 1024 / nchan);
    k_norm_squares<<<per * (uint32_t)nchan, 256, 0, st>>>(cd, cs, rhs, p, scratch, per);
    k_initial_norm<<<nchan, 64 * NORM_WAVES, 0, st>>>(cd, cs, scratch);
}
void launch_lex_solve(hipStream_t st, int nchan, const ChanDesc* cd, ChanState* cs,
                      const BEntry* be, const uint8_t* flags, const double* rhs, double* p,
                      double* scratch) {
    k_lex_solve<<<nchan, 1024, 0, st>>>(cd, cs, be, flags, rhs, p, scratch);
}

}  // namespace stm
