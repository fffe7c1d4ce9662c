// Temporally blocked red-black SOR for gfx950.
//
// Launch L of a solve advances every running channel by up to K full sweeps.
// Each workgroup owns an output tile; it loads the tile plus a halo of
// H = 2K + 2 cells, performs the K sweeps on chip and writes the output tile
// back.  A dependency reaches one cell per half-sweep: after K sweeps the red
// cells are exact from the region's ring 2K - 1 on and the black ones from 2K
// (ring 0 is its border), the ghosts refreshed from them from 2K + 1 and the
// residual that reads those from 2K + 2.  This needs every ghost of the input
// to be fresh, which the launch before leaves behind and a ghost refresh in
// front of launch 0 provides.  Nothing beyond a channel's edge feeds a tile,
// so on an edge side the region needs no halo: it starts two cells outside
// the channel (origins are even in x and y, which keeps 16-byte pairs aligned
// and one colour pattern for every tile), and edge tiles output that much more.
// The result is bit-identical to K separate global sweeps of
//     refresh all ghosts; red half-sweep; black half-sweep
// (same operations on the same operands) while the cache / HBM traffic drops
// by about K times.
//
// Schedule inside a launch: ghosts take the colour of their cell and read
// only fluid cells of the other colour, and a cell of colour c reads only
// cells of the other colour.  The refresh at the start of a sweep gives a red
// ghost the black values the sweep starts with: the red half, which leaves
// black cells alone, can form it.  It gives a black ghost the red values the
// sweep starts with, those the black half of the sweep before found.  So a
// ghost is refreshed in the half-sweep of its own colour, by a select in place
// of the update; the red ones once more after the last sweep.  Two barriers
// per sweep.
//
// Registers and LDS: the region is EX x EY cells; a strip is R rows of it,
// held by one wave in registers, p and rhs, lane m the y-pair (2m, 2m + 1) of
// every row -- one red and one black cell each.  E / W neighbours are the
// lane's own registers, one of N / S is the pair's other cell and the other
// comes from the next lane by DPP; only a
// strip's first and last row go through LDS, for the strips next to it.  A
// cell then costs 7 FP64 operations and two 32-bit moves (43 cycles per wave
// and row measured, 36 issued), and a half-sweep 150 cycles on top for the
// barrier and the LDS round trip.  An earlier form published every cell to LDS
// and spent as long on LDS as on arithmetic (2350 cycles per sweep of 96 x 96
// cells on a CU; now 2250 for 80 x 128).  Ten rows a strip is what 128
// registers hold, and 128 let two workgroups of eight strips share a CU: one
// loads and stores (2.5 us each way) while the other sweeps.  Per sweep,
// before and now: 4002 x 3002 cells 29.9 -> 17.8 us (8 a launch) and 16.4 us
// (6), 32 channels of 514 x 258 10.2 -> 6.8 us, one of 1026 x 1026, where a
// launch is a single round of workgroups and mostly its loads and stores, 2.31
// -> 2.32 us (6 a launch).  Longer strips (18 rows, one workgroup of four)
// leave a SIMD one wave, which hides no latency: 3.4 us there.
//
// Launch order: workgroups go to the XCDs round-robin; the host orders each
// channel's tiles so that every XCD gets one compact block of them (shared
// halos come from that XCD's L2).
//
// No fences, no second kernel: launch L writes one residual partial per tile;
// every workgroup of launch L + 1 folds the previous launch's partials of its
// channel in tile order, so all take the same stop decision; the channel's
// first tile records it.  p ping-pongs between two buffers (workgroups read
// each other's halos).
//
// What the cells are does not change between launches: k_rb_codes turns the
// flags into tables when the tiles are planned (and when cells are edited).
// Most strips hold updated cells only and use none of it.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"
#include "stm_internal.h"
#include "wave.h"

namespace stm {

namespace {

// For a ghost cell, the fluid neighbours its pressure copies
// (src/grid/mod.rs:343-412): N, S, E, W; one bit for a straight edge, a
// vertical and a horizontal one for a corner, whose ghost is their mean.
enum : uint32_t { C_GN = 1, C_GS = 2, C_GE = 4, C_GW = 8 };

// ghost_bits(e), 4 bits per edge kind E_N .. E_NW (0 for E_NONE and above E_NW)
constexpr uint64_t GHOST_TAB =
    (uint64_t)C_GN << (4 * E_N) | (uint64_t)(C_GN | C_GE) << (4 * E_NE) |
    (uint64_t)C_GE << (4 * E_E) | (uint64_t)(C_GS | C_GE) << (4 * E_SE) |
    (uint64_t)C_GS << (4 * E_S) | (uint64_t)(C_GS | C_GW) << (4 * E_SW) |
    (uint64_t)C_GW << (4 * E_W) | (uint64_t)(C_GN | C_GW) << (4 * E_NW);

__device__ __forceinline__ uint32_t ghost_bits(uint32_t edge) {
    return (uint32_t)(GHOST_TAB >> (4 * (edge & 15u))) & 15u;
}

// A cell's code, 16 bits (a pair's word holds cell q in bits 16q ..): updated
// by SOR; in the output tile; an output cell that no sweep changes; and a
// ghost's neighbours (ghost_bits).
enum : uint32_t { K_UPD = 1, K_OUT = 2, K_REST = 4, K_GHOST = 8 };

// A lane's word after its rows' words: in every row that is not special, the
// cell of slot 0 (0) or 1 (1) is a straight ghost of its N or S neighbour, or
// feeds nothing (walls along x).  0S and 1N are ghosts of the pair's other cell.
enum : uint32_t { G_0S = 1, G_1N = 2, G_0N = 4, G_1S = 8 };

// The workgroup's sum of v, in wave order, for thread 0 (the last use of
// wsum in the kernel: no barrier after it).
template <int NT>
__device__ __forceinline__ double block_sum_to_first(double v, double* wsum) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
#pragma unroll
        for (int w = 0; w < NT / 64; w++) s = s + wsum[w];
    return s;
}

// The next lower / higher lane's value (of lane 0 / 63: 0, which only border
// cells of the region read).
template <int CTRL>
__device__ __forceinline__ double dpp_shift(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_below(double v) { return dpp_shift<0x138>(v); }
__device__ __forceinline__ double lane_above(double v) { return dpp_shift<0x130>(v); }

constexpr int LW = 64;   // lanes of a strip: one wave

// The sweeps of one strip.  Rows start at an even x and pairs at an even y:
// cell (row r, slot q) has colour (r & 1) ^ q.
template <int R, int NS>
struct Strip {
    // the first (end 0) and last (end 1) row of every strip, by colour; strip
    // s at s + 1, so that the outer strips' reads stay in bounds (what they
    // get goes to the region's border)
    double (*E)[NS + 2][2][LW];
    const uint32_t* W;       // this lane's code words, row r at r * LW (coded waves)
    int strip, m;
    double omw, mid, rdx2, rdy2;

    struct Ends { double e, w; };
    __device__ __forceinline__ Ends ends(int c) const {   // colour c beyond the strip's rows
        return {E[c][strip + 2][0][m], E[c][strip][1][m]};
    }
    template <int r>
    __device__ __forceinline__ void publish(int c, const double (&pv)[R][2]) const {
        if (r == 0) E[c][strip + 1][0][m] = pv[0][c];
        if (r == R - 1) E[c][strip + 1][1][m] = pv[R - 1][c ^ 1];   // R is even
    }

    struct Around { double n, s, e, w; };
    template <int r, int q>
    __device__ __forceinline__ Around around(const double (&pv)[R][2], const Ends& x) const {
        Around a;
        a.n = q ? pv[r][0] : lane_below(pv[r][1]);
        a.s = q ? lane_above(pv[r][0]) : pv[r][1];
        a.e = r + 1 < R ? pv[r + 1 < R ? r + 1 : r][q] : x.e;
        a.w = r > 0 ? pv[r > 0 ? r - 1 : r][q] : x.w;
        return a;
    }

    // Ghost value (src/grid/mod.rs:343-412): one fluid neighbour, or
    // (a + b) * 0.5 of a vertical and a horizontal one; ghost bits g != 0.
    __device__ static __forceinline__ double ghost_value(uint32_t g, const Around& n) {
        const double a = (g & C_GN) ? n.n : n.s;
        const double b = (g & C_GE) ? n.e : n.w;
        const bool vert = g & (C_GN | C_GS), horz = g & (C_GE | C_GW);
        return vert ? (horz ? (a + b) * 0.5 : a) : b;
    }

    __device__ __forceinline__ double relaxed(double pc, const Around& n, double rr) const {
        const double tt = fma(n.e + n.w, rdx2, (n.s + n.n) * rdy2);
        return fma(omw, pc, mid * (tt - rr));
    }

    // Row r of the half-sweep of colour c.  Every value read has colour
    // c ^ 1, which the half does not change.
    //
    // An ordinary row holds, besides updated cells and the ghosts that the
    // lanes' words give, only cells whose value feeds nothing, and stores into
    // them: a cell with no fluid neighbour (solid) is read by no update, and an
    // output cell of that kind is taken from the input at write-back; cells on
    // the region's border or outside the channel are never output, and what
    // they hold reaches the output no sooner than their staleness would.  The
    // other rows are special: those with any other ghost or with a fluid cell
    // that is not updated.
    //
    // G: the lanes' ghosts the wave holds.
    template <int c, int r, uint32_t G, bool SPECIAL>
    __device__ __forceinline__ void row(double (&pv)[R][2], const double (&rr)[R][2],
                                        const Ends& x, uint32_t lane, uint32_t special) const {
        constexpr int q = c ^ (r & 1);
        constexpr uint32_t GS = q ? G_1S : G_0S, GN = q ? G_1N : G_0N;
        const double pc = pv[r][q];
        const Around n = around<r, q>(pv, x);
        double v = relaxed(pc, n, rr[r][q]);
        if (SPECIAL && ((special >> r) & 1u)) {
            const uint32_t k = W[r * LW] >> (16 * q), g = (k >> K_GHOST) & 15u;
            v = (k & K_UPD) ? v : pc;
            v = g ? ghost_value(g, n) : v;
        } else {
            if (G & GS) v = (lane & GS) ? n.s : v;
            if (G & GN) v = (lane & GN) ? n.n : v;
        }
        pv[r][q] = v;
        // finished here: rows whose last operation waits for the others' would
        // each hold two more registers
        asm volatile("" : "+v"(pv[r][q]));
        publish<r>(c, pv);
    }

    // Rows r0 .. r1 - 1; SPECIAL: some row of the wave is special (looked at
    // four rows at a time, so that the other rows run without branches).
    template <int c, int r0, int r1, uint32_t G, bool SPECIAL>
    __device__ __forceinline__ void rows(double (&pv)[R][2], const double (&rr)[R][2],
                                         const Ends& x, uint32_t lane, uint32_t special) const {
        if constexpr (r0 < r1) {
            row<c, r0, G, SPECIAL>(pv, rr, x, lane, special);
            rows<c, r0 + 1, r1, G, SPECIAL>(pv, rr, x, lane, special);
        }
    }
    template <int c, int r0, int r1, uint32_t G, bool SPECIAL>
    __device__ __forceinline__ void some(double (&pv)[R][2], const double (&rr)[R][2],
                                         const Ends& x, uint32_t lane, uint32_t special) const {
        if constexpr (!SPECIAL) {
            rows<c, r0, r1, G, false>(pv, rr, x, lane, special);
        } else if constexpr (r0 < r1) {
            constexpr int e = r0 + 4 < r1 ? r0 + 4 : r1;
            if ((special >> r0) & ((1u << (e - r0)) - 1u))
                rows<c, r0, e, G, true>(pv, rr, x, lane, special);
            else
                rows<c, r0, e, G, false>(pv, rr, x, lane, special);
            some<c, e, r1, G, true>(pv, rr, x, lane, special);
        }
    }
    // A half-sweep, from a barrier to a barrier: some inner rows while the
    // ends' LDS reads are on their way, the end rows, and the other inner rows
    // while their values are written.
    template <int c, uint32_t G, bool SPECIAL>
    __device__ __forceinline__ void half_as(double (&pv)[R][2], const double (&rr)[R][2],
                                            const Ends& x, uint32_t lane, uint32_t special) const {
        some<c, 1, R / 2, G, SPECIAL>(pv, rr, x, lane, special);
        some<c, 0, 1, G, SPECIAL>(pv, rr, x, lane, special);
        some<c, R - 1, R, G, SPECIAL>(pv, rr, x, lane, special);
        some<c, R / 2, R - 1, G, SPECIAL>(pv, rr, x, lane, special);
    }
    // In the wave's form (uniform branches inside one loop over the sweeps, so
    // that the forms share their registers).  A lane's ghost costs two 32-bit
    // selects in the rows that can hold it, so the usual combinations -- a wall
    // on one side, or one on each -- have their own forms.
    template <int c>
    __device__ __forceinline__ void half(double (&pv)[R][2], const double (&rr)[R][2], uint32_t g,
                                         uint32_t lane, uint32_t special) const {
        const Ends x = ends(c ^ 1);
        constexpr uint32_t ANY = G_0S | G_1N | G_0N | G_1S;
        if (special == 0) {
            if (g == 0) half_as<c, 0, false>(pv, rr, x, lane, special);
            else if (g == G_0S) half_as<c, G_0S, false>(pv, rr, x, lane, special);
            else if (g == G_1N) half_as<c, G_1N, false>(pv, rr, x, lane, special);
            else if (g == G_0N) half_as<c, G_0N, false>(pv, rr, x, lane, special);
            else if (g == (G_0S | G_1N)) half_as<c, G_0S | G_1N, false>(pv, rr, x, lane, special);
            else if (g == (G_0S | G_0N)) half_as<c, G_0S | G_0N, false>(pv, rr, x, lane, special);
            else half_as<c, ANY, false>(pv, rr, x, lane, special);
        } else {
            if (g == 0) half_as<c, 0, true>(pv, rr, x, lane, special);
            else half_as<c, ANY, true>(pv, rr, x, lane, special);
        }
        __syncthreads();
    }

    // The red ghosts from the final black values.
    template <int r = 0>
    __device__ __forceinline__ void red_ghosts(double (&pv)[R][2], const Ends& black,
                                               uint32_t lane, uint32_t g, uint32_t special) const {
        if constexpr (r < R) {
            constexpr int q = r & 1;
            constexpr uint32_t GS = q ? G_1S : G_0S, GN = q ? G_1N : G_0N;
            if ((special >> r) & 1u) {
                const uint32_t k = (W[r * LW] >> (16 * q + K_GHOST)) & 15u;
                const Around n = around<r, q>(pv, black);
                pv[r][q] = k ? ghost_value(k, n) : pv[r][q];
            } else if (g & (GS | GN)) {
                const Around n = around<r, q>(pv, black);
                const double v = (lane & GS) ? n.s : pv[r][q];
                pv[r][q] = (lane & GN) ? n.n : v;
            }
            publish<r>(0, pv);
            red_ghosts<r + 1>(pv, black, lane, g, special);
        }
    }

    // Sum of r^2 over row r's cells that `in` takes (ghosts fresh).
    template <int r>
    __device__ __forceinline__ double residual(const double (&pv)[R][2], const double (&rr)[R][2],
                                               const Ends (&x)[2], bool in0, bool in1) const {
        double acc = 0.0;
        const Around a[2] = {around<r, 0>(pv, x[(r & 1) ^ 1]), around<r, 1>(pv, x[r & 1])};
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const double pc = pv[r][q];
            const double h = (a[q].e - pc) - (pc - a[q].w);
            const double v = (a[q].s - pc) - (pc - a[q].n);
            const double res = fma(h, rdx2, v * rdy2) - rr[r][q];
            acc = acc + ((q ? in1 : in0) ? res * res : 0.0);
        }
        return acc;
    }
};

}  // namespace

template <int R, int HY, int NS>
__global__ void __launch_bounds__(NS * LW, 4)
k_rb_strip(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
           const TbTile* __restrict__ tiles, const TbWave* __restrict__ waves,
           const uint32_t* __restrict__ words, const double* __restrict__ rhs,
           double* __restrict__ pa, double* __restrict__ pb,
           const double* __restrict__ part_prev, double* __restrict__ part_cur,
           int32_t* __restrict__ active_out, int K, int L, int mode)
{
    constexpr int NT = NS * LW;
    static_assert(NT <= 1024 && HY <= LW, "workgroup size");
    static_assert(R % 2 == 0 && R >= 4 && R < 32, "rows per strip");

    __shared__ double ends[2][NS + 2][2][LW];
    __shared__ uint32_t kw[NS * R * LW];
    __shared__ double wsum[NS];

    // The tile carries its channel's geometry: the region's loads issue after
    // one scalar load, together with the channel's state.
    const TbTile t = tiles[blockIdx.x];
    const int c = t.chan;
    ChanState& s = cs[c];
    // read here, tested only after the loads: no load waits for it
    const int stopped = s.stop_launch;
    const double mean = s.rhs_mean;
    const ChanDesc& d = cd[c];
    const int budget = s.budget, d_itermax = d.itermax;
    const double tol2 = s.tol2;
    const int tid = threadIdx.x;
    const bool check = mode & TB_CHECK;
    const double* __restrict__ pin = (L & 1) ? pb : pa;
    double* __restrict__ pout = (L & 1) ? pa : pb;

    const int strip = __builtin_amdgcn_readfirstlane(tid / LW), m = tid % LW;
    const int lx0 = strip * R;
    const int gx0 = t.rx0 + lx0, gy = t.ry0 + 2 * m;   // both even
    const int64_t pitch = t.pitch;

    // The previous launch's residual partials of this channel: the first
    // share is loaded with the region below, unconditionally (clamped index).
    const bool sum_parts = L > 0 && check;
    const double part0 = part_prev[t.tb0 + min(tid, t.ntb - 1)];
    const TbWave wv = waves[(int64_t)t.idx * NS + strip];

    // ---- load; the solve is for rhs - mean (the all-Neumann problem needs
    // zero mean).  Every address is clamped into the channel (rows of pitch
    // >= ny + 1 for odd ny, so an aligned pair load at the last even y is in
    // bounds); what cells outside the channel hold feeds nothing.
    double pv[R][2], rr[R][2];
    {
        const int gyc = min(max(gy, 0), (t.ny - 1) & ~1);
        double2 pp[R], rh[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int64_t row = t.off + (int64_t)min(max(gx0 + r, 0), t.nx - 1) * pitch;
            pp[r] = *reinterpret_cast<const double2*>(pin + row + gyc);
            rh[r] = *reinterpret_cast<const double2*>(rhs + row + gyc);
        }
        // every load is issued before any of them is used
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            pv[r][0] = pp[r].x;
            pv[r][1] = pp[r].y;
            rr[r][0] = rh[r].x - mean;
            rr[r][1] = rh[r].y - mean;
            // formed here, not after the stop test
            asm volatile("" : "+v"(rr[r][0]), "+v"(rr[r][1]), "+v"(pv[r][0]), "+v"(pv[r][1]));
        }
    }
    double pacc = sum_parts && tid < t.ntb ? part0 : 0.0;
    // a channel that has stopped: nothing to do (uniform; the loads above
    // are in bounds and their results unused)
    if (stopped >= 0) return;

    // ---- every thread adds its share of the partials in a fixed order,
    // waves add theirs, and after the barrier below every thread adds the wave sums
    // in wave order: the same sum, bit for bit, in every tile of the channel
    if (sum_parts) {
        for (int i = t.tb0 + tid + NT; i < t.tb0 + t.ntb; i += NT) pacc = pacc + part_prev[i];
        const double w = wave_sum(pacc);
        if (m == 0) wsum[strip] = w;
    }

    Strip<R, NS> st;
    st.E = ends;
    st.W = kw + strip * R * LW + m;
    st.strip = strip;
    st.m = m;
    st.omw = d.omw;
    st.mid = d.mid;
    st.rdx2 = d.rdx2;
    st.rdy2 = d.rdy2;
    st.template publish<0>(0, pv);
    st.template publish<0>(1, pv);
    st.template publish<R - 1>(0, pv);
    st.template publish<R - 1>(1, pv);
    // the codes of a strip that is not all updated cells (each lane reads its own:
    // no barrier)
    const bool coded = wv.form & TBW_CODED;
    uint32_t lane = 0;
    if (coded) {
        const uint32_t* src = words + ((int64_t)t.idx * NS + strip) * (R + 1) * LW + m;
#pragma unroll
        for (int r = 0; r < R; r++) kw[(strip * R + r) * LW + m] = src[r * LW];
        lane = src[R * LW];
    }
    __syncthreads();

    // ---- stop decision on the previous launch (identical in every tile)
    const int itermax = (budget > 0 && budget < d_itermax) ? budget : d_itermax;
    const int64_t swept = (int64_t)L * K;
    const int done = swept < itermax ? (int)swept : itermax;
    if (L > 0) {
        double res2 = 0.0;
        if (check)
#pragma unroll
            for (int w = 0; w < NS; w++) res2 = res2 + wsum[w];
        const bool conv = check && res2 <= tol2;
        // a residual that is not a number never meets the test: stop there
        // (the tick then reports it) instead of sweeping to itermax
        const bool nan = check && res2 != res2;
        if (conv || nan || done >= itermax) {
            if (t.idx == t.tb0 && tid == 0) {
                s.stop_launch = L - 1;
                s.sor_iters = (uint32_t)done;
                s.pbuf = L & 1;
                s.active = 0;
                s.exhausted = check && !conv;
                if (check) {
                    s.res2 = res2;
                    s.norm2 = res2 / d.fluid_cells;
                }
                active_out[c] = 0;
            }
            return;
        }
    }
    const int nsw = itermax - done < K ? itermax - done : K;

    // ---- the sweeps, in the wave's form (all forms meet at the same barriers)
    const uint32_t special = wv.special, g = wv.form & TBW_GHOSTS;
    for (int sw = 0; sw < nsw; sw++) {
        st.template half<0>(pv, rr, g, lane, special);
        st.template half<1>(pv, rr, g, lane, special);
    }
    using Ends = typename Strip<R, NS>::Ends;
    if ((g | special) != 0) st.red_ghosts(pv, st.ends(1), lane, g, special);

    // this tile's part of the residual, before the stores: the barrier of the
    // sum then waits for the residual, not for every wave's write-back
    const bool o0 = gy >= t.y0 && gy < t.y0 + t.yn, o1 = gy + 1 >= t.y0 && gy + 1 < t.y0 + t.yn;
    double acc = 0.0;
    if (check) {
        __syncthreads();   // the strip ends' red ghosts
        const Ends x[2] = {st.ends(0), st.ends(1)};
        auto sum = [&](auto self, auto rc) -> void {
            constexpr int r = decltype(rc)::value;
            if constexpr (r < R) {
                const bool in = gx0 + r >= t.x0 && gx0 + r < t.x0 + t.xn;
                bool in0 = in && o0, in1 = in && o1;
                if (coded) {
                    const uint32_t k = st.W[r * LW];
                    in0 = in0 && (k & K_UPD);
                    in1 = in1 && (k & (K_UPD << 16));
                }
                if (in) acc = acc + st.template residual<r>(pv, rr, x, in0, in1);
                self(self, std::integral_constant<int, r + 1>{});
            }
        };
        sum(sum, std::integral_constant<int, 0>{});
    }
    const double b = block_sum_to_first<NT>(acc, wsum);
    if (tid == 0) part_cur[t.idx] = b;

    // ---- write the output tile.  Output cells that are neither updated nor
    // ghosts keep their value in every sweep of the sequence (the sweeps may
    // have stored into their registers): launch 0 copies them from its input
    // buffer to its output buffer, after which both buffers hold them, and the
    // later launches leave them out.
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int gx = gx0 + r;
        if (gx < t.x0 || gx >= t.x0 + t.xn) continue;
        const int64_t g = t.off + (int64_t)gx * pitch + gy;
        bool w0 = o0, w1 = o1;
        if (coded && ((wv.rest >> r) & 1u)) {
            const uint32_t k = st.W[r * LW];
            const bool k0 = k & K_REST, k1 = k & (K_REST << 16);
            if (L == 0) {
                if (k0) pv[r][0] = pin[g];
                if (k1) pv[r][1] = pin[g + 1];
            } else {
                w0 = w0 && !k0;
                w1 = w1 && !k1;
            }
        }
        if (w0 && w1) *reinterpret_cast<double2*>(pout + g) = make_double2(pv[r][0], pv[r][1]);
        else if (w0) pout[g] = pv[r][0];
        else if (w1) pout[g + 1] = pv[r][1];
    }
}

// The tables of every tile's strips from the cell flags (one workgroup per
// tile, the sweeps' thread layout).
__global__ void __launch_bounds__(1024)
k_rb_codes(const TbTile* __restrict__ tiles, const uint8_t* __restrict__ flags, int R, int hy,
           int ex, TbWave* __restrict__ waves, uint32_t* __restrict__ words)
{
    const TbTile t = tiles[blockIdx.x];
    const int tid = threadIdx.x, strip = tid / LW, m = tid % LW;
    const int nx = t.nx, ny = t.ny, ey = 2 * hy;
    auto flag = [&](int x, int y) -> uint32_t {   // outside the channel: no cell
        return x >= 0 && x < nx && y >= 0 && y < ny
                   ? flags[t.off + (int64_t)x * t.pitch + y] : 0xffffu;
    };
    auto code = [&](int lx, int ly) -> uint32_t {
        const int x = t.rx0 + lx, y = t.ry0 + ly;
        const uint32_t f = flag(x, y);
        if (f == 0xffffu || m >= hy) return 0;
        const bool border = lx < 1 || lx > ex - 2 || ly < 1 || ly > ey - 2;
        const bool out = x >= t.x0 && x < t.x0 + t.xn && y >= t.y0 && y < t.y0 + t.yn;
        const bool fluid = f & F_FLUID;
        uint32_t k = out ? K_OUT : 0;
        if (fluid && !border && x >= 1 && x <= nx - 2 && y >= 1 && y <= ny - 2) k |= K_UPD;
        if (!fluid && !border) k |= ghost_bits(f & 15u) << K_GHOST;
        if (out && !(k & K_UPD) && (k >> K_GHOST) == 0) k |= K_REST;
        return k;
    };
    const int64_t at = (int64_t)t.idx * (blockDim.x / LW) + strip;
    uint32_t* dst = words + at * (R + 1) * LW + m;
    // what a slot of the lane holds, by rows: updated cells, ghosts of N, of S, other ghosts
    int upd[2] = {}, ofn[2] = {}, ofs[2] = {}, odd[2] = {};
    bool whole = true;   // every inner cell is updated
    for (int r = 0; r < R; r++) {
        uint32_t w = 0;
        for (int q = 0; q < 2; q++) {
            const int lx = strip * R + r, ly = 2 * m + q;
            const uint32_t k = code(lx, ly), g = k >> K_GHOST;
            const bool border = lx < 1 || lx > ex - 2 || ly < 1 || ly > ey - 2;
            whole = whole && (border || m >= hy || (k & K_UPD));
            upd[q] += k & K_UPD;
            ofn[q] += g == C_GN;
            ofs[q] += g == C_GS;
            odd[q] += g != 0 && g != C_GN && g != C_GS;
            w |= k << (16 * q);
        }
        dst[r * LW] = w;
    }
    uint32_t lane = 0;
    for (int q = 0; q < 2; q++) {
        if (ofn[q] > upd[q] + ofs[q] + odd[q]) lane |= q ? G_1N : G_0N;
        if (ofs[q] > upd[q] + ofn[q] + odd[q]) lane |= q ? G_1S : G_0S;
    }
    dst[R * LW] = lane;
    TbWave wv{};
    for (int r = 0; r < R; r++) {
        const uint32_t w = dst[r * LW];
        bool special = false, rest = false;
        for (int q = 0; q < 2; q++) {
            const uint32_t k = (w >> (16 * q)) & 0xffffu, g = k >> K_GHOST;
            const int lx = strip * R + r, ly = 2 * m + q;
            const bool border = lx < 1 || lx > ex - 2 || ly < 1 || ly > ey - 2;
            const uint32_t f = flag(t.rx0 + lx, t.ry0 + ly);
            const bool fluid = f != 0xffffu && (f & F_FLUID) && !border && m < hy;
            const uint32_t mine = (lane & (q ? G_1N : G_0N)) ? C_GN
                                  : (lane & (q ? G_1S : G_0S)) ? C_GS : 0u;
            // a fluid cell that is not updated or that the lane's word would
            // replace, or a ghost that it does not give
            special = special || (fluid && (!(k & K_UPD) || mine != 0)) || (g != 0 && g != mine);
            rest = rest || (k & K_REST);
        }
        wv.special |= __ballot(special) ? 1u << r : 0;
        wv.rest |= __ballot(rest) ? 1u << r : 0;
    }
    for (uint32_t b : {G_0S, G_1N, G_0N, G_1S})
        if (__ballot((lane & b) != 0)) wv.form |= b;
    if (__ballot(!whole)) wv.form |= TBW_CODED;
    if (m == 0) waves[at] = wv;
}

// After a blocked solve: channels whose latest p is in the second buffer
// copy it back (what arms the next one sets pbuf to 0).
__global__ void __launch_bounds__(TILE_THREADS)
k_pbuf_fix(const ChanDesc* __restrict__ cd, const ChanState* __restrict__ cs,
           const stm::Tile* __restrict__ tiles, const double* __restrict__ pb,
           double* __restrict__ pa)
{
    const stm::Tile t = tiles[blockIdx.x];
    if (!cs[t.chan].pbuf) return;
    const ChanDesc& d = cd[t.chan];
    const int x = t.x0 + threadIdx.y, y = t.y0 + threadIdx.x;
    if (x >= d.nx || y >= d.ny) return;
    const int64_t i = d.off + x * (int64_t)d.pitch + y;
    pa[i] = pb[i];
}

// ---------------------------------------------------------------- variants

// Wide tiles of ten rows a strip suit grids of several rounds of workgroups;
// the others are faster where a launch is one round (us per launch: 133 x 69
// cells, K = 4: 32 x 128 regions 7.9, 48 x 128 8.8, 80 x 128 12.5; 1026 x 1026,
// K = 6: 72 x 128 13.9, 80 x 128 14.5, 96 x 96 16.9; K = 8: 96 x 128 17.7, 80 x
// 128 18.2, but at 4002 x 3002 178 and 136).
//
// (index, K sweeps per launch, R rows per strip, HY pairs per row, NS strips)
// loaded region (NS*R) x (2*HY); output tile (NS*R - 2H) x (2*HY - 2H) with
// H = 2K + 2; workgroup NS * 64 threads.
#define STM_TB_VARIANTS(V)   \
    V(0, 1, 4, 64, 8)        \
    V(1, 2, 4, 64, 8)        \
    V(2, 4, 6, 64, 8)        \
    V(3, 4, 4, 64, 8)        \
    V(4, 4, 10, 64, 8)       \
    V(5, 6, 10, 64, 8)       \
    V(6, 8, 10, 64, 8)       \
    V(7, 6, 6, 64, 12)       \
    V(8, 8, 6, 64, 16)       \
    V(9, 6, 6, 48, 16)

#define V_ENTRY(i, K, R, HY, NS)                                                          \
    {K, NS * R - 2 * tb_halo(K), 2 * HY - 2 * tb_halo(K), NS * R, 2 * HY,                 \
     NS * LW, R},
const TbVariant TB_VARIANTS[] = {STM_TB_VARIANTS(V_ENTRY)};
#undef V_ENTRY
const int N_TB_VARIANTS = sizeof(TB_VARIANTS) / sizeof(TB_VARIANTS[0]);
#define V_CHECK(i, K, R, HY, NS) \
    static_assert(NS * R > 2 * tb_halo(K) && 2 * HY > 2 * tb_halo(K), "tile smaller than its halo");
STM_TB_VARIANTS(V_CHECK)
#undef V_CHECK

void launch_rb_tb(hipStream_t st, int variant, int ntb, const ChanDesc* cd, ChanState* cs,
                  const TbTile* tiles, const TbWave* waves, const uint32_t* words,
                  const double* rhs, double* pa, double* pb, const double* part_prev,
                  double* part_cur, int32_t* active, int L, int mode) {
#define V_CASE(i, K, R, HY, NS)                                                              \
    case i:                                                                                  \
        k_rb_strip<R, HY, NS><<<ntb, NS * LW, 0, st>>>(                                        \
            cd, cs, tiles, waves, words, rhs, pa, pb, part_prev, part_cur, active, K, L,     \
            mode);                                                                           \
        break;
    switch (variant) {
        STM_TB_VARIANTS(V_CASE)
    default: break;
    }
#undef V_CASE
}

void launch_rb_codes(hipStream_t st, int variant, int ntb, const TbTile* tiles,
                     const uint8_t* flags, TbWave* waves, uint32_t* words) {
    const TbVariant& v = TB_VARIANTS[variant];
    k_rb_codes<<<ntb, v.nt, 0, st>>>(tiles, flags, v.rows, v.ey / 2, v.ex,
                                     waves, words);
}

void launch_pbuf_fix(hipStream_t st, int ntiles, const ChanDesc* cd, const ChanState* cs,
                     const stm::Tile* tiles, const double* pb, double* pa) {
    k_pbuf_fix<<<ntiles, dim3(TILE_Y, TILE_X), 0, st>>>(cd, cs, tiles, pb, pa);
}

}  // namespace stm
