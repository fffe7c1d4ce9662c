// The reference's lexicographic SOR (src/simulation.rs:239-285) with many
// sweeps in flight, bit-exact.
//
// A sweep visits the interior cells x-major in place, so cell (x, y) reads the
// new W and N and the old E and S values: the anti-diagonals x + y = d, taken
// in increasing d, give exactly those reads.  One sweep is a chain of nx + ny
// dependent diagonals, and on one diagonal at a time a workgroup waits for
// latency with most lanes idle.  But sweep k + 1 may follow sweep k a few
// diagonals behind, so a workgroup runs NSLOT sweeps at once: slot s does
// sweeps s, s + NSLOT, ..., each LAG diagonals behind the slot before it.
//
// A slot is LW lanes; lane l owns the RPL rows y = RPL * l .. + RPL - 1 (ring
// rows included), and takes cell (d - y, y) of each of them on diagonal d:
// independent cells.  Everything a cell needs is in registers: W is the row's
// own last result, N the last result of the row above, E and S the row's own
// and the row below's value on the next diagonal before the sweep (a DPP shift
// where the row belongs to the next lane).  A slot hands its results to the
// next through a ring of four diagonals in LDS, so a step is one barrier.
// Slot 0's ring is filled from the solve's input (A) and later from the last
// slot's results (C, a round of steps behind); the batch's last sweep writes B.
// A ghost's pressure is the copy of its fluid neighbours before the sweep
// (src/grid/mod.rs:343-412); those are inputs of the two neighbouring
// diagonals, still in the ring.  So a cell's code is the place its input is
// read from, relative to its own: itself, or the neighbour a ghost copies --
// one LDS read and no selection; only a ghost of two neighbours reads twice.
//
// The stopping rule is tested after every sweep, so sweeps in flight are
// speculative: A stays as it was until the batch is accepted.  Two ways:
//   LIGHT  The squares of the residual are added in order, so the sum is at
//          least as large as any one of them (rounding is monotone): a sweep
//          in which one square alone reaches the bound has not met the rule.
//          A third of the diagonals are looked at; when every sweep of the
//          batch shows such a square, all of them count.  The norm the solve
//          returns, its last sweep's, is formed from the final field.
//   FULL   Every sweep leaves all its squares (T), the norms are summed in the
//          reference's order and tested one after another; if sweep r of the
//          batch meets the rule, the batch is repeated from A with r + 1 sweeps.
// A solve starts LIGHT when the channel's last one ran to its limit (or there
// was none) and goes on FULL from the first batch that cannot be shown; batch
// lengths start at the last solve's and double, so little is swept for nothing.
//
// Fields are kept diagonal-major (row d + LEX_PAD of ROW = LW * RPL values,
// entry y), so a diagonal is one contiguous access.  LEX_PAD rows before the
// first and after the last diagonal hold no cells: they are 0 and their own
// inputs, and a slot whose diagonal is outside the grid passes zeros on.
//
// What bounds it: the diagonals of one sweep, one after another.  A step of one
// diagonal takes 760 to 880 cycles, the two quotients and the sums of a cell (a
// dependent FP64 addition takes 4.6 cycles), the LDS round trip to the next slot
// and the barrier; no memory and no unit is busy.  With up to 32 sweeps in
// flight, three diagonals apart, a sweep costs a few steps instead of nx + ny.
// A solve of a hundred sweeps to its limit (LIGHT: a hundred tests, one norm
// formed): 102 x 22 cells 3.58 ms with one sweep at a time, 0.30 now; 402 x 82 cells
// 53.9 ms and 2.44 (a lag of four diagonals: 8% slower).  One that meets the rule at
// the hundredth (FULL, after another such solve: a hundred norms, and what was swept
// beyond it again): 202 x 62 cells 19.8 and 2.67 (LIGHT 1.00), 402 x 82 54.5 and 8.4.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "stm_internal.h"

namespace stm {

namespace {

constexpr int LAG = 3;

// A cell's code, 16 bits: the byte offset of its input in its slot's ring (a
// multiple of 8 below 2^14, see Pipe), and in the other bits whether the sweep
// updates the cell, whether it is an interior cell, whether it is a ghost of
// two neighbours (whose vertical one the offset names), and whether the other
// one is its E neighbour (else W).
enum : uint32_t { C_UPD = 1, C_IN = 2, C_CORNER = 4, C_EAST = 0x8000, C_OFFSET = 0x3ff8 };

// Lane i takes lane i - 1's value (UP) or lane i + 1's: a DPP wave shift.
// The lane at the wave's end gets 0.0.
template <bool UP>
__device__ __forceinline__ double lane_shift(double v) {
    constexpr int CTRL = UP ? 0x138 : 0x130;
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// a / b, correctly rounded, for a divisor that stays the same: with y = RN(1/b)
// and yl = RN(1/b - y), q = a y + a yl is within one ulp of a / b, and one
// fused correction rounds it correctly (Markstein, IBM J. Res. Dev. 34 (1990);
// Brisebarre, Muller, Raina, IEEE Trans. Comput. 53 (2004)): four dependent
// operations instead of the general divide's two scalings, reciprocal, four
// Newton steps and fix-up.  It holds while nothing over- or underflows, which
// the bounds below secure (divisible), and while b's significand is not all
// ones; EXACT takes the general divide.  The sign is a's (b > 0), so a zero
// keeps its sign.
struct Divisor {
    double b, y, yl;
};
__device__ __forceinline__ Divisor make_divisor(double b) {
    Divisor v;
    v.b = b;
    v.y = 1.0 / b;
    v.yl = __builtin_fma(-b, v.y, 1.0) * v.y;
    return v;
}
__device__ __forceinline__ bool divisible(double b) {
    const uint64_t m = (uint64_t)__double_as_longlong(b) & 0xfffffffffffffull;
    return b >= 0x1p-30 && b <= 0x1p30 && m != 0xfffffffffffffull;
}
template <bool EXACT>
__device__ __forceinline__ double quotient(double a, const Divisor& v) {
    if constexpr (EXACT) return a / v.b;
    double q = __builtin_fma(a, v.y, a * v.yl);
    q = __builtin_fma(__builtin_fma(-v.b, q, a), v.y, q);
    return __hiloint2double((__double2hiint(q) & 0x7fffffff) |
                                (__double2hiint(a) & (int)0x80000000), __double2loint(q));
}
// A nonzero pressure (or right-hand side) below 2^-840 sends its batch to the
// general divide.  Without one every sum and difference of two pressures is a
// multiple of 2^-893, so no dividend but 0 is below that and no product or
// remainder of the quotient is subnormal; and a result of the update is 0 or
// at least 2^-1019 (omega in 2^-10 .. 2^10), so the upper word alone tells a
// tiny one from 0: `tiny_word` is below TINY_WORD for tiny results only.
// Towards infinity the quotient is right until something overflows; then it is
// NaN where the divide may be infinite, and a pressure that is not finite
// stays so (it is tested at the end of a batch, and so are the norms).
__device__ __forceinline__ bool tiny(double p) { return (fabs(p) < 0x1p-840) & (p != 0.0); }
constexpr uint32_t TINY_WORD = ((uint32_t)(1023 - 840) << 21) - 1u;
__device__ __forceinline__ uint32_t tiny_word(double p) {
    return ((uint32_t)__double2hiint(p) << 1) - 1u;
}
__device__ __forceinline__ bool finite(double p) { return fabs(p) < __builtin_inf(); }

// A lane's RPL values, and its codes.
typedef double double2u __attribute__((ext_vector_type(2), aligned(8)));
template <int RPL>
__device__ __forceinline__ void load_row(const void* p, double (&v)[RPL]) {
    const double* q = static_cast<const double*>(p);
#pragma unroll
    for (int i = 0; i + 1 < RPL; i += 2) {
        const double2u t = *reinterpret_cast<const double2u*>(q + i);
        v[i] = t.x;
        v[i + 1] = t.y;
    }
    if constexpr (RPL % 2 != 0) v[RPL - 1] = q[RPL - 1];
}
template <int RPL>
__device__ __forceinline__ void store_row(void* p, const double (&v)[RPL]) {
    double* q = static_cast<double*>(p);
#pragma unroll
    for (int i = 0; i + 1 < RPL; i += 2)
        *reinterpret_cast<double2u*>(q + i) = double2u{v[i], v[i + 1]};
    if constexpr (RPL % 2 != 0) q[RPL - 1] = v[RPL - 1];
}
constexpr int code_words(int rpl) { return rpl <= 2 ? 1 : rpl <= 4 ? 2 : 4; }
template <int RPL>
struct Codes {
    uint32_t w[code_words(RPL)];
    __device__ __forceinline__ uint32_t raw(int i) const { return w[i / 2] >> (16 * (i & 1)); }
    __device__ __forceinline__ bool is(int i, uint32_t bit) const {
        return (w[i / 2] & (bit << (16 * (i & 1)))) != 0;
    }
};
template <int RPL>
__device__ __forceinline__ Codes<RPL> load_codes(const void* p) {
    Codes<RPL> c;
    if constexpr (code_words(RPL) == 1) {
        c.w[0] = *static_cast<const uint32_t*>(p);
    } else if constexpr (code_words(RPL) == 2) {
        const uint2 t = *static_cast<const uint2*>(p);
        c.w[0] = t.x;
        c.w[1] = t.y;
    } else {
        const uint4 t = *static_cast<const uint4*>(p);
        c.w[0] = t.x;
        c.w[1] = t.y;
        c.w[2] = t.z;
        c.w[3] = t.w;
    }
    return c;
}

// Sum of acc and t of the row's lanes 0 .. 15, added one after another in that
// order by every lane of the row of 16 (a broadcast within the row and a fused
// multiply by one, which rounds as the addition does).
__device__ __forceinline__ double add_row(double acc, double t) {
#define STM_ADD_LANE(k) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
    asm volatile("s_nop 1\n\t"
                 STM_ADD_LANE(0) STM_ADD_LANE(1) STM_ADD_LANE(2) STM_ADD_LANE(3)
                 STM_ADD_LANE(4) STM_ADD_LANE(5) STM_ADD_LANE(6) STM_ADD_LANE(7)
                 STM_ADD_LANE(8) STM_ADD_LANE(9) STM_ADD_LANE(10) STM_ADD_LANE(11)
                 STM_ADD_LANE(12) STM_ADD_LANE(13) STM_ADD_LANE(14) STM_ADD_LANE(15)
                 : "+v"(acc) : "v"(t), "v"(1.0));
#undef STM_ADD_LANE
    return acc;
}

// One workgroup's view of its channel: its buffers as byte offsets from `base`
// (32 bits: lex_class keeps a channel's scratch below 4 GB).
struct LexWork {
    char* base;
    uint32_t a, b, c, rhs, t, codes;   // codes: code_words per lane, the others 8 bytes per entry
    uint32_t bytes;           // of one diagonal-major field
    int dmax;                 // the last diagonal, nx + ny - 2
    int ny;
    double omw, mid;
    Divisor dx2, dy2;
};

enum : int { LIGHT = 0, FULL = 1, FULL_DIV = 2 };   // FULL_DIV: FULL with the general divide

template <int LW, int RPL, int NSLOT, int TS>
struct Pipe {
    static constexpr int ROW = LW * RPL, NT = LW * NSLOT;
    static constexpr uint32_t ROWB = ROW * 8, ROWC = LW * 4 * code_words(RPL);   // bytes of a row
    static constexpr int Q = 3;              // steps of a group; loads are a group ahead
    static_assert(LAG == Q && TS <= NSLOT, "slots change sweeps between groups");
    // rows of the pads a slot reads and writes: -3 - 6 - 1 and up to
    // -3 + 3 * last() + 2 + 3 <= dmax + 8
    static_assert(LEX_PAD >= 10, "pads");

    // A slot's ring: four diagonals of ROWP places (a power of two).  In step
    // e the slot before it writes place e & 3; diagonals d, d + 1, d + 2 are
    // the results of its steps e - 3, e - 2, e - 1.
    static constexpr uint32_t pow2(uint32_t n) { return n <= 1 ? 1 : 2 * pow2((n + 1) / 2); }
    static constexpr uint32_t ROWP = pow2(ROW) * 8, RINGB = 4 * ROWP;        // bytes
    static constexpr uint32_t SHARED = (NSLOT + 1) * RINGB / 8;              // doubles
    static_assert(RINGB <= 0x4000, "offsets of codes");
    // The code of cell (x, y) with flag f: the offset is relative to the
    // lane's first row on diagonal d, the cell being on d + 1.
    __device__ static __forceinline__ uint32_t code(uint8_t f, int y, bool inner) {
        int dd = 1, dy = 0;
        uint32_t c = inner ? C_IN : 0u;
        if (flag_fluid(f)) {
            if (inner) c |= C_UPD;
        } else {
            const uint8_t e = flag_edge(f);
            if (e == E_N || e == E_NE || e == E_NW) { dd = 0; dy = -1; }
            else if (e == E_S || e == E_SE || e == E_SW) { dd = 2; dy = 1; }
            else if (e == E_E) dd = 2;
            else if (e == E_W) dd = 0;
            if (e == E_NE || e == E_SE) c |= C_CORNER | C_EAST;
            if (e == E_NW || e == E_SW) c |= C_CORNER;
        }
        return c | ((uint32_t)(dd * (int)ROWP + (y % RPL + dy) * 8) & (RINGB - 8));
    }

    // Where the code of row y of a diagonal (a row of the codes) is.  (A lane of
    // three rows leaves its fourth code unread.)
    __device__ static __forceinline__ uint16_t* code_place(char* codes, uint32_t row, uint32_t y) {
        return reinterpret_cast<uint16_t*>(codes) + row * (ROWC / 2) +
               y / RPL * 2 * code_words(RPL) + y % RPL;
    }

    // Groups of a sweep, and of a round: a slot starts its next sweep a round
    // after this one.  Slot 0's ring takes row q of C in step q of its round,
    // loaded a group earlier; the last slot stores row q in step 3 NSLOT + q of
    // the round before: at least 12 steps earlier.  A wave's global loads and
    // stores complete in order, and in every step it uses loads issued a group
    // (3 steps) before, so that store has long been complete.
    __device__ static __forceinline__ int last(const LexWork& w) { return (w.dmax + 4 + Q - 1) / Q; }
    __device__ static __forceinline__ int round(const LexWork& w) { return max(last(w) + 1, NSLOT + 5); }

    struct Result {
        int mode;
        bool bad;      // a pressure the fixed quotient is not right for
        bool open;     // LIGHT: a sweep that may have met the stopping rule
    };

    // Sweeps 0 .. n - 1 from A; the last one's result in B.  LIGHT: sweeps
    // below `need` are shown not to have met the rule by a square of `bound`
    // or more.  FULL: n <= TS, the squares of sweep k in T, field k.
    template <int MODE>
    __device__ static __forceinline__ Result sweeps(const LexWork& w, int n, int need,
                                                    double bound, double* ring) {
        constexpr bool EXACT = MODE == FULL_DIV;
        // (a wave's slot is uniform when a slot is a wave)
        const int slot = LW == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / LW)
                                  : threadIdx.x / LW;
        const int y0 = (threadIdx.x % LW) * RPL;
        const int glast = last(w), ground = round(w);
        const int groups = (n - 1) / NSLOT * ground + (n - 1) % NSLOT + glast;
        Result res{MODE, false, false};
        for (uint32_t i = threadIdx.x; i < SHARED; i += NT) ring[i] = 0.0;
        __syncthreads();
        // waves without a slot of the batch only keep the barriers
        if ((int)(threadIdx.x & ~63u) / LW >= n) {
            for (int e = 0; e < groups * Q; e++) asm volatile("s_barrier" ::: "memory");
            return res;
        }
        const bool rows_in = y0 < w.ny;      // lanes below the last row: zeros, inputs themselves
        const bool first = slot == 0;
        const uint32_t yb = (uint32_t)y0 * 8u;
        // this lane's first row in its slot's ring, and in the next slot's
        char* const lds = reinterpret_cast<char*>(ring);
        const uint32_t ring_in = (uint32_t)slot * RINGB, ring_out = ring_in + RINGB + yb;
        // the slot's group g of its sweep k: diagonals d = -3 + 3 g .. + 2.
        // Before its first and after its last group a slot is on the pads.
        int g = -slot, k = slot;
        auto row0 = [&](int gg) -> uint32_t {   // row -3 + 3 gg of a field
            return (uint32_t)(min(max(gg, -2), glast) * Q + (LEX_PAD - 3));
        };
        // this lane's codes of row r
        auto code_at = [&](uint32_t r) -> uint32_t {
            return w.codes + r * ROWC + (threadIdx.x % LW) * (4u * code_words(RPL));
        };
        // what slot 0's ring takes in sweep kk: rows from d + 3 on
        auto from = [&](int kk, uint32_t r0) -> uint32_t {
            return (kk == 0 ? w.a : w.c) + (r0 + 3) * ROWB + yb;
        };
        const bool wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x) < 64;   // holds slot 0
        double in0[RPL];                     // the input of diagonal d (ghosts formed)
        double o1[RPL], dxp[RPL], dvp[RPL], rp[RPL];   // diagonal d - 1: result, its differences
                                                       // to W and N, rhs
        Codes<RPL> code0{}, codep{};         // codes of diagonals d, d - 1
        double aq[Q][RPL], rq[Q][RPL];       // slot 0's input of d + 3, rhs of d
        Codes<RPL> cq[Q];                    // codes of d + 1
#pragma unroll
        for (int i = 0; i < RPL; i++) in0[i] = o1[i] = dxp[i] = dvp[i] = rp[i] = 0.0;
        {
            const uint32_t r0 = row0(g), f0 = from(k, r0);
#pragma unroll
            for (int j = 0; j < Q; j++) {
                if (wave0) load_row<RPL>(w.base + (f0 + j * ROWB), aq[j]);
                load_row<RPL>(w.base + (w.rhs + r0 * ROWB + yb + j * ROWB), rq[j]);
                cq[j] = load_codes<RPL>(w.base + (code_at(r0) + (j + 1) * ROWC));
            }
        }
        uint32_t cur = ROWP;                 // byte offset of diagonal d in the rings: (e + 1) & 3
        uint32_t small = ~0u;                // the least tiny_word
        bool shown = false;                  // LIGHT: this lane's square for sweep k
        auto slot_any = [&](bool v) -> bool {   // some lane of the slot
            const uint64_t m = __ballot(v);
            const int base = (threadIdx.x & 63) / LW * LW;
            return LW == 64 ? m != 0 : ((m >> base) & ((1ull << (LW & 63)) - 1ull)) != 0;
        };
        for (int e = 0; e < groups; e++) {
            const uint32_t r0 = row0(g);
            int gn = g + 1, kn = k;
            if (gn == ground) {
                gn = 0;
                kn = k + NSLOT;
            }
            const uint32_t rn0 = row0(gn), fn0 = from(kn, rn0);
            const bool final_sweep = k == n - 1;
            const bool keep = rows_in & (final_sweep | ((slot == NSLOT - 1) & (k < n)));
            const uint32_t ob = (final_sweep ? w.b : w.c) + r0 * ROWB + yb;
            const uint32_t tb = w.t + (uint32_t)min(slot, TS - 1) * w.bytes + (r0 - 1) * ROWB + yb;
            const uint32_t rb = w.rhs + rn0 * ROWB + yb, cb = code_at(rn0) + ROWC;
            const bool keep_t = rows_in & (k < n);
#pragma unroll
            for (int j = 0; j < Q; j++) {
                // the inputs of diagonal d + 1, ghosts' from their neighbours
                double in1[RPL];
                const Codes<RPL> code1 = cq[j];
                const uint32_t at = yb + cur;
#pragma unroll
                for (int i = 0; i < RPL; i++)
                    in1[i] = *reinterpret_cast<const double*>(
                        lds + (((code1.raw(i) + at) & (RINGB - 8)) | ring_in));
                // slot 0's ring takes diagonal d + 3
                if (wave0 && first) store_row<RPL>(lds + (((cur + 3 * ROWP) & (RINGB - 8)) + yb), aq[j]);
                bool corner = false;
#pragma unroll
                for (int i = 0; i < RPL; i++) corner |= code1.is(i, C_CORNER);
                if (__ballot(corner) != 0) {   // uniform
#pragma unroll
                    for (int i = 0; i < RPL; i++) {
                        const uint32_t q = at + (code1.is(i, C_EAST) ? 2 * ROWP : 0u) + i * 8;
                        const double h = *reinterpret_cast<const double*>(
                            lds + ((q & (RINGB - 8)) | ring_in));
                        in1[i] = code1.is(i, C_CORNER) ? (in1[i] + h) * 0.5 : in1[i];
                    }
                }
                // the update of diagonal d (src/simulation.rs:266-270)
                double o[RPL], nb[RPL];
                {
                    const double un = lane_shift<true>(o1[RPL - 1]);
                    const double dn = lane_shift<false>(in1[0]);
#pragma unroll
                    for (int i = 0; i < RPL; i++) {
                        nb[i] = i > 0 ? o1[i > 0 ? i - 1 : 0] : un;
                        const double s = i + 1 < RPL ? in1[i + 1 < RPL ? i + 1 : i] : dn;
                        const double lap = quotient<EXACT>(in1[i] + o1[i], w.dx2) +
                                           quotient<EXACT>(s + nb[i], w.dy2);
                        const double v = (w.omw * in0[i]) + (w.mid * (lap - rq[j][i]));
                        o[i] = code0.is(i, C_UPD) ? v : in0[i];
                        if constexpr (!EXACT) small = min(small, tiny_word(o[i]));
                    }
                }
                store_row<RPL>(lds + (((cur + 3 * ROWP) & (RINGB - 8)) + ring_out), o);
                // the residual of diagonal d - 1 (src/math.rs:176-186): c - W of
                // a cell is E - c of the cell before it, c - N is S - c of the
                // cell above
                if (MODE != LIGHT || j == 0 || j == Q - 1) {
                    double dx[RPL], dv[RPL];
#pragma unroll
                    for (int i = 0; i < RPL; i++) {
                        dx[i] = o[i] - o1[i];
                        dv[i] = o[i] - nb[i];
                    }
                    if (MODE != LIGHT || j == 0) {
                        double tt[RPL];
                        const double dn = lane_shift<false>(dv[0]);
#pragma unroll
                        for (int i = 0; i < RPL; i++) {
                            const double sc = i + 1 < RPL ? dv[i + 1 < RPL ? i + 1 : i] : dn;
                            const double r = (quotient<EXACT>(dx[i] - dxp[i], w.dx2) +
                                              quotient<EXACT>(sc - dvp[i], w.dy2)) - rp[i];
                            tt[i] = r * r;
                            if (MODE == LIGHT)
                                shown |= codep.is(i, C_IN) & (tt[i] >= bound);
                        }
                        if (MODE != LIGHT && keep_t)
                            store_row<RPL>(w.base + (tb + j * ROWB), tt);
                    }
#pragma unroll
                    for (int i = 0; i < RPL; i++) {
                        dxp[i] = dx[i];
                        dvp[i] = dv[i];
                        rp[i] = rq[j][i];
                    }
                }
                if (keep) {
                    store_row<RPL>(w.base + (ob + j * ROWB), o);
                    if (!EXACT && final_sweep)
#pragma unroll
                        for (int i = 0; i < RPL; i++) res.bad |= !finite(o[i]);
                }
                // on to the next diagonal
#pragma unroll
                for (int i = 0; i < RPL; i++) {
                    in0[i] = in1[i];
                    o1[i] = o[i];
                }
                codep = code0;
                code0 = code1;
                cur = (cur + ROWP) & (RINGB - 8);
                if (wave0) load_row<RPL>(w.base + (fn0 + j * ROWB), aq[j]);
                load_row<RPL>(w.base + (rb + j * ROWB), rq[j]);
                cq[j] = load_codes<RPL>(w.base + (cb + j * ROWC));
                // the ring's writes are done before the others read them; global
                // loads and stores stay in flight
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
            if (MODE == LIGHT && __ballot(kn != k) != 0) {   // a slot of the wave ends its sweep
                const bool any = slot_any(shown);
                res.open |= (kn != k) & (k < need) & !any;
                shown = shown & (kn == k);
            }
            g = gn;
            k = kn;
        }
        res.bad |= small < TINY_WORD;
        if (MODE == LIGHT) {
            const bool any = slot_any(shown);
            // a slot that has gone round waits for a sweep past the batch's last
            res.open |= (k < need) & !any;
        }
        return res;
    }

    // The sum from 0.0 of a diagonal-major field's squares over the interior,
    // x-major, by a row of 16 lanes: U * 16 terms are gathered (that many
    // ahead) and added one by one.  Places past the end add +0.0, which
    // changes no sum of squares.
    static constexpr int U = 8, CHUNK = U * 16;
    __device__ static __forceinline__ double norm_sum(const char* t, int nxi, int nyi) {
        const int lane = threadIdx.x & 15;
        const int n = nxi * nyi;
        const int sx = CHUNK / nyi, sy = CHUNK - sx * nyi;
        int x[U], y[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = u * 16 + lane;
            x[u] = 1 + k / nyi;
            y[u] = 1 + k - (k / nyi) * nyi;
        }
        auto gather = [&]() {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t at = (uint32_t)(min(x[u], nxi) + y[u] + LEX_PAD) * ROWB + y[u] * 8u;
                const double q = *reinterpret_cast<const double*>(t + at);
                v[u] = x[u] <= nxi ? q : 0.0;
                x[u] += sx;
                y[u] += sy;
                if (y[u] > nyi) {
                    y[u] -= nyi;
                    x[u]++;
                }
            }
        };
        double acc = 0.0;
        gather();
        for (int k = 0; k < n; k += CHUNK) {
            double c[U];
#pragma unroll
            for (int u = 0; u < U; u++) c[u] = v[u];
            gather();
#pragma unroll
            for (int u = 0; u < U; u++) acc = add_row(acc, c[u]);
        }
        return acc;
    }

    // The same for n squares in the norm's order in memory (T, which is longer
    // than they are by more than two chunks).
    __device__ static __forceinline__ double norm_sum_linear(const char* t, int n) {
        const double* q = reinterpret_cast<const double*>(t) + (threadIdx.x & 15);
        double v[U], acc = 0.0;
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = q[u * 16];
        int k = 0;
        for (; k + CHUNK <= n; k += CHUNK) {
            double c[U];
            q += CHUNK;
#pragma unroll
            for (int u = 0; u < U; u++) c[u] = v[u];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = q[u * 16];
            __builtin_amdgcn_sched_barrier(0);   // the loads go first
#pragma unroll
            for (int u = 0; u < U; u++) acc = add_row(acc, c[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            acc = add_row(acc, k + u * 16 + (int)(threadIdx.x & 15) < n ? v[u] : 0.0);
        return acc;
    }

    // The squares of the residual of the field at `p` (every interior cell;
    // the general divide) to the start of T in the norm's order.
    __device__ static __forceinline__ void squares(const LexWork& w, uint32_t p, int nxi, int nyi) {
        const int n = (nxi + nyi - 1) * ROW;   // diagonals 2 .. nxi + nyi
        for (int k = threadIdx.x; k < n; k += NT) {
            const int y = k % ROW, x = 2 + k / ROW - y;
            if (x < 1 || x > nxi || y < 1 || y > nyi) continue;
            const uint32_t at = (uint32_t)(x + y + LEX_PAD) * ROWB + y * 8u;
            const double* q = reinterpret_cast<const double*>(w.base + (p + at));
            const double c = q[0];
            const double a = ((q[ROW] - c) - (c - q[-ROW])) / w.dx2.b;
            const double b = ((q[ROW + 1] - c) - (c - q[-ROW - 1])) / w.dy2.b;
            const double r = (a + b) - *reinterpret_cast<const double*>(w.base + (w.rhs + at));
            *reinterpret_cast<double*>(w.base + (w.t + (uint32_t)((x - 1) * nyi + y - 1) * 8u)) = r * r;
        }
    }
};

}  // namespace

// Class of a channel: which instance solves it; -1 (k_lex_solve) with more
// rows than a wave can own, or beyond the 32-bit offsets.
int lex_class(int nx, int ny) {
    for (int c = 0; c < N_LEX_CLASSES; c++)
        if (ny <= LEX_CLASSES[c].row) return lex_work_doubles(c, nx, ny) < (1ll << 29) ? c : -1;
    return -1;
}

// The most sweeps of a solve that k_lex_solve begins (0: none), which has no fields
// to set up and goes through a diagonal with the whole workgroup.  One sweep in LDS is
// always the faster there.  In the fields it is while they are small where a lane here
// has four rows, whose step is the longer one: a tick of one sweep there over here, 64
// rows of 96, 192 and 384 cells 0.88, 0.91 and 1.00, 128 of 48, 96 and 192 0.87, 0.93
// and 1.01, 256 of 24, 48 and 192 0.82, 0.85 and 0.96 (224 rows 1.06); with three rows
// 0.97 to 1.25.  With eight rows it is for two sweeps as well: ticks of one 0.28 to
// 0.70; solves of 502 x 62 cells in one sweep 585 and 1055 us, in two 1049 and 1451,
// in three 1569 and 1548.
int lex_begin(int cls, int nx, int ny) {
    if (cls < 0) return 0;
    const int rows = LEX_CLASSES[cls].rows_lane;
    if (rows >= 8) return 2;
    return (int64_t)nx * ny <= (rows == 4 ? 3 : 1) * LEX_LDS_CELLS ? 1 : 0;
}

// A, B, C, rhs, the squares of the FULL sweeps, the codes.
int64_t lex_work_doubles(int cls, int nx, int ny) {
    if (cls < 0) return 0;
    const int64_t rows = (int64_t)nx + ny - 1 + 2 * LEX_PAD, cells = rows * LEX_CLASSES[cls].row;
    return cells * (4 + LEX_CLASSES[cls].full) + rows * LEX_CLASSES[cls].codes / 8;
}

constexpr int LIGHT_MOST = 256;   // sweeps of a LIGHT batch

// Entries of the scratch that are no cell: code of a cell that is its own input
// (the fields hold 0 from the allocation on).  Once, with the allocation.
template <int CLASS, int LW, int RPL, int NSLOT, int TS>
__global__ void __launch_bounds__(256)
k_lex_init(const ChanDesc* __restrict__ cd, const int64_t* __restrict__ work_off,
           double* __restrict__ work, uint32_t per)   // per: workgroups of a channel
{
    using P = Pipe<LW, RPL, NSLOT, TS>;
    const uint32_t c = blockIdx.x / per, part = blockIdx.x - c * per;
    const ChanDesc& d = cd[c];
    if (d.solver != SOLVER_LEX || d.lex_class != CLASS) return;
    const uint32_t cells = (uint32_t)(d.nx + d.ny - 1 + 2 * LEX_PAD) * P::ROW;
    char* codes = reinterpret_cast<char*>(work + work_off[c]) + (4 + TS) * (uint64_t)cells * 8;
    for (uint32_t k = part * 256 + threadIdx.x; k < cells; k += per * 256)
        *P::code_place(codes, k / P::ROW, k % P::ROW) =
            (uint16_t)P::code(make_flag(T_NOSLIP, E_NONE), (int)(k % P::ROW), false);
}

template <int CLASS, int LW, int RPL, int NSLOT, int TS>
__global__ void __launch_bounds__(LW * NSLOT)
k_lex_pipe(const ChanDesc* __restrict__ cd, ChanState* __restrict__ cs,
           const int64_t* __restrict__ work_off, const uint8_t* __restrict__ flags,
           const double* __restrict__ rhs, double* __restrict__ p, double* work)
{
    using P = Pipe<LW, RPL, NSLOT, TS>;
    constexpr int ROW = P::ROW, NT = P::NT;
    __shared__ __attribute__((aligned(16))) double ring[P::SHARED];
    __shared__ double snorm[TS];
    const ChanDesc d = cd[blockIdx.x];
    if (d.solver != SOLVER_LEX || d.lex_class != CLASS) return;
    ChanState& s = cs[blockIdx.x];
    const int begun = s.budget;    // sweeps that k_lex_solve has done
    if (begun < 0) return;         // it has ended the solve
    const int tid = threadIdx.x;
    if (d.itermax <= 0) {          // nothing to sweep: no need of the fields' copies
        if (tid == 0) {
            s.sor_iters = (uint32_t)d.itermax;
            s.norm2 = 0.0;
            s.exhausted = 1;
            s.active = 0;
        }
        return;
    }
    const int nxi = d.nx - 2, nyi = d.ny - 2;
    LexWork w;
    w.dmax = d.nx + d.ny - 2;
    w.ny = d.ny;
    w.omw = d.omw;
    w.mid = d.mid;
    w.dx2 = make_divisor(d.delx2);
    w.dy2 = make_divisor(d.dely2);
    const uint32_t cells = (uint32_t)(w.dmax + 1 + 2 * LEX_PAD) * ROW;
    w.bytes = cells * 8;
    w.base = reinterpret_cast<char*>(work + work_off[blockIdx.x]);
    w.a = 0;
    w.b = w.bytes;
    w.c = 2 * w.bytes;
    w.rhs = 3 * w.bytes;
    w.t = 4 * w.bytes;
    w.codes = (4 + TS) * w.bytes;

    // the fields, diagonal-major, cell by cell (entries that are no cell keep what
    // k_lex_init gave them: 0, and the code of a cell that is its own input; a
    // sweep stores there what it read).  All entries, a parallelogram of which a
    // 152 x 152 channel fills a quarter, took 92 us to set of 403 for a solve of
    // one sweep; its cells take 49 of 360.
    bool odd = !divisible(d.delx2) || !divisible(d.dely2) ||
               !(d.omega >= 0x1p-10 && d.omega <= 0x1p10);
    const uint32_t ny = (uint32_t)d.ny, ncell = (uint32_t)d.nx * ny;
#pragma unroll 8
    for (uint32_t k0 = tid; k0 < ncell; k0 += NT) {
        const uint32_t x = k0 / ny, y = k0 - x * ny, row = x + y + LEX_PAD;
        const int64_t g = d.off + x * (int64_t)d.pitch + y;
        const double pv = p[g], rv = rhs[g];
        const uint8_t f = flags[g];
        const uint32_t k = row * ROW + y;
        double* e = reinterpret_cast<double*>(w.base) + k;
        e[0] = pv;
        e[3 * (int64_t)cells] = rv;
        *P::code_place(w.base + w.codes, row, y) =
            (uint16_t)P::code(f, (int)y, x >= 1 && (int)x <= nxi && y >= 1 && (int)y <= nyi);
        odd |= tiny(pv) | !finite(pv) | tiny(rv);
    }
    __syncthreads();
    bool exact = __syncthreads_or(odd) != 0;

    const double init = s.init_norm2, fluid = d.fluid_cells;
    // a square of `bound` or more makes the norm neither < init nor < eps2
    // (the factor covers the roundings of this product and of the norm's division)
    const double bound = (init > d.eps2 ? init : d.eps2) * fluid * (1.0 + 0x1p-48);
    double norm2 = 0.0;
    int iters = d.itermax, exhausted = 1, done = begun;
    const int before = begun > 0 ? 0 : (int)min(s.sor_iters, (uint32_t)LIGHT_MOST);
    bool light = before == 0 || s.exhausted;
    int len = before > 0 ? before : NSLOT;
    int replay = 0;   // sweeps of the batch to be repeated, ending with the one that met the rule
    while (done < d.itermax) {
        const int most = light && !exact ? len : min(len, TS);
        const int n = replay > 0 ? replay : min(most, d.itermax - done);
        const bool end = done + n == d.itermax;
        // a single sweep's norm is the final field's: no need of T
        const bool lt = !exact && ((light && replay == 0) || n == 1), field = lt && (end || n == 1);
        typename P::Result r;
        if (lt) r = P::template sweeps<LIGHT>(w, n, field ? n - 1 : n, bound, ring);
        else if (!exact) r = P::template sweeps<FULL>(w, n, 0, 0.0, ring);
        else r = P::template sweeps<FULL_DIV>(w, n, 0, 0.0, ring);
        __syncthreads();
        exact = exact || __syncthreads_or(r.bad) != 0;
        const bool open = lt && __syncthreads_or(r.open) != 0;
        light = light && !open;
        if (open || (exact && r.mode != FULL_DIV)) continue;   // again from A
        if (field) {
            P::squares(w, w.b, nxi, nyi);
            __syncthreads();
        }
        int stop = -1;
        if (!lt || field) {
            // the first norm in T that meets the rule
            const int nt = lt ? 1 : n;
            if (tid / 16 < nt) {
                const char* t = w.base + (w.t + (tid / 16) * w.bytes);
                const double acc = lt ? P::norm_sum_linear(t, nxi * nyi) : P::norm_sum(t, nxi, nyi);
                if (tid % 16 == 0) snorm[tid / 16] = acc / fluid;
            }
            __syncthreads();
            for (int k = 0; k < nt && stop < 0; k++) {
                norm2 = snorm[k];
                if ((norm2 < init) || (norm2 < d.eps2)) stop = k;
            }
            __syncthreads();   // snorm is written again
            if (r.mode == FULL && !finite(norm2)) {   // an overflow the quotient may have made a NaN
                exact = true;
                continue;
            }
            if (stop >= 0 && stop + 1 < n && !lt) {
                replay = stop + 1;
                continue;
            }
        }
        const uint32_t old = w.a;
        w.a = w.b;
        w.b = old;
        done += n;
        len = min(2 * len, LIGHT_MOST);
        if (stop >= 0) {
            iters = done;
            exhausted = 0;
            break;
        }
    }
    for (int k = tid; k < d.nx * d.ny; k += NT) {
        const int x = k / d.ny, y = k - x * d.ny;
        p[d.off + x * (int64_t)d.pitch + y] = *reinterpret_cast<const double*>(
            w.base + (w.a + (uint32_t)(x + y + LEX_PAD) * P::ROWB + y * 8u));
    }
    if (tid == 0) {
        s.sor_iters = (uint32_t)iters;
        s.norm2 = norm2;
        s.exhausted = exhausted;
        s.lex_exact = exact ? LEX_EXACT : 0;
        s.active = 0;
    }
}

// (class, lanes per slot, rows per lane, slots, slots of a FULL batch): rows
// up to LW * RPL
// A workgroup is eight waves (four where a lane has eight rows and their
// registers): few lanes to a slot make many slots, few rows to a lane a short
// step.  A tick of 22 rows measured 374 us with 16 lanes of two rows and 408 with
// eight lanes of three; 82 rows 3.23 ms with 32 lanes of three and 4.0 before
// there was that class.
#define STM_LEX_CLASSES(V) \
    V(0, 16, 2, 32, 16)    \
    V(1, 16, 3, 32, 16)    \
    V(2, 16, 4, 32, 16)    \
    V(3, 32, 3, 16, 16)    \
    V(4, 32, 4, 16, 16)    \
    V(5, 64, 3, 8, 8)      \
    V(6, 64, 4, 8, 8)      \
    V(7, 64, 8, 4, 4)

#define L_ENTRY(c, LW, RPL, NSLOT, TS) {LW * RPL, TS, LW * 4 * code_words(RPL), RPL},
const LexClass LEX_CLASSES[] = {STM_LEX_CLASSES(L_ENTRY)};
#undef L_ENTRY
const int N_LEX_CLASSES = sizeof(LEX_CLASSES) / sizeof(LEX_CLASSES[0]);

void launch_lex_init(hipStream_t st, int cls, int nchan, const ChanDesc* cd,
                     const int64_t* work_off, double* work) {
    const uint32_t per = (uint32_t)std::max(1, std::min(16, 65536 / nchan));
#define L_CASE(c, LW, RPL, NSLOT, TS)                                                          \
    case c:                                                                                   \
        k_lex_init<c, LW, RPL, NSLOT, TS><<<per * (uint32_t)nchan, 256, 0, st>>>(cd, work_off, work, \
                                                                              per);           \
        break;
    switch (cls) {
        STM_LEX_CLASSES(L_CASE)
    default: break;
    }
#undef L_CASE
}
void launch_lex_pipe(hipStream_t st, int cls, int nchan, const ChanDesc* cd, ChanState* cs,
                     const int64_t* work_off, const uint8_t* flags, const double* rhs, double* p,
                     double* work) {
#define L_CASE(c, LW, RPL, NSLOT, TS)                                                             \
    case c:                                                                                   \
        k_lex_pipe<c, LW, RPL, NSLOT, TS><<<nchan, LW * NSLOT, 0, st>>>(cd, cs, work_off, flags, rhs, \
                                                                    p, work);                 \
        break;
    switch (cls) {
        STM_LEX_CLASSES(L_CASE)
    default: break;
    }
#undef L_CASE
}

}  // namespace stm
