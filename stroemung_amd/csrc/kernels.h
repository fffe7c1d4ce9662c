// Host-side launchers of the gfx950 kernels (one translation unit per group).
#pragma once
#include <hip/hip_runtime.h>

#include "stm_internal.h"

namespace stm {

// kernels_step.hip
void launch_bc_velocity(hipStream_t, int nbtot, const BEntry*, double2* restore, double* u,
                        double* v, int nchan, const ChanDesc*, ChanState*);
void launch_fg(hipStream_t, int ntiles, const ChanDesc*, const ChanState*, const Tile*,
               const uint8_t* flags, const double* u, const double* v, double* f, double* g);
void launch_rhs(hipStream_t, int ntiles, const ChanDesc*, const ChanState*, const Tile*,
                const double* f, const double* g, double* rhs);
// launch_fg then launch_rhs in one pass (the same bits)
void launch_fg_rhs(hipStream_t, int ntiles, const ChanDesc*, const ChanState*, const Tile*,
                   const uint8_t* flags, const double* u, const double* v, double* f, double* g,
                   double* rhs);
void launch_restore(hipStream_t, int nbtot, const BEntry*, const double2* restore, double* u,
                    double* v);
void launch_ranges(hipStream_t, int ntiles, int nchan, const ChanDesc*, ChanState*, const Tile*,
                   const uint8_t* flags, const double* u, const double* v, const double* p,
                   double* part, int want_pressure);
// ADAP_UV on the fluid cells fused with the ranges; after launch_restore
void launch_adap_ranges(hipStream_t, int ntiles, int nchan, const ChanDesc*, ChanState*,
                        const Tile*, const uint8_t* flags, const double* f, const double* g,
                        const double* p, double* u, double* v, double* part,
                        int want_pressure, int end_tick);
void launch_fill(hipStream_t, int64_t n, double* a, double val);
void launch_zero_cells(hipStream_t, int n, const int64_t* idx, double* u, double* v,
                       double* p);
// Rows of several fields of a channel against dense arrays (dense[f] holds the
// rows [x0, x0 + rows) of field f, y contiguous without padding).
struct FieldRows {
    double* dev[6];
    double* dense[6];
    int64_t off, pitch;
    int32_t x0, rows, ny;
};
void launch_rows(hipStream_t, const FieldRows&, int nfields, bool pack);
void launch_copy(hipStream_t, int64_t bytes, const double* src, double* dst);

// kernels_pressure.hip
void launch_ghost(hipStream_t, int nbtot, const BEntry*, const ChanState*, double* p, int colour,
                  int only_active);
// rhs_mean and the sum of (rhs - mean)^2 per channel (partials in slots 0, 1)
void launch_rhs_stats(hipStream_t, int ntiles, int nchan, const ChanDesc*, ChanState*,
                      const Tile*, const uint8_t* flags, const double* rhs, double* part);
// The same and launch_solve_begin in one launch, for channels of at most
// STATS_TILES tiles each: four for each of a workgroup's waves.  The four launches
// take 66 or 88 us of a solve without sweeps, as the host is quick or slow to
// launch, whatever the size; the one takes 58 to 79 (16 tiles), 65 to 77 (64), 78 to
// 80 (120), 83 to 86 (144) and 108 to 110 (256).
constexpr int STATS_TILES = 64;
void launch_solve_stats(hipStream_t, int nchan, const ChanDesc*, ChanState*, const Tile*,
                        const uint8_t* flags, const double* rhs, int32_t* active);
void launch_solve_begin(hipStream_t, int nchan, const ChanDesc*, ChanState*, const double* part,
                        int32_t* active);
void launch_initial_norm(hipStream_t, int nchan, const ChanDesc*, ChanState*, const double* rhs,
                         const double* p, double* scratch);
// Does launch_lex_solve begin a solve that the pipelined one takes too?  If it is
// expected to take at most `begin` sweeps (lex_begin): its limit, or what the channel's
// last solve took if that met the stopping rule.  Two for the LEX_EXACT solves after
// one in which the pipeline found values that its quotient is not right for, and did
// its sweeps twice (a pressure that falls off to nothing in a long channel: ticks of
// one sweep of 768 x 64 cells 1.6 times as long, of 768 x 256 2.1 times).
constexpr int LEX_EXACT = 16;
__host__ __device__ inline bool lex_few(int begin, int itermax, const ChanState& s) {
    const int e = s.sor_iters == 0 || s.exhausted || s.sor_iters > (uint32_t)itermax
                      ? itermax : (int)s.sor_iters;
    return e > 0 && e <= (s.lex_exact > 0 ? 2 : begin);
}
constexpr int LEX_LDS_CELLS = 4608;   // channels of up to so many cells are solved in LDS there
void launch_lex_solve(hipStream_t, int nchan, const ChanDesc*, ChanState*, const BEntry*,
                      const uint8_t* flags, const double* rhs, double* p, double* scratch);

// kernels_lex.hip: the lexicographic solve with several sweeps in flight
struct LexClass {
    int row;        // most rows (ring included) a channel of the class has
    int full;       // sweeps whose squares are kept at once
    int codes;      // bytes of a diagonal's codes
    int rows_lane;  // rows of a lane
};
extern const LexClass LEX_CLASSES[];
extern const int N_LEX_CLASSES;
int lex_class(int nx, int ny);
int lex_begin(int cls, int nx, int ny);
int64_t lex_work_doubles(int cls, int nx, int ny);   // scratch of one channel
// What the scratch of class `cls` holds where there is no cell (the rest zeroed before).
void launch_lex_init(hipStream_t, int cls, int nchan, const ChanDesc*, const int64_t* work_off,
                     double* work);
// The channels of class `cls`; work_off: each channel's element offset in work.
void launch_lex_pipe(hipStream_t, int cls, int nchan, const ChanDesc*, ChanState*,
                     const int64_t* work_off, const uint8_t* flags, const double* rhs, double* p,
                     double* work);

// kernels_rbtb.hip: temporally blocked red-black SOR
struct TbVariant {
    int k;          // sweeps per launch
    int oxm, oym;   // largest output tile away from a channel's edges
    int ex, ey;     // loaded region; the halo is (ex - oxm) / 2 = tb_halo(k)
    int nt;         // threads per workgroup
    int rows;       // rows per strip (a wave each)
};
extern const TbVariant TB_VARIANTS[];
extern const int N_TB_VARIANTS;
constexpr int tb_halo(int k) { return 2 * k + 2; }
// What a wave of a tile holds (k_rb_codes): masks of its rows, and its form.
struct TbWave {
    uint32_t special;   // rows whose half-sweeps take the cells' codes
    uint32_t rest;      // rows with output cells that no sweep changes
    uint32_t form;      // TBW_GHOSTS: ghosts its lanes' words give; TBW_CODED
    uint32_t pad;
};
static_assert(sizeof(TbWave) == 16, "one 16-byte scalar load per wave");
enum : uint32_t { TBW_GHOSTS = 15, TBW_CODED = 16 };   // CODED: not all inner cells are updated
// The waves' table has one entry per wave of every tile (by tile idx), the
// words' table (rows + 1) * 64 words for each of them.
void launch_rb_codes(hipStream_t, int variant, int ntb, const TbTile*, const uint8_t* flags,
                     TbWave* waves, uint32_t* words);
enum : int { TB_CHECK = 1 };   // mode: form the residual after the sweeps and stop on it
// Launch L of a blocked solve: reads the partials of launch L - 1 from
// part_prev, writes its own to part_cur (one double per tile).  The ghosts of
// the input are fresh.
void launch_rb_tb(hipStream_t, int variant, int ntb, const ChanDesc*, ChanState*, const TbTile*,
                  const TbWave* waves, const uint32_t* words, const double* rhs, double* pa,
                  double* pb, const double* part_prev, double* part_cur, int32_t* active, int L,
                  int mode);
void launch_pbuf_fix(hipStream_t, int ntiles, const ChanDesc*, const ChanState*,
                     const Tile*, const double* pb, double* pa);

// kernels_view.hip: the GUI image of one channel (npix = nx * ny pixels)
void launch_render(hipStream_t, const ChanDesc*, const ChanState*, int ch, int64_t npix,
                   const uint8_t* flags, const double* u, const double* v, const double* p,
                   int mode, uint32_t* rgba);
// The static image buffer of stm_render_static: RENDER_STATIC_PIXELS pixels of
// 4 B (16 MiB) per device, devices 0 .. RENDER_STATIC_DEVICES - 1.  init looks
// its device address up (the device must be current; once per device);
// buffer returns it, or null before init.
constexpr int64_t RENDER_STATIC_PIXELS = (int64_t)4 << 20;
constexpr int RENDER_STATIC_DEVICES = 64;
hipError_t render_static_init(int device);
uint32_t* render_static_buffer(int device);

// kernels_learn.hip: the FP64 side of the learned correction and of capture
void launch_learn_residual(hipStream_t, int ntiles, const ChanDesc*, const ChanState*,
                           const LearnChan*, int first, const Tile*, const uint8_t* flags,
                           const double* rhs, const double* p, double* res, double* part);
void launch_learn_check(hipStream_t, int nch, const ChanDesc*, ChanState*, LearnChan*,
                        const double* part, int first);
// pixel blocks of an H x W frame (the size of cpart per channel)
int learn_coarse_blocks(int H, int W);
void launch_learn_restrict(hipStream_t, int nch, const ChanDesc*, LearnChan*,
                           const uint8_t* flags, const double* res, int H, int W, int f,
                           float* rc, float* mc, double2* cpart, int save);
// running channels -> batch entries (map), channels -> entries (inv), count
void launch_learn_compact(hipStream_t, int nch, const LearnChan*, int32_t* map, int32_t* inv,
                          int32_t* live);
void launch_learn_pack(hipStream_t, int nch, const LearnChan*, const float* rc, const float* mc,
                       int H, int W, __bf16* a0, __bf16* dx, int slot0, int dcap,
                       const int32_t* map = nullptr, const int32_t* live = nullptr);
void launch_learn_prolong(hipStream_t, int ntiles, const ChanDesc*, const Tile*,
                          const LearnChan*, const uint8_t* flags, const float* y,
                          const float* mc, int H, int W, int f, const int32_t* inv, double* cf);
void launch_learn_dots(hipStream_t, int ntiles, const ChanDesc*, const Tile*, const LearnChan*,
                       const uint8_t* flags, const double* res, const double* cf, const double* p,
                       const double* prev, const double* prev2, double* part);
void launch_learn_alpha(hipStream_t, int nch, const ChanDesc*, LearnChan*, const double* part,
                        int step, int f, int first);
void launch_learn_apply(hipStream_t, int ntiles, const ChanDesc*, const Tile*, const LearnChan*,
                        const uint8_t* flags, const double* cf, double* p, double* prev,
                        double* prev2);
void launch_learn_arm(hipStream_t, int nch, const ChanDesc*, ChanState*, const LearnChan*,
                      int32_t* active, int budget);
void launch_learn_collect(hipStream_t, int nch, ChanState*, LearnChan*, int final_phase);
void launch_learn_phase_end(hipStream_t, int nch, ChanState*, LearnChan*, int launches);
void launch_learn_target(hipStream_t, int ntiles, int nch, const ChanDesc*, const Tile*,
                         LearnChan*, const uint8_t* flags, const double* p, const double* p0,
                         double* part, int H, int W, int f, float* dt, int slot0, int dcap,
                         int which);

// kernels_sync.hip: the cost of a resident blocked solver's waits (measurement)
constexpr int SYNC_THREADS = 768;
void launch_sync_tile(hipStream_t, int nwg, double* out, int step);
void launch_sync_hold(hipStream_t, int nwg, double* out, int64_t ticks);
// hipSuccess when nwg workgroups of both waiting kernels fit on the device at once
hipError_t sync_coresident(int nwg, int device);
hipError_t launch_sync_grid(hipStream_t, int nwg, double* out, int steps, int write);
hipError_t launch_sync_neighbours(hipStream_t, int side, double* out, unsigned* flags,
                                  int steps, int write, unsigned spin_limit, unsigned* err);

}  // namespace stm
