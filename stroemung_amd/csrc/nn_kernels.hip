// gfx950 kernels of the pressure network: a U-Net of 3x3 convolutions in
// BF16 with FP32 accumulation on the matrix cores.
//
// Tensors are NHWC (channels contiguous), bf16, with channel counts that are
// multiples of 32.  A 3x3 convolution with padding 1 is an implicit GEMM:
//   forward      out[pix, co]  = sum_{tap, ci} in[pix + off(tap), ci] * w[co, tap, ci]
//   backward-in  gin[pix, ci]  = sum_{tap, co} gz[pix - off(tap), co] * w[co, tap, ci]
//                              = forward with w'[ci, 8 - tap, co] (rotated, transposed)
//   backward-w   dw[co, tap, ci] = sum_pix gz[pix, co] * in[pix + off(tap), ci]
// v_mfma_f32_16x16x32_bf16 operands (checked on the device): lane l holds row
// l % 16 of A and column l % 16 of B, each with k = 8 * (l / 16) + 0..7, and
// column l % 16, rows 4 * (l / 16) + 0..3 of the f32 result.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "nn_kernels.h"

namespace stm {
namespace nn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 load8(const bf16* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}
__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
    for (int i = 0; i < 8; i++) z[i] = (bf16)0.0f;
    return z;
}

// ------------------------------------------------------------ convolution

// Block: 256 threads = 4 waves in a 2 x 2 grid; block tile BM pixels x 64
// output channels, each wave (BM/2) x 32 as (BM/32) x 2 MFMA tiles.
// flags: 1 = add bias, 2 = ReLU.
template <int BM>
__global__ void __launch_bounds__(256)
k_conv3x3(const bf16* __restrict__ in, int cin, const bf16* __restrict__ w,
          const float* __restrict__ bias, bf16* __restrict__ out, float* __restrict__ out32,
          int cout, int nb, int H, int W, int flags, const int* __restrict__ live)
{
    constexpr int MT = BM / 32;          // M tiles per wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int npix = (live ? min(nb, *live) : nb) * H * W;
    if ((int)(blockIdx.x * BM) >= npix) return;   // the whole block is beyond the live images
    const int m_base = blockIdx.x * BM + wm * (BM / 2);
    const int n_base = blockIdx.y * 64 + wn * 32;
    if (n_base >= cout) return;          // 32-channel layers use half the tile (no barriers here)
    const int row = lane & 15, kq = (lane >> 4) * 8;

    // the pixels this lane loads for each M tile
    int pb[MT], ph[MT], pw[MT];
    bool pv[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int pix = m_base + t * 16 + row;
        pv[t] = pix < npix;
        const int pp = pv[t] ? pix : 0;
        pb[t] = pp / (H * W);
        const int r = pp - pb[t] * H * W;
        ph[t] = r / W;
        pw[t] = r - ph[t] * W;
    }
    f32x4 acc[MT][2];
#pragma unroll
    for (int t = 0; t < MT; t++)
        for (int u = 0; u < 2; u++) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int tap = 0; tap < 9; tap++) {
        const int dy = tap / 3 - 1, dx = tap % 3 - 1;
        const bf16* arow[MT];
        bool aok[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int hh = ph[t] + dy, ww = pw[t] + dx;
            aok[t] = pv[t] && hh >= 0 && hh < H && ww >= 0 && ww < W;
            arow[t] = in + ((int64_t)(pb[t] * H + (aok[t] ? hh : 0)) * W + (aok[t] ? ww : 0)) * cin;
        }
        const bf16* brow[2];
#pragma unroll
        for (int u = 0; u < 2; u++) brow[u] = w + ((int64_t)tap * cout + n_base + u * 16 + row) * 32 + kq;
        for (int c0 = 0; c0 < cin; c0 += 32) {
            bf16x8 a[MT], b[2];
#pragma unroll
            for (int t = 0; t < MT; t++) a[t] = aok[t] ? load8(arow[t] + c0 + kq) : zero8();
#pragma unroll
            for (int u = 0; u < 2; u++) b[u] = load8(brow[u] + (int64_t)c0 * 9 * cout);
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[u], acc[t][u], 0, 0, 0);
        }
    }
    // epilogue: lane holds column n = l % 16, rows 4 * (l / 16) + i
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int n = n_base + u * 16 + row;
        const float bv = (flags & 1) ? bias[n] : 0.f;
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int pix = m_base + t * 16 + (lane >> 4) * 4 + i;
                if (pix >= npix) continue;
                float v = acc[t][u][i] + bv;
                if (flags & 2) v = v > 0.f ? v : 0.f;
                if (out) out[(int64_t)pix * cout + n] = (bf16)v;
                if (out32) out32[(int64_t)pix * cout + n] = v;
            }
    }
}

// The same product, term by term in the same order (taps outermost), for images
// of at most 64 pixels whose sides the tiles below do not divide: the deep
// levels of a small frame.  A workgroup holds one whole image with its border of
// zeros in LDS (all its channels), and each of its four waves one 16-pixel by
// 16-channel tile.  A step's weights are a kilobyte in one piece (packed_at), and a
// wave streams them from L2, nine steps ahead.  The kernel above
// waits for two loads from memory at every step, with a workgroup on a few CUs:
// 31 us for 32 images of 8 x 4 pixels and 256 to 256 channels, 12.6 here.
constexpr int SMALL_PIXELS = 64, SMALL_LDS = 64 * 1024;
static inline int small_patch_bytes(int cin, int H, int W) {
    return (H + 2) * (W + 2) * (cin + 8) * (int)sizeof(bf16);
}
__global__ void __launch_bounds__(256)
k_conv3x3_small(const bf16* __restrict__ in, int cin, const bf16* __restrict__ w,
                const float* __restrict__ bias, bf16* __restrict__ out, float* __restrict__ out32,
                int cout, int H, int W, int mt, int flags, const int* __restrict__ live)
{
    extern __shared__ __attribute__((aligned(16))) bf16 patch[];   // [(H + 2) (W + 2)][cin + 8]
    const int img = blockIdx.x, HW = H * W, PW = W + 2, cs = cin + 8;
    if (live && img >= *live) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, kq = (lane >> 4) * 8;
    const int nv = cin / 8;
    for (int v = tid; v < (H + 2) * PW * nv; v += 256) {
        const int px = v / nv, c = (v - px * nv) * 8, y = px / PW - 1, x = px - px / PW * PW - 1;
        const bool inside = y >= 0 && y < H && x >= 0 && x < W;
        const int64_t from = ((int64_t)img * HW + (inside ? y * W + x : 0)) * cin + c;
        const bf16x8 q = load8(in + from);
        *reinterpret_cast<bf16x8*>(&patch[px * cs + c]) = inside ? q : zero8();
    }
    __syncthreads();
    const int tile = wave & (mt - 1), n0 = (blockIdx.y * (4 / mt) + wave / mt) * 16;
    if (n0 >= cout || tile * 16 >= HW) return;
    const int pix = min(tile * 16 + row, HW - 1), py = pix / W, px = pix - py * W;
    const bf16* pa = &patch[(py * PW + px) * cs + kq];   // tap 0: one row up, one left
    const bf16* pw = w + (n0 + row) * 32 + kq;
    // steps of 32 k's: tap-major, then the channels; nine at a time
    const int per = cin / 32, batches = per;             // 9 * per steps
    bf16x8 cur[9], nxt[9];
    int tw = 0, cw = 0;                                  // step of the next load
    auto weights = [&](bf16x8 (&q)[9]) {
#pragma unroll
        for (int j = 0; j < 9; j++) {
            q[j] = load8(pw + (int64_t)(cw * 9 + tw) * cout * 32);
            if (++cw == per) {
                cw = 0;
                tw = tw == 8 ? 0 : tw + 1;               // (past the end: loaded, not used)
            }
        }
    };
    weights(cur);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int tap = 0, c = 0;
    for (int b = 0; b < batches; b++) {
        weights(nxt);
        __builtin_amdgcn_sched_barrier(0);   // the loads issue before the MFMAs
#pragma unroll
        for (int j = 0; j < 9; j++) {
            const bf16x8 a = load8(pa + (tap / 3 * PW + tap % 3) * cs + c * 32);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, cur[j], acc, 0, 0, 0);
            if (++c == per) {
                c = 0;
                tap++;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 9; j++) cur[j] = nxt[j];
    }
    const int n = n0 + row;
    const float bv = (flags & 1) ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int p = tile * 16 + (lane >> 4) * 4 + i;
        if (p >= HW) continue;
        float v = acc[i] + bv;
        if (flags & 2) v = v > 0.f ? v : 0.f;
        const int64_t o = ((int64_t)img * HW + p) * cout + n;
        if (out) out[o] = (bf16)v;
        if (out32) out32[o] = v;
    }
}

// LDS-tiled variant.  A workgroup owns a TH x TW pixel tile of one image
// (TH * TW = 64 or 128) and NW = 32 * WN output channels; for every
// 32-channel slice of the input it stages in LDS the (TH + 2) x (TW + 2)
// patch and the slice's weights of its NW channels, and serves all nine taps
// and all four waves from them: each input value is read from memory once per
// slice and channel block, each weight once per workgroup.  Waves: (4 / WN) in
// M x WN in N; a wave owns MT M tiles of 16 pixels (RM = 16 / TW image rows
// each) on consecutive rows, and 32 output channels (two N tiles).  The
// MFMAs take the weights as their first operand, so each result holds
// channels as rows and pixels as columns, and a lane ends with four
// consecutive channels of one pixel to store.
//
// The MFMA operand of tap (dy, dx) for M tile i is the patch block that
// starts RM * i + dy rows below the wave's first row, shifted by dx: the
// wave walks the distinct starts s once per dx and feeds each fragment to
// every (i, dy) with RM * i + dy = s, so a fragment is read from LDS once for
// up to three taps.  Each output's taps are added in the order dx-major,
// dy ascending (0, 3, 6, 1, 4, 7, 2, 5, 8), slice after slice.
//
// The input is described by ConvIn: channels [0, ca) come from `a` read
// directly, as the 2x2 max of an image twice the size (the U-Net's pooling)
// or as the nearest upsampling of an image half the size; channels
// [ca, ca + cb) come from `b` read directly (the skip half of a
// concatenation).  Pooling, upsampling and concatenation thus happen while
// staging, without materialising their outputs.
//
// With PIPE (chosen for workgroups with at least three input slices, in
// launches of at most two workgroups per CU) patch and weights are
// double-buffered in LDS and the loads run two slices ahead in registers, so
// one barrier per slice suffices and the load latency hides behind two
// slices of matrix work.  The other launches (few slices, or enough
// workgroups that occupancy hides the latency) stage each slice and then
// multiply, in half the LDS.
//
// LDS strides: a 16-byte read serves 16 lanes at once, lanes 0 to 3 and 12 to 15
// of one 8-channel group (kq) with lanes 4 to 11 of the next, over 64 banks.  In
// units of 16 bytes an operand's 16 rows then miss each other if their stride is 2
// more than a multiple of 4: a pixel takes 6 units, a channel's nine weight rows
// 38, and where a fragment is eight pixels of two image rows, those lie 4 units
// further apart.  With 5 units a pixel and 45 a channel a read took 8 to 12 cycles
// instead of 4 (4.8 cycles of conflicts per LDS instruction counted, 0.7 now, the
// stores'): the 14 layers of 32 frames of 64 x 64 147 us, 138 now; of 64 frames of
// 128 x 64 399 and 381.
template <int TW, int TH, int WN, bool POOL, bool PIPE>
__global__ void __launch_bounds__(256)
k_conv3x3_tile(ConvIn src, const bf16* __restrict__ w, const float* __restrict__ bias,
               bf16* __restrict__ out, float* __restrict__ out32, int cout, int nb, int H, int W,
               int flags)
{
    constexpr int PH = TH + 2, PW = TW + 2;
    constexpr int CS = 48;                       // padded channel stride of a staged pixel
    constexpr int RS = PW * CS + (TW == 8 ? 32 : 0);   // stride of a patch row
    constexpr int CHS = 9 * 32 + 16;             // stride of a channel's nine weight rows
    constexpr int NW = 32 * WN;                  // output channels of the workgroup
    constexpr int WM = 4 / WN;                   // waves along M
    constexpr int RM = 16 / TW;                  // image rows per M tile
    constexpr int MT = TH * TW / WM / 16;        // M tiles per wave
    constexpr int NS = RM * (MT - 1) + 3;        // distinct fragment starts per dx
    constexpr int NPV = PH * PW * 4;             // 16-byte vectors of one staged slice
    constexpr int NV = (NPV + 255) / 256;        // of them per thread
    constexpr int NWVEC = NW * 9 * 4;            // 16-byte vectors of one slice's weights
    constexpr int NWV = (NWVEC + 255) / 256;
    constexpr int NB = PIPE ? 2 : 1;
    static_assert(TW == 8 || TW == 16, "tile width");
    static_assert(MT >= 1 && TH * TW % (WM * 16) == 0, "tile shape");
    __shared__ __attribute__((aligned(16))) bf16 patch[NB][PH * RS];
    __shared__ __attribute__((aligned(16))) bf16 wl[NB][NW * CHS];

    const int cin = src.ca + src.cb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int tiles_w = (W + TW - 1) / TW, tiles_h = (H + TH - 1) / TH;
    int t = blockIdx.x;
    const int tw0 = (t % tiles_w) * TW;
    t /= tiles_w;
    const int th0 = (t % tiles_h) * TH;
    const int b = t / tiles_h;
    if (src.live && b >= *src.live) return;      // uniform over the block, before any barrier
    const int nb0 = blockIdx.y * NW;
    const int n_base = nb0 + wn * 32;
    const int row = lane & 15, kq = (lane >> 4) * 8;

    // this lane's LDS offsets: its pixel of the wave's first M tile at tap
    // (0, 0), and its weight row (channel n_base + row) at tap 0
    const int aoff = (wm * MT * RM + row / TW) * RS + row % TW * CS + kq;
    const int boff = (wn * 32 + row) * CHS + kq;
    f32x4 acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
        for (int u = 0; u < 2; u++) acc[i][u] = f32x4{0.f, 0.f, 0.f, 0.f};

    // split K: block z of gridDim.z takes its share of the 32-channel slices
    const int nsl = cin / 32, z = blockIdx.z, nz = gridDim.z;
    const int sl0 = z * nsl / nz, sl1 = (z + 1) * nsl / nz;

    // Staging: the loads of a slice are issued unconditionally (addresses
    // clamped into the image, out-of-image vectors zeroed when stored), with
    // no branch between them, so the compiler can count them exactly; a
    // pooled input (POOL, src.mode == IN_POOL, never with a skip part) keeps
    // its four window values in registers and takes their max when storing.
    constexpr bool pool = POOL;
    constexpr int NR = POOL ? 4 : 1;
    struct Stage {               // one slice's loads in flight
        bf16x8 raw[NV][NR];
        bf16x8 w[NWV];
        uint32_t valid;
    };
    auto fetch = [&](Stage& g, int c0) {
        const bool first = c0 < src.ca;
        const bf16* base = first ? src.a : src.b;
        const int cs = first ? src.ca : src.cb, cc = first ? c0 : c0 - src.ca;
        const int up = (first && src.mode == IN_UP) ? 1 : 0, dn = pool ? 1 : 0;
        const int Hs = (H << dn) >> up, Ws = (W << dn) >> up;     // source image
        g.valid = 0;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int v = threadIdx.x + k * 256;
            const int vv = v < NPV ? v : 0;
            const int pix = vv >> 2, part = vv & 3;
            const int ph = pix / PW, pw = pix - ph * PW;
            const int gh = th0 + ph - 1, gw = tw0 + pw - 1;
            if (v < NPV && gh >= 0 && gh < H && gw >= 0 && gw < W) g.valid |= 1u << k;
            const int ghc = min(max(gh, 0), H - 1), gwc = min(max(gw, 0), W - 1);
            const int64_t r0 = (((int64_t)b * Hs + ((ghc << dn) >> up)) * Ws + ((gwc << dn) >> up))
                               * cs + cc + part * 8;
            g.raw[k][0] = load8(base + r0);
            if constexpr (POOL) {
                const int64_t rs = (int64_t)Ws * cs;
                g.raw[k][1] = load8(base + r0 + cs);
                g.raw[k][2] = load8(base + r0 + rs);
                g.raw[k][3] = load8(base + r0 + rs + cs);
            }
        }
        // the slice's weights: vector v = (tap * NW + n) * 4 + part
        const bf16* ws = w + ((int64_t)(c0 / 32) * 9 * cout + nb0) * 32;
#pragma unroll
        for (int k = 0; k < NWV; k++) {
            const int v = threadIdx.x + k * 256;
            const int vv = v < NWVEC ? v : 0;
            g.w[k] = load8(ws + (int64_t)(vv / (NW * 4)) * cout * 32 + vv % (NW * 4) * 8);
        }
    };
    auto put = [&](const Stage& g, int buf) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int v = threadIdx.x + k * 256;
            if (v >= NPV) continue;
            bf16x8 x = g.raw[k][0];
            if constexpr (POOL) {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    x[e] = (bf16)fmaxf(fmaxf((float)g.raw[k][0][e], (float)g.raw[k][1][e]),
                                       fmaxf((float)g.raw[k][2][e], (float)g.raw[k][3][e]));
            }
            if (!((g.valid >> k) & 1u)) x = zero8();
            *reinterpret_cast<bf16x8*>(&patch[buf][(v >> 2) * CS + (v >> 2) / PW * (RS - PW * CS) +
                                                    (v & 3) * 8]) = x;
        }
#pragma unroll
        for (int k = 0; k < NWV; k++) {
            const int v = threadIdx.x + k * 256;
            if (v >= NWVEC) continue;
            *reinterpret_cast<bf16x8*>(&wl[buf][(v >> 2) % NW * CHS + v / (NW * 4) * 32 + (v & 3) * 8]) = g.w[k];
        }
    };
    auto mfmas = [&](int buf) {
        const bf16* pa = &patch[buf][aoff];
        const bf16* pb = &wl[buf][boff];
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
            bf16x8 bq[3][2];
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    bq[dy][u] = *reinterpret_cast<const bf16x8*>(pb + u * 16 * CHS + (dy * 3 + dx) * 32);
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(pa + s * RS + dx * CS);
#pragma unroll
                for (int dy = 0; dy < 3; dy++) {
                    const int d = s - dy;
                    if (d < 0 || d % RM != 0 || d / RM >= MT) continue;
#pragma unroll
                    for (int u = 0; u < 2; u++)   // channels as rows, pixels as columns
                        acc[d / RM][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            bq[dy][u], a, acc[d / RM][u], 0, 0, 0);
                }
            }
        }
    };

    if constexpr (PIPE) {
        // Two slices in flight: slice s is multiplied out of one LDS buffer
        // while slice s + 1 (loaded during the previous slice) is stored to
        // the other and slice s + 2 is being loaded, so each load has two
        // slices' time to arrive.  Slice s of the split sits in buffer
        // (s - sl0) & 1 and in stage g0 / g1 by the same parity.  The
        // workgroup has at least three slices (the launcher's condition);
        // the loads in the main loop are unconditional, so the compiler's
        // wait counts stay exact.
        Stage g0, g1;
        fetch(g0, sl0 * 32);
        fetch(g1, min(sl0 + 1, sl1 - 1) * 32);
        put(g0, 0);
        __syncthreads();
        int s = sl0;
        for (; s + 3 < sl1; s += 2) {
            fetch(g0, (s + 2) * 32);
            __builtin_amdgcn_sched_barrier(0);   // the loads issue before the MFMAs
            mfmas(0);
            put(g1, 1);          // buffer 1 was last read before the previous barrier
            __syncthreads();
            fetch(g1, (s + 3) * 32);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(1);
            put(g0, 0);
            __syncthreads();
        }
        // the last one to three slices: s in buffer 0, s + 1 in g1
        if (s + 2 < sl1) fetch(g0, (s + 2) * 32);
        mfmas(0);
        if (s + 1 < sl1) {
            put(g1, 1);
            __syncthreads();
            mfmas(1);
            if (s + 2 < sl1) {
                put(g0, 0);
                __syncthreads();
                mfmas(0);
            }
        }
    } else {
        Stage g;
        for (int s = sl0; s < sl1; s++) {
            if (s > sl0) __syncthreads();        // the previous slice's MFMAs are done
            fetch(g, s * 32);
            put(g, 0);
            __syncthreads();
            mfmas(0);
        }
    }
    // epilogue: the result tile is (channels x pixels), so the lane holds
    // pixel row of each M tile and its four consecutive channels
    // n_base + 16 u + 4 (l / 16) + 0..3: one 8-byte store of bf16 (16 bytes
    // of fp32) per tile and channel half
    const int q4 = (lane >> 4) * 4;
    // with the fused head (32 channels, WN == 1, no split) each wave also
    // stages its bf16 outputs, one row of CS per pixel, where the patch was
    constexpr int HROWS = MT * 16;
    static_assert(WN != 1 || 4 * HROWS <= PH * PW, "head staging fits the patch buffer");
    const bool head = WN == 1 && src.head_y != nullptr;      // uniform
    bf16* hs = &patch[0][0] + wave * HROWS * CS;
    if (head) __syncthreads();       // every wave's MFMAs are done with the patch
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int n = n_base + u * 16 + q4;
        float4 bv = {0.f, 0.f, 0.f, 0.f};
        if ((flags & 1) && nz == 1) bv = *reinterpret_cast<const float4*>(bias + n);
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int m = (wm * MT + i) * 16 + row;
            const int gh = th0 + m / TW, gw = tw0 + m % TW;
            if (gh >= H || gw >= W) continue;
            const int64_t o = (((int64_t)b * H + gh) * W + gw) * cout + n;
            const f32x4 r = acc[i][u];
            if (nz > 1) {   // split z's partial sum in its own slice; k_conv_finish adds them
                *reinterpret_cast<float4*>(src.acc32 + (int64_t)z * ((int64_t)nb * H * W * cout) + o) =
                    float4{r[0], r[1], r[2], r[3]};
                continue;
            }
            float v[4] = {r[0] + bv.x, r[1] + bv.y, r[2] + bv.z, r[3] + bv.w};
            if (flags & 2)
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = v[j] > 0.f ? v[j] : 0.f;
            typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
            const bf16x4 vb = {(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
            if (out) *reinterpret_cast<bf16x4*>(out + o) = vb;
            if (out32) *reinterpret_cast<float4*>(out32 + o) = float4{v[0], v[1], v[2], v[3]};
            if (head) *reinterpret_cast<bf16x4*>(hs + (i * 16 + row) * CS + u * 16 + q4) = vb;
        }
    }
    if (head) {
        __syncthreads();
        if (lane < HROWS) {
            const int m = wm * HROWS + lane;
            const int gh = th0 + m / TW, gw = tw0 + m % TW;
            if (gh < H && gw < W) {
                float sum = src.head_b[0];
#pragma unroll
                for (int c = 0; c < 32; c += 8) {
                    const bf16x8 x = *reinterpret_cast<const bf16x8*>(hs + lane * CS + c);
#pragma unroll
                    for (int e = 0; e < 8; e++) sum += (float)x[e] * src.head_w[c + e];
                }
                src.head_y[((int64_t)b * H + gh) * W + gw] = sum;
            }
        }
    }
}

// Completes a split-K convolution: the ks partial sums added in split order
// (the same bits on every run), then bias, ReLU and BF16; four consecutive
// channels per thread (n and cout are multiples of 4).
__global__ void __launch_bounds__(256)
k_conv_finish(const float* __restrict__ acc32, int ks, const float* __restrict__ bias,
              bf16* __restrict__ out, float* __restrict__ out32, int64_t n, int cout, int flags,
              const int* __restrict__ live, int64_t per_image)
{
    const int64_t k = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (k >= n) return;
    if (live && k >= (int64_t)*live * per_image) return;   // images the splits skipped
    float4 v = *reinterpret_cast<const float4*>(acc32 + k);
    for (int z = 1; z < ks; z++) {
        const float4 a = *reinterpret_cast<const float4*>(acc32 + (int64_t)z * n + k);
        v.x = v.x + a.x;
        v.y = v.y + a.y;
        v.z = v.z + a.z;
        v.w = v.w + a.w;
    }
    if (flags & 1) {
        const float4 bv = *reinterpret_cast<const float4*>(bias + (int)(k % cout));
        v.x = v.x + bv.x;
        v.y = v.y + bv.y;
        v.z = v.z + bv.z;
        v.w = v.w + bv.w;
    }
    if (flags & 2) {
        v.x = v.x > 0.f ? v.x : 0.f;
        v.y = v.y > 0.f ? v.y : 0.f;
        v.z = v.z > 0.f ? v.z : 0.f;
        v.w = v.w > 0.f ? v.w : 0.f;
    }
    if (out) {
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<bf16x4*>(out + k) = bf16x4{(bf16)v.x, (bf16)v.y, (bf16)v.z, (bf16)v.w};
    }
    if (out32) *reinterpret_cast<float4*>(out32 + k) = v;
}

// w'[ci][8 - tap][co] = w[co][tap][ci] for every layer of the list, each at the
// offset of its own weights: one launch in front of the backward pass (3.7 us
// for each layer by itself before, 6.5 for all now)
__global__ void __launch_bounds__(256)
k_weight_flip(FlipList l, const bf16* __restrict__ w, bf16* __restrict__ wt)
{
    // a block turns 32 co x 32 ci of one tap in LDS, so that reads and stores both
    // run along the channels
    __shared__ bf16 tile[32][33];
    int k = 0;
    while (k + 1 < l.n && blockIdx.x >= l.block[k + 1]) k++;
    const int cin = l.cin[k], cout = l.cout[k];
    const int b = blockIdx.x - l.block[k], tap = b % 9, ci0 = b / 9 % (cin / 32) * 32,
              co0 = b / 9 / (cin / 32) * 32;
    const int lane = threadIdx.x & 31, row = threadIdx.x >> 5;   // eight rows at a time
    const bf16* from = w + l.off[k];
    bf16* to = wt + l.off[k];
#pragma unroll
    for (int r = row; r < 32; r += 8)
        tile[r][lane] = from[((int64_t)(ci0 / 32 * 9 + 8 - tap) * cout + co0 + r) * 32 + lane];
    __syncthreads();
#pragma unroll
    for (int r = row; r < 32; r += 8)
        to[((int64_t)(co0 / 32 * 9 + tap) * cin + ci0 + r) * 32 + lane] = tile[lane][r];
}

// dw[co][tap][ci] over a pixel chunk: sum of gz[pix][co] * in[pix+off][ci].
// Block: 256 threads, a tile of up to 64 co x 64 ci for the three taps of one
// dy.  The MFMAs' k is the pixel, so both operands are read transposed: 128
// pixels at a time are staged as they lie in memory (gz's rows, and of `in` the
// 130 pixels that the three dx reach, whatever the width), and
// ds_read_b64_tr_b16 hands lane c of 16 the channel c of four pixels; a lane
// whose pixel has no neighbour there reads a row of zeros instead.  The next
// 128 pixels are loaded while these are multiplied.  Transposing with 2-byte LDS
// stores, for each tap by itself, was what bounded the pass before.  What bounds
// a round is the transposed reads (16 for 12 MFMAs): eight waves with 32 x 16
// pieces, loads two and three rounds ahead and a pixel padded to 160 bytes
// measured no faster (16.0 us for a layer on average, 15.7 to 16.6 those).  The
// layers of a network run together, a launch for each kind of tile: by themselves
// most are a few dozen workgroups.  All 14 layers of 32 frames of 64 x 64: 416 us
// with the stores, 224 layer by layer, 135 in four launches.
//
// The four waves cover the tile in 32 x 32 pieces and split the four 32-pixel
// k steps among themselves when the tile is narrower than 64 x 64, so no wave
// multiplies padding; those waves then add their sums in LDS in wave order.
// With one pixel chunk (chunk_stride 0) the block adds its sums into dw; with
// several, chunk z writes its own slice out[z * chunk_stride + ...] and
// k_grad_finish adds the slices in chunk order, so the result does not depend
// on the order in which blocks finish.
template <int CO, int CI>   // the tile: 32 or 64 of each
__global__ void __launch_bounds__(256)
k_conv3x3_dw(DwList l)
{
    int q = 0;
    while (q + 1 < l.n && blockIdx.x >= l.block[q + 1]) q++;
    const DwLayer& a = l.layer[q];
    const bf16* __restrict__ gz = a.gz;
    const bf16* __restrict__ in = a.in;
    float* __restrict__ out = a.out;
    const int cout = a.cout, cin = a.cin, H = a.H, W = a.W, npix = a.nb * a.H * a.W;
    // workgroups of a layer: input tile, output tile, dy, chunk
    int at_block = blockIdx.x - l.block[q];
    const int ti = at_block % a.ntile_ci;
    at_block /= a.ntile_ci;
    const int to = at_block % (cout / CO);
    at_block /= cout / CO;
    const int dy = at_block % 3 - 1, chunk = at_block / 3;
    const int64_t chunk_stride = a.chunk_stride;
    // KP pixels at once; a staged pixel takes LS channels (144 bytes: the 16
    // rows of a read then cover the banks evenly)
    constexpr int KP = 128, WP = KP + 2, LS = 72;
    constexpr int GV = CO / 8, IV = CI / 8;                       // 16-byte vectors of a pixel
    constexpr int NG = KP * GV / 256, NI = (WP * IV + 255) / 256; // of them per thread
    constexpr int WO = CO / 32, WI = CI / 32, KS = 4 / (WO * WI);
    __shared__ __attribute__((aligned(16))) bf16 smem[(KP + WP + 1) * LS];
    __shared__ uint8_t near[KP];   // bit dx + 1: the pixel has that neighbour in row h + dy
    bf16* sg = smem;               // [pixel][co]
    bf16* si = smem + KP * LS;     // [pixel + dx + 1][ci], then a row of zeros
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int co0 = to * CO;
    const int ci0 = a.ci_first + ti * CI;
    const int p_begin = chunk * a.per;
    const int p_end = min(npix, p_begin + a.per);
    const int mo = wave % WO, ni = wave / WO % WI, kg = wave / (WO * WI);
    f32x4 acc[3][2][2];
    for (int x = 0; x < 3; x++)
        for (int t = 0; t < 2; t++)
            for (int u = 0; u < 2; u++) acc[x][t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int row = lane & 15;

    // a thread's vectors of the next 128 pixels: loaded from addresses clamped
    // into the batch, without branches, and zeroed when stored if they lie
    // outside the chunk
    bf16x8 vg[NG], vi[NI];
    uint32_t edge = 0;
    auto fetch = [&](int p0) {
#pragma unroll
        for (int k = 0; k < NG; k++) {
            const int v = tid + k * 256, pix = min(p0 + v / GV, npix - 1);
            vg[k] = load8(gz + (int64_t)pix * cout + co0 + v % GV * 8);
        }
#pragma unroll
        for (int k = 0; k < NI; k++) {
            const int v = min(tid + k * 256, WP * IV - 1);
            const int pix = min(max(p0 + dy * W - 1 + v / IV, 0), npix - 1);
            vi[k] = load8(in + (int64_t)pix * cin + ci0 + v % IV * 8);
        }
        const int pix = p0 + (tid & (KP - 1)), w = pix % W, hh = pix / W % H + dy;
        const bool inside = pix < p_end && hh >= 0 && hh < H;
        edge = inside ? (w > 0 ? 1u : 0u) | 2u | (w + 1 < W ? 4u : 0u) : 0u;
    };
    if (tid < LS / 8) *reinterpret_cast<bf16x8*>(&si[WP * LS + tid * 8]) = zero8();

    // a transposed read's source: pixel 8 (lane / 16) + row / 4 (+ 4), four channels
    const int src = (8 * (lane >> 4) + row / 4) * LS + 4 * (row % 4);
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) bf16x4 lds4;
    auto pair = [](const bf16* lo, const bf16* hi) -> bf16x8 {
        const bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4*)lo);
        const bf16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4*)hi);
        return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    fetch(p_begin);
    for (int p0 = p_begin; p0 < p_end; p0 += KP) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NG; k++) {
            const int v = tid + k * 256;
            *reinterpret_cast<bf16x8*>(&sg[v / GV * LS + v % GV * 8]) =
                p0 + v / GV < p_end ? vg[k] : zero8();
        }
#pragma unroll
        for (int k = 0; k < NI; k++) {   // (a pixel that is no neighbour is not read)
            const int v = tid + k * 256;
            if (v < WP * IV) *reinterpret_cast<bf16x8*>(&si[v / IV * LS + v % IV * 8]) = vi[k];
        }
        if (tid < KP) near[tid] = (uint8_t)edge;
        __syncthreads();
        fetch(p0 + KP);   // (past the chunk's end: loaded, not used)
        __builtin_amdgcn_sched_barrier(0);   // the loads issue before the MFMAs
        uint32_t n0[4 / KS], n1[4 / KS];
#pragma unroll
        for (int j = 0; j < 4 / KS; j++) {
            const int px = (kg + j * KS) * 32 + 8 * (lane >> 4) + row / 4;
            n0[j] = near[px];
            n1[j] = near[px + 4];
        }
#pragma unroll
        for (int j = 0; j < 4 / KS; j++) {
            const int k = kg + j * KS;
            const bf16* ga = sg + k * 32 * LS + src + mo * 32;
            bf16x8 a[2];
#pragma unroll
            for (int t = 0; t < 2; t++) a[t] = pair(ga + t * 16, ga + t * 16 + 4 * LS);
#pragma unroll
            for (int x = 0; x < 3; x++) {
                const bf16* ib = si + (k * 32 + x) * LS + src;
                const bf16* zero = si + WP * LS;
                const bf16* lo = ((n0[j] >> x) & 1u ? ib : zero) + ni * 32;
                const bf16* hi = ((n1[j] >> x) & 1u ? ib + 4 * LS : zero) + ni * 32;
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const bf16x8 b = pair(lo + u * 16, hi + u * 16);
#pragma unroll
                    for (int t = 0; t < 2; t++)
                        acc[x][t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b, acc[x][t][u],
                                                                              0, 0, 0);
                }
            }
        }
    }
    if (KS > 1) {
#pragma unroll
        for (int x = 0; x < 3; x++) {
            // wave w + g * WO * WI holds k group g of wave w's piece: 16 floats a
            // lane, 4 KB a wave, in the staging memory once every wave is past
            // its last read of it
            float* red = reinterpret_cast<float*>(smem);
            __syncthreads();
            if (kg > 0)
                for (int t = 0; t < 2; t++)
                    for (int u = 0; u < 2; u++)
                        for (int i = 0; i < 4; i++)
                            red[(wave * 16 + (t * 2 + u) * 4 + i) * 64 + lane] = acc[x][t][u][i];
            __syncthreads();
            if (kg == 0)
                for (int g = 1; g < KS; g++) {
                    const int w2 = wave + g * WO * WI;
                    for (int t = 0; t < 2; t++)
                        for (int u = 0; u < 2; u++)
                            for (int i = 0; i < 4; i++)
                                acc[x][t][u][i] += red[(w2 * 16 + (t * 2 + u) * 4 + i) * 64 + lane];
                }
        }
        if (kg != 0) return;
    }
    // the wave's piece: lane l % 16 is a ci, so each store writes four runs of 64 bytes
    const int cr = co0 + mo * 32 + (lane >> 4) * 4, cc = ci0 + ni * 32 + row;
    float* dst = out + (int64_t)chunk * chunk_stride + ((int64_t)cr * 9 + (dy + 1) * 3) * cin + cc;
    auto at = [&](int x, int t, int u, int i) -> float& {
        return dst[((t * 16 + i) * 9 + x) * cin + u * 16];
    };
    if (chunk_stride == 0) {   // the loads together, before any store
        float old[3][2][2][4];
#pragma unroll
        for (int k = 0; k < 48; k++)
            old[k / 16][k / 8 % 2][k / 4 % 2][k % 4] = at(k / 16, k / 8 % 2, k / 4 % 2, k % 4);
#pragma unroll
        for (int k = 0; k < 48; k++)
            acc[k / 16][k / 8 % 2][k / 4 % 2][k % 4] =
                old[k / 16][k / 8 % 2][k / 4 % 2][k % 4] + acc[k / 16][k / 8 % 2][k / 4 % 2][k % 4];
    }
#pragma unroll
    for (int k = 0; k < 48; k++)
        at(k / 16, k / 8 % 2, k / 4 % 2, k % 4) = acc[k / 16][k / 8 % 2][k / 4 % 2][k % 4];
}

// The sum of a block's 256 values in a fixed LDS tree; for thread 0.
__device__ __forceinline__ float tree256(float s, float* red) {
    red[threadIdx.x] = s;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
        __syncthreads();
    }
    return red[0];
}

// The layers' partial gradients into their gradients, in one launch (a launch of
// 4.6 us for each of 14 layers before; 28 us for all of 64 x 64 frames' now, 13 of
// 64 x 32 ones').  A layer's first `cout`
// blocks take its bias: channel j's db += the sum over k of bpart[k * cout + j],
// thread t adding k = t, t + 256, ... in order, then a fixed LDS tree.  The others
// take its weights, if there were several chunks: dw[i] += part[i] + part[n + i]
// + ... + part[(chunks - 1) n + i], in that order.
__global__ void __launch_bounds__(256)
k_grad_finish(GradList l, const float* __restrict__ parts, const float* __restrict__ bparts,
              float* __restrict__ grads)
{
    __shared__ float red[256];
    int q = 0;
    while (q + 1 < l.n && blockIdx.x >= l.block[q + 1]) q++;
    const int j = blockIdx.x - l.block[q], c = l.cout[q];
    if (j < c) {
        const float* bpart = bparts + l.bpoff[q];
        float s = 0.f;
        for (int k = threadIdx.x; k < l.bblocks[q]; k += 256) s += bpart[(int64_t)k * c + j];
        s = tree256(s, red);
        float* db = grads + l.boff[q];
        if (threadIdx.x == 0) db[j] = db[j] + s;
        return;
    }
    const float* part = parts + l.poff[q];
    const int64_t n = (int64_t)c * 9 * l.cin[q], i = ((int64_t)(j - c) * 256 + threadIdx.x) * 4;
    if (i >= n) return;   // (n is a multiple of 4)
    float4 s = *reinterpret_cast<const float4*>(part + i);
#pragma unroll 8
    for (int k = 1; k < l.chunks[q]; k++) {
        const float4 v = *reinterpret_cast<const float4*>(part + (int64_t)k * n + i);
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
    }
    float4* dw = reinterpret_cast<float4*>(grads + l.woff[q] + i);
    float4 o = *dw;
    o.x += s.x;
    o.y += s.y;
    o.z += s.z;
    o.w += s.w;
    *dw = o;
}

// Block j: the sum over k of part[k * stride + col0 + j], k in [0, nparts):
// thread t adds k = t, t + 256, ... in order, then a fixed LDS tree.  dst[j]
// gets it added (add) or assigned.
__global__ void __launch_bounds__(256)
k_block_sum(const float* __restrict__ part, int nparts, int stride, int col0,
            float* __restrict__ dst, int add)
{
    __shared__ float red[256];
    const int j = blockIdx.x;
    float s = 0.f;
    for (int k = threadIdx.x; k < nparts; k += 256) s += part[(int64_t)k * stride + col0 + j];
    s = tree256(s, red);
    if (threadIdx.x == 0) dst[j] = add ? dst[j] + s : s;
}

// ------------------------------------------------------------ elementwise

// The gradient through a ReLU whose output is y, g = g * (y > 0), and its sums
// for the bias: part[block][c] = sum over the block's pixels of g[pix][c].  c is
// 32, 64, 128 or 256: thread t takes the 8 channels of vector v = t % (c / 8)
// (one 16-byte load per pixel) for pixels j, j + lanes, ... of the block's chunk
// (j = t / (c / 8), lanes = 256 / (c / 8)), each channel added in pixel order;
// then the lanes' partials of each channel are added in LDS in lane order.  The
// loads of several pixels are in flight at once.  (Bound by memory; in two
// passes, the first a value per thread, 9.4 us a layer on average at 32 frames
// of 64 x 64, 5.4 now.)
__global__ void __launch_bounds__(256)
k_relu_bias_bwd(const bf16* __restrict__ y, bf16* __restrict__ g, int c, int npix, int per,
                float* __restrict__ part)
{
    __shared__ float red[256 * 8];
    const int nv = c / 8, v = threadIdx.x % nv, j = threadIdx.x / nv, lanes = 256 / nv;
    const int p0 = blockIdx.x * per, p1 = min(npix, p0 + per);
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;
    for (int p = p0 + j; p < p1; p += U * lanes) {
        bf16x8 x[U], o[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t at = (int64_t)min(p + u * lanes, p1 - 1) * c + v * 8;
            x[u] = load8(g + at);
            o[u] = load8(y + at);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (p + u * lanes >= p1) break;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (!((float)o[u][e] > 0.f)) x[u][e] = (bf16)0.f;
                s[e] += (float)x[u][e];
            }
            *reinterpret_cast<bf16x8*>(g + (int64_t)(p + u * lanes) * c + v * 8) = x[u];
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) red[threadIdx.x * 8 + e] = s[e];
    __syncthreads();
    if (threadIdx.x < c) {
        const int cv = threadIdx.x / 8, ce = threadIdx.x % 8;
        float t = 0.f;
        for (int k = 0; k < lanes; k++) t += red[(k * nv + cv) * 8 + ce];
        part[(int64_t)blockIdx.x * c + threadIdx.x] = t;
    }
}

// The elementwise passes take eight channels a thread, one 16-byte access each:
// they are bound by memory (upsampling to 64 x 64 x 64 of 32 frames 17.7 us and
// 6.1 for the skip's copy with a channel a thread, 6.1 together now).
__device__ __forceinline__ void store8(bf16* p, bf16x8 v) { *reinterpret_cast<bf16x8*>(p) = v; }

// 2x2 max pooling, H and W even
__global__ void __launch_bounds__(256)
k_maxpool(const bf16* __restrict__ x, bf16* __restrict__ y, int nb, int H, int W, int c,
          const int* __restrict__ live)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int Ho = H / 2, Wo = W / 2, nv = c / 8;
    const int64_t n = (int64_t)(live ? min(nb, *live) : nb) * Ho * Wo * nv;
    if (k >= n) return;
    const int ch = (int)(k % nv) * 8;
    const int64_t q = k / nv;
    const int wo = (int)(q % Wo), ho = (int)((q / Wo) % Ho), b = (int)(q / ((int64_t)Wo * Ho));
    const int64_t base = ((int64_t)(b * H + 2 * ho) * W + 2 * wo) * c + ch, down = (int64_t)W * c;
    const bf16x8 v[4] = {load8(x + base), load8(x + base + c), load8(x + base + down),
                         load8(x + base + down + c)};
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        float m = fmaxf((float)v[0][e], (float)v[1][e]);
        m = fmaxf(m, (float)v[2][e]);
        r[e] = (bf16)fmaxf(m, (float)v[3][e]);
    }
    store8(y + k * 8, r);
}

// gradient of max pooling: to the first maximal input of each window
__global__ void __launch_bounds__(256)
k_maxpool_bwd(const bf16* __restrict__ x, const bf16* __restrict__ y, const bf16* __restrict__ gy,
              bf16* __restrict__ gx, int nb, int H, int W, int c)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int Ho = H / 2, Wo = W / 2, nv = c / 8;
    const int64_t n = (int64_t)nb * Ho * Wo * nv;
    if (k >= n) return;
    const int ch = (int)(k % nv) * 8;
    const int64_t q = k / nv;
    const int wo = (int)(q % Wo), ho = (int)((q / Wo) % Ho), b = (int)(q / ((int64_t)Wo * Ho));
    const int64_t base = ((int64_t)(b * H + 2 * ho) * W + 2 * wo) * c + ch;
    const int64_t off[4] = {0, c, (int64_t)W * c, (int64_t)W * c + c};
    bf16x8 v[4], g[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[i] = load8(x + base + off[i]);
        g[i] = load8(gx + base + off[i]);
    }
    const bf16x8 m = load8(y + k * 8), t = load8(gy + k * 8);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        bool hit = false;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool take = !hit && (float)v[i][e] == (float)m[e];
            if (take) g[i][e] = (bf16)((float)g[i][e] + (float)t[e]);
            hit = hit || take;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) store8(gx + base + off[i], g[i]);
}

// The input of a decoder convolution: the nearest 2x upsampling of x (nb, H/2,
// W/2, ca) in channels [0, ca) of y (nb, H, W, ca + cb), the skip s in the rest
__global__ void __launch_bounds__(256)
k_join(const bf16* __restrict__ x, int ca, const bf16* __restrict__ s, int cb,
       bf16* __restrict__ y, int nb, int H, int W, const int* __restrict__ live)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nv = (ca + cb) / 8;
    const int64_t n = (int64_t)(live ? min(nb, *live) : nb) * H * W * nv;
    if (k >= n) return;
    const int ch = (int)(k % nv) * 8;
    const int64_t q = k / nv;
    const int w = (int)(q % W), h = (int)((q / W) % H), b = (int)(q / ((int64_t)W * H));
    const bf16* from = ch < ca ? x + ((int64_t)(b * (H / 2) + h / 2) * (W / 2) + w / 2) * ca + ch
                               : s + q * cb + ch - ca;
    store8(y + k * 8, load8(from));
}

// Its backward: gx = the sums of gy's channels [0, ca) over each 2 x 2 block, gs
// = its channels [ca, ca + cb).  A thread takes one block of eight channels.
__global__ void __launch_bounds__(256)
k_join_bwd(const bf16* __restrict__ gy, bf16* __restrict__ gx, int ca, bf16* __restrict__ gs,
           int cb, int nb, int H, int W)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int Ho = H / 2, Wo = W / 2, cy = ca + cb, nv = cy / 8;
    if (k >= (int64_t)nb * Ho * Wo * nv) return;
    const int ch = (int)(k % nv) * 8;
    const int64_t q = k / nv;
    const int wo = (int)(q % Wo), ho = (int)((q / Wo) % Ho), b = (int)(q / ((int64_t)Wo * Ho));
    const int64_t p = (int64_t)(b * H + 2 * ho) * W + 2 * wo;
    const int64_t at[4] = {p, p + 1, p + W, p + W + 1};
    bf16x8 v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = load8(gy + at[i] * cy + ch);
    if (ch < ca) {
        bf16x8 r;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) s += (float)v[i][e];
            r[e] = (bf16)s;
        }
        store8(gx + q * ca + ch, r);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) store8(gs + at[i] * cb + ch - ca, v[i]);
    }
}

// 1x1 head: y[pix] = b + sum_c x[pix, c] * w[c]   (fp32 out)
__global__ void k_head(const bf16* __restrict__ x, int c, const float* __restrict__ w,
                       const float* __restrict__ b, float* __restrict__ y, int64_t npix,
                       const int* __restrict__ live, int64_t hw)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    if (live && p >= (int64_t)*live * hw) return;
    float s = b[0];
    const bf16* xp = x + p * c;              // c is a multiple of 8: 16-byte loads
    for (int i = 0; i < c; i += 8) {
        const bf16x8 q = load8(xp + i);
#pragma unroll
        for (int e = 0; e < 8; e++) s += (float)q[e] * w[i + e];
    }
    y[p] = s;
}

// head backward (32 channels): gx[pix, c] = gy[pix] * w[c]; per block,
// part[block][0] = sum gy and part[block][1 + c] = sum gy * x[c] over the block's
// pixels: per wave by shuffles, eight channels at a time, so that a shuffle's
// latency is shared, then the four waves in LDS.  (33.6 us for 32 frames of 64 x
// 64 with 2-byte accesses and the channels one after another, 9.5 now.)
__global__ void __launch_bounds__(256)
k_head_bwd(const bf16* __restrict__ x, const float* __restrict__ w,
           const float* __restrict__ gy, bf16* __restrict__ gx,
           float* __restrict__ part, int64_t npix)
{
    constexpr int C = 32;
    __shared__ float red[4][C + 1];
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool in = p < npix;
    const int64_t at = (in ? p : npix - 1) * C;
    const float g = in ? gy[p] : 0.f;
    bf16x8 v[C / 8];
#pragma unroll
    for (int k = 0; k < C / 8; k++) v[k] = load8(x + at + k * 8);
    if (in)
#pragma unroll
        for (int k = 0; k < C / 8; k++) {
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = (bf16)(g * w[k * 8 + e]);
            store8(gx + at + k * 8, o);
        }
    float t = g;
    for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
    if (lane == 0) red[wave][0] = t;
#pragma unroll
    for (int k = 0; k < C / 8; k++) {
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] = in ? g * (float)v[k][e] : 0.f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int e = 0; e < 8; e++) s[e] += __shfl_down(s[e], off, 64);
        if (lane == 0)
#pragma unroll
            for (int e = 0; e < 8; e++) red[wave][1 + k * 8 + e] = s[e];
    }
    __syncthreads();
    if (threadIdx.x <= C) {
        const float r = (red[0][threadIdx.x] + red[1][threadIdx.x]) +
                        (red[2][threadIdx.x] + red[3][threadIdx.x]);
        part[(int64_t)blockIdx.x * (C + 1) + threadIdx.x] = r;
    }
}

// masked MSE, normalised per sample: loss_s = sum m (y-t)^2 / sum m t^2;
// gy = 2 m (y - t) / (denominator * nb).  A sample whose target is zero (a
// solve that made no change) has weight zero.
__global__ void k_loss(const float* __restrict__ y, const float* __restrict__ t,
                       const float* __restrict__ m, const float* __restrict__ denom,
                       float* __restrict__ gy, float* __restrict__ part, int64_t npix_per,
                       int nb)
{
    __shared__ float red[256];
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = npix_per * nb;
    float l = 0.f;
    if (k < n) {
        const int s = (int)(k / npix_per);
        const float d = y[k] - t[k];
        const float mm = denom[s] > 1e-12f ? m[k] : 0.f;
        l = mm * d * d / denom[s];
        gy[k] = 2.f * mm * d / (denom[s] * nb);
    }
    red[threadIdx.x] = l / nb;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// per-sample sum of m * t^2 (+1e-30), in parts: part[block x][sample]
__global__ void k_target_norm(const float* __restrict__ t, const float* __restrict__ m,
                              float* __restrict__ part, int64_t npix_per)
{
    __shared__ float red[256];
    const int s = blockIdx.y;
    float acc = 0.f;
    for (int64_t k = blockIdx.x * 256 + threadIdx.x; k < npix_per; k += (int64_t)gridDim.x * 256) {
        const float v = t[s * npix_per + k];
        acc += m[s * npix_per + k] * v * v;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        part[(int64_t)blockIdx.x * gridDim.y + s] = red[0] + (blockIdx.x == 0 ? 1e-30f : 0.f);
}

// Where the bf16 copy keeps parameter k: a layer's weights w[co][tap][ci] lie there
// as [ci / 32][tap][co][ci % 32], so that what a workgroup reads for 32 input
// channels is whole lines.  (In the masters' order they were 64-byte pieces cin * 2
// bytes apart, in as few as four of an L2's 16 channels at once: the forward pass of
// 64 frames of 128 x 64 379 us, 358 so, of 32 of 64 x 64 139 and 137, a training
// step of 32 of 64 x 32 481 and 472.)
// Four parameters from a multiple of 4 on stay together (all counts and offsets
// are multiples of 4); what is no 3x3 weight keeps its place.
typedef __bf16 bf16x4p __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ int64_t packed_at(const WeightList& l, int64_t k) {
    int q = 0;
    while (q + 1 < l.n && k >= l.off[q + 1]) q++;
    const int r = (int)(k - l.off[q]), cin = l.cin[q];
    if (r < 0 || r >= 9 * cin * l.cout[q]) return k;
    const int t = r / cin, ci = r - t * cin, co = t / 9, tap = t - co * 9;
    return l.off[q] + ((int64_t)(ci / 32 * 9 + tap) * l.cout[q] + co) * 32 + ci % 32;
}
static __device__ __forceinline__ void put_packed(const WeightList& l, int64_t k, float4 p,
                                                  bf16* __restrict__ pb) {
    *reinterpret_cast<bf16x4p*>(pb + packed_at(l, k)) =
        bf16x4p{(bf16)p.x, (bf16)p.y, (bf16)p.z, (bf16)p.w};
}

// Adam on fp32 master weights; refreshes the bf16 copy used by the kernels.  Four
// parameters a thread (n a multiple of 4), so that finding their place in the copy,
// two divisions, is a small part: 12 us for the 1 955 240 of a network with one a
// thread and no place to find, 21 with it, 12 now.
__global__ void __launch_bounds__(256)
k_adam(WeightList l, int64_t n, float* __restrict__ p, const float* __restrict__ g,
       float* __restrict__ m, float* __restrict__ v, bf16* __restrict__ pb, float lr, float b1,
       float b2, float eps, float c1, float c2, float clip)
{
    const int64_t k = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (k >= n) return;
    const float4 g4 = *reinterpret_cast<const float4*>(g + k);
    float4 m4 = *reinterpret_cast<const float4*>(m + k), v4 = *reinterpret_cast<const float4*>(v + k);
    float4 p4 = *reinterpret_cast<const float4*>(p + k);
    auto step = [&](float gk, float& mq, float& vq, float& pq) {
        gk = gk * clip;
        const float mk = b1 * mq + (1.f - b1) * gk;
        const float vk = b2 * vq + (1.f - b2) * gk * gk;
        mq = mk;
        vq = vk;
        const float upd = lr * (mk / c1) / (sqrtf(vk / c2) + eps);
        pq -= upd;
    };
    step(g4.x, m4.x, v4.x, p4.x);
    step(g4.y, m4.y, v4.y, p4.y);
    step(g4.z, m4.z, v4.z, p4.z);
    step(g4.w, m4.w, v4.w, p4.w);
    *reinterpret_cast<float4*>(m + k) = m4;
    *reinterpret_cast<float4*>(v + k) = v4;
    *reinterpret_cast<float4*>(p + k) = p4;
    put_packed(l, k, p4, pb);
}

__global__ void __launch_bounds__(256)
k_to_bf16(WeightList l, int64_t n, const float* __restrict__ x, bf16* __restrict__ y)
{
    const int64_t k = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (k < n) put_packed(l, k, *reinterpret_cast<const float4*>(x + k), y);
}

// ------------------------------------------------------------ launchers

static inline unsigned nblk(int64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

template <int TW, int TH, int WN>
static void conv_tile(hipStream_t st, const ConvIn& src, const bf16* w, const float* bias,
                      bf16* out, float* out32, int cout, int nb, int H, int W, int flags) {
    const unsigned tiles = (unsigned)(((W + TW - 1) / TW) * ((H + TH - 1) / TH) * nb);
    const unsigned nblocks = tiles * (unsigned)(cout / (32 * WN));
    // small layers (fewer workgroups than CUs, e.g. the deep levels of a small
    // batch): split the input channels over up to 4 blocks per tile, each with
    // at least two 32-channel slices, writing its partial sums to its own
    // slice of the scratch.  From one workgroup per CU up, the finishing pass
    // costs more than the split gains.
    const int nsl = (src.ca + src.cb) / 32;
    const int64_t nout = (int64_t)nb * H * W * cout;
    int ks = 1;
    if (src.acc32 && nblocks < 256 && !src.head_y)
        while (ks < 4 && nblocks * ks < 1024 && nsl / (2 * ks) >= 2 &&
               2 * ks * nout <= src.acc_cap)
            ks *= 2;
    dim3 grid(tiles, cout / (32 * WN), ks);
    const bool pool = src.mode == IN_POOL, pipe = nsl / ks >= 3 && nblocks * ks <= 512;
#define STM_CONV_TILE(P, Q)                                                                    \
    k_conv3x3_tile<TW, TH, WN, P, Q><<<grid, 256, 0, st>>>(src, w, bias, out, out32, cout, nb, H, \
                                                           W, flags)
    if (pool && pipe) STM_CONV_TILE(true, true);
    else if (pool) STM_CONV_TILE(true, false);
    else if (pipe) STM_CONV_TILE(false, true);
    else STM_CONV_TILE(false, false);
#undef STM_CONV_TILE
    if (ks > 1)
        k_conv_finish<<<nblk(nout / 4), 256, 0, st>>>(src.acc32, ks, bias, out, out32, nout, cout,
                                                  flags, src.live, (int64_t)H * W * cout);
}

bool conv_tiles_fit(int H, int W) { return W % 8 == 0 && H % 8 == 0; }

void conv3x3_in(hipStream_t st, const ConvIn& src, const bf16* w, const float* bias, bf16* out,
                float* out32, int cout, int nb, int H, int W, int flags) {
    // two N blocks per workgroup only where that still leaves >= 512 workgroups
    const int64_t pix = (int64_t)nb * H * W;
    const bool n64 = cout % 64 == 0 && (pix / 128) * (cout / 64) >= 512;
    if (W % 16 == 0) {
        if (n64) conv_tile<16, 8, 2>(st, src, w, bias, out, out32, cout, nb, H, W, flags);
        else conv_tile<16, 8, 1>(st, src, w, bias, out, out32, cout, nb, H, W, flags);
    } else if (H % 16 == 0) {
        if (n64) conv_tile<8, 16, 2>(st, src, w, bias, out, out32, cout, nb, H, W, flags);
        else conv_tile<8, 16, 1>(st, src, w, bias, out, out32, cout, nb, H, W, flags);
    } else {   // 8 x 8 tiles of 64 pixels
        conv_tile<8, 8, 1>(st, src, w, bias, out, out32, cout, nb, H, W, flags);
    }
}

void conv3x3(hipStream_t st, const bf16* in, int cin, const bf16* w, const float* bias, bf16* out,
             float* out32, int cout, int nb, int H, int W, int flags, const int* live) {
    const int64_t npix = (int64_t)nb * H * W;
    if (conv_tiles_fit(H, W)) {
        const ConvIn src{in, cin, IN_DIRECT, nullptr, 0, live};
        conv3x3_in(st, src, w, bias, out, out32, cout, nb, H, W, flags);
        return;
    }
    if (H * W <= SMALL_PIXELS && small_patch_bytes(cin, H, W) <= SMALL_LDS) {
        const int mt = H * W <= 16 ? 1 : H * W <= 32 ? 2 : 4;
        dim3 grid(nb, (cout / 16 + 4 / mt - 1) / (4 / mt));
        k_conv3x3_small<<<grid, 256, small_patch_bytes(cin, H, W), st>>>(
            in, cin, w, bias, out, out32, cout, H, W, mt, flags, live);
        return;
    }
    if (npix >= 64 * 256) {
        dim3 grid(nblk(npix, 128), (cout + 63) / 64);
        k_conv3x3<128><<<grid, 256, 0, st>>>(in, cin, w, bias, out, out32, cout, nb, H, W, flags,
                                             live);
    } else {
        dim3 grid(nblk(npix, 64), (cout + 63) / 64);
        k_conv3x3<64><<<grid, 256, 0, st>>>(in, cin, w, bias, out, out32, cout, nb, H, W, flags,
                                            live);
    }
}
void weight_flip(hipStream_t st, FlipList& l, const bf16* w, bf16* wt) {
    unsigned n = 0;
    for (int k = 0; k < l.n; k++) {
        l.block[k] = n;
        n += (unsigned)(l.cin[k] / 32 * 9 * (l.cout[k] / 32));
    }
    k_weight_flip<<<n, 256, 0, st>>>(l, w, wt);
}
void relu_bias_bwd(hipStream_t st, const bf16* y, bf16* g, int c, int64_t npix, float* bpart) {
    // at most about one block per CU, so the sums of their partials stay short
    k_relu_bias_bwd<<<(int)bias_blocks(npix), 256, 0, st>>>(y, g, c, (int)npix,
                                                           bias_pixels_per_block(npix), bpart);
}
void conv3x3_dw(hipStream_t st, const DwLayer* layers, int n, float* grads, float* part) {
    // the channels in tiles of 64, and of 32 what is left: a launch per kind of tile
    auto launch = [&](auto kernel, int co, int ci) {
        DwList l;
        unsigned blocks = 0;
        for (int k = 0; k < n; k++) {
            const DwLayer& d = layers[k];
            const int wide = d.cin / 64 * 64, left = d.cin - wide;
            if ((d.cout % 64 == 0) != (co == 64) || (ci == 64 ? wide : left) == 0) continue;
            DwLayer& o = l.layer[l.n];
            o = d;
            const int64_t npix = (int64_t)d.nb * d.H * d.W, nw = (int64_t)d.cout * 9 * d.cin;
            const int chunks = (int)dw_chunks(npix);
            o.per = dw_pixels_per_chunk(npix);
            o.ci_first = ci == 64 ? 0 : wide;
            o.ntile_ci = (ci == 64 ? wide : left) / ci;
            o.out = chunks == 1 ? grads + d.woff : part + d.poff;
            o.chunk_stride = chunks == 1 ? 0 : nw;
            l.block[l.n++] = blocks;
            blocks += (unsigned)(o.ntile_ci * (d.cout / co) * 3 * chunks);
        }
        if (blocks) kernel<<<blocks, 256, 0, st>>>(l);
    };
    launch(k_conv3x3_dw<64, 64>, 64, 64);
    launch(k_conv3x3_dw<64, 32>, 64, 32);
    launch(k_conv3x3_dw<32, 64>, 32, 64);
    launch(k_conv3x3_dw<32, 32>, 32, 32);
}
void grad_finish(hipStream_t st, GradList& l, const float* part, const float* bpart,
                 float* grads) {
    unsigned n = 0;
    for (int k = 0; k < l.n; k++) {
        l.block[k] = n;
        l.chunks[k] = (int)dw_chunks(l.npix[k]);
        l.bblocks[k] = (int)bias_blocks(l.npix[k]);
        n += l.cout[k] + (l.chunks[k] > 1 ? nblk((int64_t)l.cout[k] * 9 * l.cin[k] / 4) : 0);
    }
    k_grad_finish<<<n, 256, 0, st>>>(l, part, bpart, grads);
}
void maxpool(hipStream_t st, const bf16* x, bf16* y, int nb, int H, int W, int c, const int* live) {
    k_maxpool<<<nblk((int64_t)nb * H * W * c / 32), 256, 0, st>>>(x, y, nb, H, W, c, live);
}
void maxpool_bwd(hipStream_t st, const bf16* x, const bf16* y, const bf16* gy, bf16* gx, int nb,
                 int H, int W, int c) {
    k_maxpool_bwd<<<nblk((int64_t)nb * H * W * c / 32), 256, 0, st>>>(x, y, gy, gx, nb, H, W, c);
}
void join(hipStream_t st, const bf16* x, int ca, const bf16* s, int cb, bf16* y, int nb, int H,
          int W, const int* live) {
    k_join<<<nblk((int64_t)nb * H * W * (ca + cb) / 8), 256, 0, st>>>(x, ca, s, cb, y, nb, H, W,
                                                                      live);
}
void join_bwd(hipStream_t st, const bf16* gy, bf16* gx, int ca, bf16* gs, int cb, int nb, int H,
              int W) {
    k_join_bwd<<<nblk((int64_t)nb * H * W * (ca + cb) / 32), 256, 0, st>>>(gy, gx, ca, gs, cb, nb, H,
                                                                           W);
}
void head(hipStream_t st, const bf16* x, int c, const float* w, const float* b, float* y,
          int64_t npix, const int* live, int64_t hw) {
    k_head<<<nblk(npix), 256, 0, st>>>(x, c, w, b, y, npix, live, hw);
}
void head_bwd(hipStream_t st, const bf16* x, const float* w, const float* gy, bf16* gx,
              float* dw, float* db, int64_t npix, float* part) {
    const int nblocks = (int)nblk(npix);
    k_head_bwd<<<nblocks, 256, 0, st>>>(x, w, gy, gx, part, npix);
    k_block_sum<<<1, 256, 0, st>>>(part, nblocks, 33, 0, db, 1);
    k_block_sum<<<32, 256, 0, st>>>(part, nblocks, 33, 1, dw, 1);
}
void loss(hipStream_t st, const float* y, const float* t, const float* m, float* denom, float* gy,
          float* loss_out, int64_t npix_per, int nb, float* part) {
    k_target_norm<<<dim3(64, nb), 256, 0, st>>>(t, m, part, npix_per);
    k_block_sum<<<nb, 256, 0, st>>>(part, 64, nb, 0, denom, 0);
    const int nblocks = (int)nblk(npix_per * nb);
    k_loss<<<nblocks, 256, 0, st>>>(y, t, m, denom, gy, part, npix_per, nb);
    k_block_sum<<<1, 256, 0, st>>>(part, nblocks, 1, 0, loss_out, 1);
}
void adam(hipStream_t st, const WeightList& l, int64_t n, float* p, const float* g, float* m, float* v, bf16* pb,
          float lr, float b1, float b2, float eps, int step, float clip) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    k_adam<<<nblk(n / 4), 256, 0, st>>>(l, n, p, g, m, v, pb, lr, b1, b2, eps, c1, c2, clip);
}
void to_bf16(hipStream_t st, const WeightList& l, int64_t n, const float* x, bf16* y) {
    k_to_bf16<<<nblk(n / 4), 256, 0, st>>>(l, n, x, y);
}

}  // namespace nn
}  // namespace stm
