// HIP kernels of the polar-ring 2D alignment path for CDNA4 (gfx950, wave64).
//
// Data layout in HBM:
//   images       [n][D][D] float32, row-major (y, x)
//   spec         [n][S][R][128] float2: raw ring spectra of every image at every
//                grid shift, slot 0 = (X[0], X[128]), slot k = X[k], k=1..127; the
//                order of the slots' parts within a row is slot_re's
//   norm         [n][S] float2 = (mu*L, 1/(sd+1e-7)) of the radius-weighted
//                normalisation (reference cuda/gpu_aln_noref.cu:1294-1351)
//   rspec        [N][R][128] float2: reference spectra, normalised and weighted (i+1),
//                rows as those of spec
//   rec          PeakRec per (particle, reference)
// The reference's psi-CCF table (particles x refs x shifts x 2 x (L+2) floats,
// cuda/gpu_aln_noref.cu:2343-2461) is never materialised: the contraction over
// rings, the psi inverse FFT of both mirrors and the first-max-wins search run
// fused in registers / LDS of one wavefront.
#include "isac_internal.h"

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <type_traits>
#include <utility>

namespace isac {
namespace {

constexpr int kWave = 64;

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float2 f2(float x, float y) { return make_float2(x, y); }

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return f2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ float2 shfl2(float2 v, int src) {
    return f2(__shfl(v.x, src, kWave), __shfl(v.y, src, kWave));
}

// Radix-4 butterfly: forward Y_m = sum_r v_r e^{-2 pi i rm/4}; INV uses e^{+}.
template <bool INV>
__device__ __forceinline__ void radix4(float2 (&v)[4]) {
    const float2 a0 = f2(v[0].x + v[2].x, v[0].y + v[2].y);
    const float2 a1 = f2(v[0].x - v[2].x, v[0].y - v[2].y);
    const float2 a2 = f2(v[1].x + v[3].x, v[1].y + v[3].y);
    const float2 a3 = f2(v[1].x - v[3].x, v[1].y - v[3].y);
    v[0] = f2(a0.x + a2.x, a0.y + a2.y);
    v[2] = f2(a0.x - a2.x, a0.y - a2.y);
    if (!INV) {  // a1 -/+ i a3
        v[1] = f2(a1.x + a3.y, a1.y - a3.x);
        v[3] = f2(a1.x - a3.y, a1.y + a3.x);
    } else {
        v[1] = f2(a1.x - a3.y, a1.y + a3.x);
        v[3] = f2(a1.x + a3.y, a1.y - a3.x);
    }
}

// Position of element a of a wave's 256-float2 exchange buffer: a ^ ((a >> 2) & 31).
// Every access pattern of fft256_wave (4 l + q, l + 64 q, and the two stage
// writes) then hits 32 distinct bank pairs per half-wavefront.
__device__ __forceinline__ int fswz(int a) { return a ^ ((a >> 2) & 31); }

// Twiddles of the three Stockham stages, in the order the stages read them
// (entry (q - 1) NS + k of stage NS is e^{-2 pi i q k (64 / NS) / 256}): the
// reads of a stage are consecutive or broadcast, so free of bank conflicts.
constexpr int kFftTw = 3 * (4 + 16 + 64);   // 252 entries
__device__ __forceinline__ void fill_fft_twiddles(float2 *tw, const float2 *twg, int tid,
                                                  int nthreads) {
    for (int i = tid; i < kFftTw; i += nthreads) {
        const int NS = i < 12 ? 4 : i < 60 ? 16 : 64;
        const int j = i - (NS == 4 ? 0 : NS == 16 ? 12 : 60);
        const int q = j / NS + 1, k = j % NS;
        tw[i] = twg[q * k * (64 / NS)];
    }
}

// One Stockham radix-4 stage (Govindaraju et al., SC'08) with sub-transform size NS.
template <bool INV, int NS, bool WRITE>
__device__ __forceinline__ void stockham_stage(float2 (&v)[4], const float2 *in, float2 *out,
                                               const float2 *tw, int lane) {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = in[fswz(lane + 64 * q)];
    const int k = lane & (NS - 1);
    constexpr int off = NS == 4 ? 0 : NS == 16 ? 12 : 60;
#pragma unroll
    for (int q = 1; q < 4; ++q) {
        float2 w = tw[off + (q - 1) * NS + k];
        if (INV) w.y = -w.y;
        v[q] = cmul(v[q], w);
    }
    radix4<INV>(v);
    if (WRITE) {
        const int base = (lane - k) * 4 + k;
#pragma unroll
        for (int q = 0; q < 4; ++q) out[fswz(base + q * NS)] = v[q];
    }
}

// 256-point complex FFT by one wavefront.  In: v[q] = x[lane + 64 q].
// Out: v[q] = X[lane + 64 q] (natural order).  b0/b1: 256-float2 wave-private
// LDS buffers (swizzled, fswz); tw: the stage twiddles of fill_fft_twiddles, in
// LDS.  Unnormalised.
template <bool INV>
__device__ __forceinline__ void fft256_wave(float2 (&v)[4], float2 *b0, float2 *b1,
                                            const float2 *tw, int lane) {
    wave_lds_sync();
    radix4<INV>(v);
#pragma unroll
    for (int q = 0; q < 4; ++q) b0[fswz(4 * lane + q)] = v[q];
    wave_lds_sync();
    stockham_stage<INV, 4, true>(v, b0, b1, tw, lane);
    wave_lds_sync();
    stockham_stage<INV, 16, true>(v, b1, b0, tw, lane);
    wave_lds_sync();
    stockham_stage<INV, 64, false>(v, b0, nullptr, tw, lane);
}

// The four pixels around (x, y), each tap clamped to the image, and the fractions.  The two
// pixels of a row come in one 8-byte load (4-byte aligned) from column clamp(x, 0, D - 2).
struct Quad {
    float2 top, bot;
    float fx, fy;
    int ix;
};
__device__ __forceinline__ Quad load_quad(const float *img, int D, float x, float y) {
    const float x0 = floorf(x), y0 = floorf(y);
    const int ix = (int)x0, iy = (int)y0;
    const int xl = min(max(ix, 0), D - 2);
    const int ya = min(max(iy, 0), D - 1), yb = min(max(iy + 1, 0), D - 1);
    Quad q;
    __builtin_memcpy(&q.top, img + ya * D + xl, sizeof(float2));
    __builtin_memcpy(&q.bot, img + yb * D + xl, sizeof(float2));
    q.fx = x - x0;
    q.fy = y - y0;
    q.ix = ix;
    return q;
}
__device__ __forceinline__ float mix_quad(const Quad &q, int D) {
    const bool left = q.ix < 0, right = q.ix > D - 2;   // both taps on the edge column
    const float v00 = right ? q.top.y : q.top.x, v01 = left ? q.top.x : q.top.y;
    const float v10 = right ? q.bot.y : q.bot.x, v11 = left ? q.bot.x : q.bot.y;
    return (1.0f - q.fy) * ((1.0f - q.fx) * v00 + q.fx * v01) + q.fy * ((1.0f - q.fx) * v10 + q.fx * v11);
}

// Blocks are dispatched round-robin over the 8 XCDs; remap so that consecutive
// logical blocks (which share particle spectra) run on the same XCD and L2.
__device__ __forceinline__ int xcd_remap(int b, int nb) {
    const int q = nb >> 3, r = nb & 7;
    const int xcd = b & 7, idx = b >> 3;
    return (xcd < r) ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

// One slot of a ring row.
__device__ __forceinline__ float2 load_slot(const float2 *row, int k) {
    const float *q = reinterpret_cast<const float *>(row) + slot_re(k);
    return make_float2(q[0], q[kPartOff]);
}

// Transforms over 16 lanes, four per wavefront: the twiddles of the last two stages.
constexpr int kIfftTw = 15 * 16;  // lane twiddles of the last two stages

// entry q - 1: stage 3, e^{-2 pi i 4 q u / 256}; entry 3 + 3 q3 + q - 1: stage 4,
// e^{-2 pi i q (u + 16 q3) / 256}
__device__ __forceinline__ void fill_ifft_twiddles(float2 *tw, const float2 *twg, int tid, int nthreads) {
    for (int i = tid; i < kIfftTw; i += nthreads) {
        const int e = i >> 4, u = i & 15;
        tw[i] = e < 3 ? twg[4 * (e + 1) * u] : twg[((e - 3) % 3 + 1) * (u + 16 * ((e - 3) / 3))];
    }
}

// v conj(w), with the operation order of cmul under INV
__device__ __forceinline__ float2 cmulc(float2 v, float2 w) {
    return f2(fmaf(v.x, w.x, v.y * w.y), fmaf(v.y, w.x, -(v.x * w.y)));
}

// cos, sin of -2 pi m / 256 for the m = 16 q k of the second stage (the table's values)
__device__ __forceinline__ constexpr float2 stage2_tw(int m) {
    return m == 16    ? float2{0.92387953251128674f, -0.38268343236508977f}
           : m == 32  ? float2{0.70710678118654757f, -0.70710678118654757f}
           : m == 48  ? float2{0.38268343236508984f, -0.92387953251128674f}
           : m == 64  ? float2{6.123233995736766e-17f, -1.0f}
           : m == 96  ? float2{-0.70710678118654746f, -0.70710678118654757f}
                      : float2{-0.92387953251128685f, 0.38268343236508967f};   // m == 144
}

// v w, the rounding of cmul
__device__ __forceinline__ float2 cmulf(float2 v, float2 w) {
    return f2(fmaf(v.x, w.x, -(v.y * w.y)), fmaf(v.y, w.x, v.x * w.y));
}

// Last two radix-4 stages of a 256-point transform over 16 lanes, x[a] = point u + 16 a
// after the second stage in, natural order u + 16 m out.
template <bool INV>
__device__ __forceinline__ void fft256_tail(float2 (&x)[16], const float2 *tw, int u) {
    float2 w3[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) w3[q] = tw[q * 16 + u];
#pragma unroll
    for (int h = 0; h < 4; ++h) {      // stage 3, butterfly 16 h + u
        float2 v[4] = {x[h], x[h + 4], x[h + 8], x[h + 12]};
#pragma unroll
        for (int q = 1; q < 4; ++q) v[q] = INV ? cmulc(v[q], w3[q - 1]) : cmulf(v[q], w3[q - 1]);
        radix4<INV>(v);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[h + 4 * q] = v[q];
    }
#pragma unroll
    for (int q3 = 0; q3 < 4; ++q3) {   // stage 4, butterfly u + 16 q3
        float2 v[4] = {x[4 * q3], x[4 * q3 + 1], x[4 * q3 + 2], x[4 * q3 + 3]};
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            const float2 w4 = tw[(3 + 3 * q3 + q - 1) * 16 + u];
            v[q] = INV ? cmulc(v[q], w4) : cmulf(v[q], w4);
        }
        radix4<INV>(v);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[4 * q3 + q] = v[q];
    }
    // x[4 q3 + q] = z[u + 16 q3 + 64 q]: to natural order
    float2 y[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) y[m] = x[4 * (m & 3) + (m >> 2)];
#pragma unroll
    for (int m = 0; m < 16; ++m) x[m] = y[m];
}

// ------------------------------------------------------------------ stage A
// Ring FFTs, four per wavefront: 16 lanes each, lane u holds points u + 16 m.  The
// radix-4 stages run in pairs inside a lane with one LDS exchange between (real, then
// imaginary parts, kXchLd floats per transform), in the arithmetic of the Stockham
// stages (inputs, twiddles, operation order).
constexpr int kXchLd = 276;       // floats per transform (two lane rows hit 32 distinct banks)

// 16 x 16 transpose within each lane row: in x[4 k + q] = point 16 u + k + 4 q, out
// x[a] = point u + 16 a.  xb: the lane row's kXchLd floats, free to overwrite.
__device__ __forceinline__ void row_exchange(float2 (&x)[16], float *xb, int u) {
    float *xw = xb + 17 * u;
    const float *xr = xb + u;
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) xw[k + 4 * q] = x[4 * k + q].x;
    wave_lds_sync();
    float re[16];
#pragma unroll
    for (int a = 0; a < 16; ++a) re[a] = xr[17 * a];
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) xw[k + 4 * q] = x[4 * k + q].y;
    wave_lds_sync();
#pragma unroll
    for (int a = 0; a < 16; ++a) x[a] = f2(re[a], xr[17 * a]);
}

// Forward transform, x[m] = point u + 16 m in and out.
__device__ __forceinline__ void fft256_rows4(float2 (&x)[16], float *xb, const float2 *tw, int u) {
#pragma unroll
    for (int q2 = 0; q2 < 4; ++q2) {   // stage 1, butterfly u + 16 q2
        float2 v[4] = {x[q2], x[q2 + 4], x[q2 + 8], x[q2 + 12]};
        radix4<false>(v);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q2 + 4 * q] = v[q];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {      // stage 2, butterfly 4 u + k
        float2 v[4] = {x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
        if (k > 0) {
#pragma unroll
            for (int q = 1; q < 4; ++q) v[q] = cmulf(v[q], stage2_tw(16 * q * k));
        }
        radix4<false>(v);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[4 * k + q] = v[q];
    }
    row_exchange(x, xb, u);
    fft256_tail<false>(x, tw, u);
}

// Spectra of the two real rings of a transform Z = FFT(ring a + i ring b): lane u's slots
// k = u + 16 m, m < 8, from Z[k] and Z[256 - k] (in lane (16 - u) & 15, through LDS).
// Slot 0 packs the real bins 0 and 128.
__device__ __forceinline__ void unpack_rings(const float2 (&z)[16], float2 (&a)[8], float2 (&b)[8], float *xb,
                                             int u) {
    // Z[128 + i] at 2 i; Z[256 - k] = entry 128 - k = (16 - u) + 16 (7 - m)
    float2 *hw = reinterpret_cast<float2 *>(xb) + u;
    const float2 *hr = reinterpret_cast<const float2 *>(xb) + (16 - u);
    wave_lds_sync();
#pragma unroll
    for (int m = 0; m < 8; ++m) hw[16 * m] = z[8 + m];
    wave_lds_sync();
    float2 p[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) p[m] = hr[16 * (7 - m)];   // entry 128 (u = 0, m = 0) is not used
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        a[m] = f2(0.5f * (z[m].x + p[m].x), 0.5f * (z[m].y - p[m].y));
        b[m] = f2(0.5f * (z[m].y + p[m].y), 0.5f * (p[m].x - z[m].x));
    }
    if (u == 0) {
        a[0] = f2(z[0].x, z[8].x);
        b[0] = f2(z[0].y, z[8].y);
    }
}

// Bilinear sample at (x, y) of an LDS copy of the image with a one-pixel border that
// repeats the edge (pitch W = D + 2): the cell is clamped to -1 .. D - 1, where both taps
// of a row read the same edge values as clamping each tap.  img1 points at pixel (0, 0).
__device__ __forceinline__ float tap(const float *img1, float Wf, float lim, int W, float x, float y) {
    const float x0 = floorf(x), y0 = floorf(y);
    const float fx = x - x0, fy = y - y0;
    const float cx = __builtin_amdgcn_fmed3f(x0, -1.0f, lim), cy = __builtin_amdgcn_fmed3f(y0, -1.0f, lim);
    const float *q = img1 + (int)fmaf(cy, Wf, cx);   // exact: below 2^24
    const float v00 = q[0], v01 = q[1], v10 = q[W], v11 = q[W + 1];
    const float gx = 1.0f - fx, gy = 1.0f - fy;
    const float top = fmaf(fx, v01, v00 * gx), bot = fmaf(gx, v10, fx * v11);
    return fmaf(gy, top, fy * bot);
}

__device__ __forceinline__ double row_sum(double v) {   // over each row of 16 lanes
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// (mu L, 1 / (sd + 1e-7)) from the radius-weighted sum and sum of squares
__device__ __forceinline__ float2 ring_norm(double a, double q, int R) {
    const double nn = (double)kRingLen * 0.5 * (double)R * (double)(R + 1);
    const double mu = a / nn;
    const double sd = sqrt(fabs(q / nn - mu * mu));
    return f2((float)(mu * kRingLen), (float)(1.0 / (sd + 1e-7)));
}

// LDS floats of a polar kernel with nw wavefronts: lane twiddles, exchange buffers, image.
__host__ __device__ constexpr int polar_lds_floats(int D, int nw) {
    return 2 * kIfftTw + nw * 4 * kXchLd + (D + 2) * (D + 2);
}

// Bordered copy of an image (see tap), all threads; the caller synchronises.
__device__ __forceinline__ void load_bordered(float *img, const float *src, int D) {
    const int W = D + 2;
    for (int r = threadIdx.x >> 6; r < W; r += blockDim.x >> 6) {
        const float *s = src + min(max(r - 1, 0), D - 1) * D;
        for (int c = threadIdx.x & 63; c < W; c += 64) img[r * W + c] = s[min(max(c - 1, 0), D - 1)];
    }
}

// Samples and transform of ring pair (i, i + 1) of one row about (cx, cy): lane u takes
// angles u + 16 m; spectra of both rings out (b = 0 past R).  Returns the lane's part of the
// pair's sums (FP64).  A lane's parts are added in ring order from 0, then its row's lanes,
// whichever wavefronts took the pairs: a row's sums do not depend on the launch's shape.  (A
// variance far below the mean's square shows any other order.)
__device__ __forceinline__ double2 ring_pair(const float *img1, float Wf, float lim, int W, const float2 *tmpl, int i,
                                             int R, float cx, float cy, int u, float *xb, const float2 *tw,
                                             float2 (&a)[8], float2 (&b)[8]) {
    float2 x[16];
    const float2 *ta = tmpl + (size_t)i * kRingLen + u;
    double a1 = 0.0, a2 = 0.0, b1 = 0.0, b2 = 0.0;
    const bool hb = i + 1 < R;   // uniform over the lane row
    const float2 *tb = hb ? ta + kRingLen : ta;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const float2 pa = ta[16 * m], pb = tb[16 * m];
        const float va = tap(img1, Wf, lim, W, cx + pa.x, cy + pa.y);
        const float t = tap(img1, Wf, lim, W, cx + pb.x, cy + pb.y);
        const float vb = hb ? t : 0.0f;
        x[m] = f2(va, vb);
        const double da = va, db = vb;
        a1 += da;
        a2 = fma(da, da, a2);
        b1 += db;
        b2 = fma(db, db, b2);
    }
    const double wa = (double)(i + 1), wb = (double)(i + 2);
    const double2 sum = make_double2(fma(wa, a1, wb * b1), fma(wa, a2, wb * b2));
    fft256_rows4(x, xb, tw, u);
    unpack_rings(x, a, b, xb, u);
    return sum;
}

// A lane's slots u + 16 m of one ring row: four 16-byte accesses (slot_re).
__device__ __forceinline__ void store_slots(float2 *row, const float2 (&a)[8], int u) {
    float4 *o = reinterpret_cast<float4 *>(row) + 2 * u;
#pragma unroll
    for (int mh = 0; mh < 2; ++mh) {
        o[32 * mh] = make_float4(a[4 * mh].x, a[4 * mh + 1].x, a[4 * mh + 2].x, a[4 * mh + 3].x);
        o[32 * mh + 1] = make_float4(a[4 * mh].y, a[4 * mh + 1].y, a[4 * mh + 2].y, a[4 * mh + 3].y);
    }
}

// Raw ring spectra of an image at every grid shift.  Workgroup = one image (staged once in
// LDS) and `rows` of its rows (shifts) from blockIdx.y * rows on.  MASKED: only the shifts
// whose bit is set in smask[p] (S <= 64) are computed, all by one workgroup; the other rows
// of spec / norm are left as they were.
// Unspread, a wavefront takes four rows at a time, one per 16 lanes, and their ring pairs in
// turn.  SPREAD, the pairs of all rows go round over the 16-lane groups, and a lane's parts
// of a row's sums come together in LDS after each round: no lanes without a row and no
// wavefronts without a group of four, for two barriers a round.
// What bounds it: vector instructions (about 25 a sample with its FP64 sums, 20 a point
// of the transform) and the writes; 6000 images of 76 x 76, 49 shifts, 34 rings, 10.2 GB:
// 3.5 ms, 2.7 without the stores, 2.7 with stores but no transforms.  A transform over 64
// lanes with an exchange at each stage made it 3.9.  Four wavefronts per SIMD (128
// registers) are needed to hide the taps.  Unspread / spread: 8000 images of 100 x 100, 1
// shift 1.93 / 0.39 ms, 5000 of 128 x 128, 9 shifts 3.23 / 1.36, 3000 of 128 x 128, 25 shifts
// 2.51 / 1.94, 10000 of 76 x 76, 9 shifts 1.55 / 1.36, 25 shifts of 5000 1.61 / 1.69, 49 shifts
// of 5000 3.05 / 3.28.
template <bool MASKED, bool SPREAD>
__global__ __launch_bounds__(1024, 4) void k_polar_spectra(
    const float *__restrict__ imgs, int D, ShiftView acc, const int2 *__restrict__ shift_i,
    int S, const float2 *__restrict__ tmpl, int R, const float2 *__restrict__ twg,
    float2 *__restrict__ spec, float2 *__restrict__ norm,
    const unsigned long long *__restrict__ smask, int rows) {
    extern __shared__ float4 smem4[];
    __shared__ int slist[64];
    __shared__ int scnt;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = blockDim.x >> 6, f = lane >> 4, u = lane & 15;
    const int p = blockIdx.x;
    if (MASKED && smask[p] == 0ull) return;   // uniform over the workgroup
    float2 *tw = reinterpret_cast<float2 *>(smem4);
    float *xb0 = reinterpret_cast<float *>(tw + kIfftTw);
    float *xb = xb0 + (wave * 4 + f) * kXchLd, *img = xb0 + nw * 4 * kXchLd;
    const int W = D + 2;
    load_bordered(img, imgs + (size_t)p * D * D, D);
    fill_ifft_twiddles(tw, twg, tid, blockDim.x);
    if (MASKED && tid == 0) {
        const unsigned long long mk = smask[p];
        int c = 0;
        for (int b = 0; b < S && b < 64; ++b)
            if ((mk >> b) & 1ull) slist[c++] = b;
        scnt = c;
    }
    __syncthreads();
    const int row0 = MASKED ? 0 : blockIdx.y * rows;
    const int n_rows = MASKED ? scnt : min(rows, S - row0);
    const int pairs = (R + 1) / 2, slots = 4 * nw;
    float ax = 0.0f, ay = 0.0f;
    if (acc.base) {
        ax = acc.base[(size_t)p * acc.stride];
        ay = acc.base[(size_t)p * acc.stride + 1];
    }
    const float *img1 = img + W + 1;
    const float Wf = (float)W, lim = (float)(D - 1);
    auto shift_of = [&](int j) { return MASKED ? slist[j] : row0 + j; };
    if (!SPREAD) {
        for (int j0 = 4 * wave; j0 < n_rows; j0 += slots) {
            const bool live = j0 + f < n_rows;   // lanes past the last row repeat it, without its stores
            const int s = shift_of(min(j0 + f, n_rows - 1));
            const int2 si = shift_i[s];
            const float cx = (float)(D / 2 + si.x) + ax, cy = (float)(D / 2 + si.y) + ay;
            double sA = 0.0, sQ = 0.0;
            float2 *row = spec + ((size_t)p * S + s) * (size_t)R * kSlots;
            for (int i = 0; i < R; i += 2) {
                float2 a[8], b[8];
                const double2 t = ring_pair(img1, Wf, lim, W, tmpl, i, R, cx, cy, u, xb, tw, a, b);
                sA += t.x;
                sQ += t.y;
                if (live) {
                    store_slots(row + (size_t)i * kSlots, a, u);
                    if (i + 1 < R) store_slots(row + (size_t)(i + 1) * kSlots, b, u);
                }
            }
            sA = row_sum(sA);
            sQ = row_sum(sQ);
            if (live && u == 0) norm[(size_t)p * S + s] = ring_norm(sA, sQ, R);
        }
        return;
    }
    // task t: ring pair t % pairs of row t / pairs, on slot t % slots
    const int slot = 4 * wave + f, n_task = n_rows * pairs;
    double sA = 0.0, sQ = 0.0;   // of the row that this slot adds up: rows slot, slot + slots, ..
    for (int t0 = 0; t0 < n_task; t0 += slots) {
        const int t1 = min(t0 + slots, n_task);
        if (t0 + 4 * wave < t1) {   // uniform over the wavefront
            const int t = min(t0 + slot, t1 - 1);   // lanes past the last task repeat it, without its stores
            const bool live = t0 + slot < t1;
            const int j = t / pairs, i = 2 * (t - j * pairs);
            const int s = shift_of(j);
            const int2 si = shift_i[s];
            const float cx = (float)(D / 2 + si.x) + ax, cy = (float)(D / 2 + si.y) + ay;
            float2 a[8], b[8];
            const double2 part = ring_pair(img1, Wf, lim, W, tmpl, i, R, cx, cy, u, xb, tw, a, b);
            if (live) {
                float2 *row = spec + (((size_t)p * S + s) * (size_t)R + i) * kSlots;
                store_slots(row, a, u);
                if (i + 1 < R) store_slots(row + kSlots, b, u);
            }
            wave_lds_sync();
            reinterpret_cast<double2 *>(xb)[u] = part;   // the exchange buffer is free until the next round
        }
        __syncthreads();
        // the row of this slot that has tasks in this round, if any: they are in ring order
        const int ja = t0 / pairs, jb = (t1 - 1) / pairs;
        const int j = ja + (slot + slots - ja % slots) % slots;
        if (j <= jb) {
            const int ta = max(j * pairs, t0), tb = min((j + 1) * pairs, t1);
            const float *q = xb0 + (ta - t0) * kXchLd + 4 * u;
            int n = tb - ta;
            for (; n >= 4; n -= 4, q += 4 * kXchLd) {   // four loads in flight
                double2 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const double2 *>(q + k * kXchLd);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    sA += v[k].x;
                    sQ += v[k].y;
                }
            }
            for (; n > 0; --n, q += kXchLd) {
                const double2 v = *reinterpret_cast<const double2 *>(q);
                sA += v.x;
                sQ += v.y;
            }
            if (tb == (j + 1) * pairs) {
                sA = row_sum(sA);
                sQ = row_sum(sQ);
                if (u == 0) norm[(size_t)p * S + shift_of(j)] = ring_norm(sA, sQ, R);
                sA = sQ = 0.0;
            }
        }
        __syncthreads();
    }
}

// Reference spectra (centre D / 2, no shift), normalised and multiplied by the ring
// weight i + 1; rsum0[n] = sum of slot 0's real parts (the particle DC correction).
// Workgroup = one reference, one ring pair per 16 lanes (up to 64 pairs), so the
// transforms of all its rings run at once and stay in registers until the sums are
// complete: a search of few references waits for one such pass.  5 references of
// 64 x 64, 29 rings: 12 us, 100 of 76 x 76, 34 rings: 21 us; with four wavefronts for all
// rings and a normalising pass the 5 took 25 + 6.
__global__ __launch_bounds__(1024) void k_ref_spectra(const float *__restrict__ imgs, int D,
                                                      const float2 *__restrict__ tmpl, int R,
                                                      const float2 *__restrict__ twg, float2 *__restrict__ rspec,
                                                      float *__restrict__ rsum0) {
    extern __shared__ float4 smem4[];
    __shared__ double red[2][64];
    __shared__ float dc[2 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = blockDim.x >> 6, f = lane >> 4, u = lane & 15;
    const int n = blockIdx.x, W = D + 2;
    float2 *tw = reinterpret_cast<float2 *>(smem4);
    float *xb = reinterpret_cast<float *>(tw + kIfftTw) + (wave * 4 + f) * kXchLd;
    float *img = reinterpret_cast<float *>(tw + kIfftTw) + nw * 4 * kXchLd;
    load_bordered(img, imgs + (size_t)n * D * D, D);
    fill_ifft_twiddles(tw, twg, tid, blockDim.x);
    __syncthreads();
    const int i = 2 * (4 * wave + f);
    const bool live = i < R;
    float2 a[8], b[8];
    const float c = (float)(D / 2);
    const double2 t = ring_pair(img + W + 1, (float)W, (float)(D - 1), W, tmpl, live ? i : 0, R, c, c, u, xb, tw, a, b);
    const double sA = row_sum(t.x), sQ = row_sum(t.y);
    if (u == 0) {
        red[0][4 * wave + f] = live ? sA : 0.0;
        red[1][4 * wave + f] = live ? sQ : 0.0;
    }
    __syncthreads();
    double tA = 0.0, tQ = 0.0;
    for (int k = 0; k < 4 * nw; ++k) {
        tA += red[0][k];
        tQ += red[1][k];
    }
    const float2 nm = ring_norm(tA, tQ, R);
    auto finish = [&](float2 (&v)[8], int ring) {
        const float gw = nm.y * (float)(ring + 1);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const float re = (m == 0 && u == 0) ? v[m].x - nm.x : v[m].x;
            v[m] = f2(re * gw, v[m].y * gw);
        }
        store_slots(rspec + ((size_t)n * R + ring) * kSlots, v, u);
        if (u == 0) dc[ring] = v[0].x;
    };
    if (live) finish(a, i);
    if (live && i + 1 < R) finish(b, i + 1);
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int k = 0; k < R; ++k) s += (double)dc[k];
        rsum0[n] = (float)s;
    }
}

// Stage A of the mixed-precision search: the normalised ring spectra of every
// image at every grid shift, written directly as 16-bit MFMA operand rows (the
// GEMM layout of kernels_mixed.hip): row p * S_pad + s holds, per slot, the
// parts a = g (Re S + Im S) c_p and b = g (Re S - Im S) c_p over the rings (slot
// 0: a = g (S[0] - mu L) c_p, b = g S[128] c_p), K padded with zeros.  Rows
// s >= S and images p >= n_img (padding of the last group of 16) are zero.
// Workgroup = one image, staged in LDS as (image - m) / s with its own mean and
// standard deviation (so the raw spectra of a row fit FP16 and the DC term needs
// no large cancellation); wavefront w computes rows w, w + 4, ...  A row's raw
// parts (Re + Im, Re - Im) stay in registers as packed FP16 (2 slots x R rings
// per lane) until the row's normalisation sums are complete; the exact row
// normalisation is applied in FP32 at the final conversion, and every slot is
// one contiguous store.  Sampling positions are the centre plus (i + 1)(cos,
// sin) of the lane's four angles; the normalisation sums add FP32 partial sums
// of four samples in FP64.
template <bool BF16>
__device__ __forceinline__ unsigned short frag16(float x) {
    if (BF16) {
        unsigned u = __float_as_uint(x);
        u += 0x7fffu + ((u >> 16) & 1u);
        return (unsigned short)(u >> 16);
    }
    return __builtin_bit_cast(unsigned short, (_Float16)x);
}

__device__ __forceinline__ unsigned h2pack(float lo, float hi) {
    return (unsigned)__builtin_bit_cast(unsigned short, (_Float16)lo) |
           ((unsigned)__builtin_bit_cast(unsigned short, (_Float16)hi) << 16);
}
__device__ __forceinline__ float h2lo(unsigned v) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(v & 0xffffu));
}
__device__ __forceinline__ float h2hi(unsigned v) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(v >> 16));
}

constexpr int kFragMaxRings = 40;
constexpr int kFragBorder = 8;   // border of k_polar_frag's image copy, pixels

template <bool BF16>
__global__ __launch_bounds__(256, 2) void k_polar_frag(
    const float *__restrict__ imgs, int n_img, int D, ShiftView acc,
    const int2 *__restrict__ shift_i, int S, int S_pad, int R, int full16, int tail,
    int slot_bytes, float cp, const float2 *__restrict__ twg, unsigned char *__restrict__ frag) {
    extern __shared__ float4 smem4[];
    __shared__ double red[2][4];
    float2 *tw = reinterpret_cast<float2 *>(smem4);
    float2 *fb = tw + 256;
    float *img = reinterpret_cast<float *>(fb + 4 * 512);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = blockIdx.x;
    const size_t row_bytes = (size_t)kSlots * slot_bytes;
    unsigned char *prow = frag + (size_t)p * S_pad * row_bytes;
    const int n_rows = (p < n_img) ? S : 0;
    // zero rows: shifts S .. S_pad - 1 (and every row of a padding image)
    {
        const size_t zb = (size_t)(S_pad - n_rows) * row_bytes;
        uint4 *z = reinterpret_cast<uint4 *>(prow + (size_t)n_rows * row_bytes);
        for (size_t i = tid; i < zb / 16; i += 256) z[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (n_rows == 0) return;   // uniform over the workgroup
    const float *src = imgs + (size_t)p * D * D;
    // image mean and standard deviation (FP64)
    double s1 = 0.0, s2 = 0.0;
    for (int i = tid; i < D * D; i += 256) {
        const double v = src[i];
        s1 += v;
        s2 += v * v;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        s1 += __shfl_xor(s1, off, kWave);
        s2 += __shfl_xor(s2, off, kWave);
    }
    if (lane == 0) {
        red[0][wave] = s1;
        red[1][wave] = s2;
    }
    __syncthreads();
    const double t1 = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    const double t2 = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    const double im = t1 / (double)(D * D);
    double isd = sqrt(fmax(t2 / (double)(D * D) - im * im, 0.0));
    if (!(isd > 1e-30)) isd = 1.0;
    const float mimg = (float)im, rs = (float)(1.0 / isd);
    // standardised copy with a kFragBorder-pixel border that repeats the edge
    // (cell c of a row holds pixel clamp(c - kFragBorder))
    const int W = D + 2 * kFragBorder;
    for (int i = tid; i < W * W; i += 256) {
        const int r = i / W, c = i - r * W;
        img[i] = (src[min(max(r - kFragBorder, 0), D - 1) * D + min(max(c - kFragBorder, 0), D - 1)] -
                  mimg) * rs;
    }
    fill_fft_twiddles(tw, twg, tid, 256);
    __syncthreads();
    float ax = 0.0f, ay = 0.0f;
    if (acc.base) {
        ax = acc.base[(size_t)p * acc.stride];
        ay = acc.base[(size_t)p * acc.stride + 1];
    }
    float cq[4], sq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sincospif((float)(lane + 64 * q) / 128.0f, &sq[q], &cq[q]);
    float2 *b0 = fb + wave * 512;
    float2 *b1 = b0 + 256;
    const int pl = (64 - lane) & 63;
    const float Wf = (float)W;

    // bilinear sample at (X, Y) of the bordered copy (coordinates include the
    // border).  INSIDE: the caller guarantees 0 <= floor(X), floor(Y) <= W - 2,
    // so the cell index is one exact FP32 multiply-add.  Otherwise the cell is
    // clamped to the copy, which reads the same edge values as clamping each tap
    // to the image.
    auto tap = [&](float X, float Y, auto inside_tag) __attribute__((always_inline)) {
        const float x0 = floorf(X), y0 = floorf(Y);
        const float fx = X - x0, fy = Y - y0;
        const float *q;
        if constexpr (decltype(inside_tag)::value) {
            q = img + (int)fmaf(y0, Wf, x0);
        } else {
            const int cx = min(max((int)x0, 0), W - 2), cy = min(max((int)y0, 0), W - 2);
            q = img + (int)__umul24((unsigned)cy, (unsigned)W) + cx;
        }
        const float v00 = q[0], v01 = q[1], v10 = q[W], v11 = q[W + 1];
        const float t0 = fmaf(fx, v01 - v00, v00), t1 = fmaf(fx, v11 - v10, v10);
        return fmaf(fy, t1 - t0, t0);
    };

    // ring pair (i, i + 1) of one shift row from the lane's samples of both
    // rings: normalisation sums, one complex FFT, both spectra packed as FP16
    // (Re + Im, Re - Im); slot 0: (S[0], S[128])
    auto ring_pair = [&](int i, const float (&va)[4], const float (&vb)[4],
                         unsigned (&sp)[kFragMaxRings][2], double &sA, double &sQ)
        __attribute__((always_inline)) {
        const float ra = (float)(i + 1), rb = (float)(i + 2);
        float2 v[4];
        float pa = 0.f, qa = 0.f, pb = 0.f, qb = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = f2(va[q], vb[q]);
            pa += va[q];
            qa = fmaf(va[q], va[q], qa);
            pb += vb[q];
            qb = fmaf(vb[q], vb[q], qb);
        }
        sA += (double)ra * pa + (double)rb * pb;
        sQ += (double)ra * qa + (double)rb * qb;
        fft256_wave<false>(v, b0, b1, tw, lane);
        const float2 u2 = shfl2(v[2], pl), u3 = shfl2(v[3], pl);
        const float2 zl = v[0], zlp = lane ? u3 : v[0];
        const float2 zh = v[1], zhp = lane ? u2 : v[3];
        const float2 al = f2(0.5f * (zl.x + zlp.x), 0.5f * (zl.y - zlp.y));
        const float2 bl = f2(0.5f * (zl.y + zlp.y), 0.5f * (zlp.x - zl.x));
        const float2 ah = f2(0.5f * (zh.x + zhp.x), 0.5f * (zh.y - zhp.y));
        const float2 bh = f2(0.5f * (zh.y + zhp.y), 0.5f * (zhp.x - zh.x));
        // slot 0 (lane 0) keeps the two real bins (S[0], S[128]) instead of
        // (Re + Im, Re - Im): selected, not branched
        const unsigned na = h2pack(al.x + al.y, al.x - al.y), za = h2pack(zl.x, v[2].x);
        sp[i][0] = lane ? na : za;
        if (i + 1 < kFragMaxRings) {
            const unsigned nb = h2pack(bl.x + bl.y, bl.x - bl.y), zb = h2pack(zl.y, v[2].y);
            sp[i + 1][0] = lane ? nb : zb;
        }
        sp[i][1] = h2pack(ah.x + ah.y, ah.x - ah.y);
        if (i + 1 < kFragMaxRings) sp[i + 1][1] = h2pack(bh.x + bh.y, bh.x - bh.y);
    };

    // row j's normalisation and 16-bit operand stores
    auto store_row = [&](int j, const unsigned (&sp)[kFragMaxRings][2], double sA, double sQ)
        __attribute__((always_inline)) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            sA += __shfl_xor(sA, off, kWave);
            sQ += __shfl_xor(sQ, off, kWave);
        }
        // row statistics of the standardised samples; the row's normalisation of
        // the original image is g = 1 / (isd sd + 1e-7), applied to spectra / rs
        const double nn = (double)kRingLen * 0.5 * (double)R * (double)(R + 1);
        const double mu = sA / nn;
        const double sd = sqrt(fabs(sQ / nn - mu * mu));
        const float gf = (float)(isd / (isd * sd + 1e-7)) * cp;
        const float muL = (float)(mu * kRingLen);
        unsigned char *rowp = prow + (size_t)j * row_bytes;
#pragma unroll
        for (int h = 0; h < 2; ++h) {   // slot lane (h = 0) and lane + 64 (h = 1)
            const int k = lane + 64 * h;
            unsigned char *dst = rowp + (size_t)k * slot_bytes;
            const float dc = (k == 0) ? muL : 0.0f;
#pragma unroll
            for (int ks = 0; ks < (kFragMaxRings + 15) / 16; ++ks) {
                if (ks < full16 + (tail == 16 ? 1 : 0)) {
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                        for (int hh = 0; hh < 2; ++hh) {
                            unsigned e[4];
#pragma unroll
                            for (int jj = 0; jj < 4; ++jj) {
                                unsigned short lo = 0, hi = 0;
                                const int i0 = 16 * ks + 8 * hh + 2 * jj;
                                if (i0 < kFragMaxRings && i0 < R) {
                                    const unsigned v = sp[i0][h];
                                    lo = frag16<BF16>(pt ? h2hi(v) * gf : (h2lo(v) - dc) * gf);
                                }
                                if (i0 + 1 < kFragMaxRings && i0 + 1 < R) {
                                    const unsigned v = sp[i0 + 1][h];
                                    hi = frag16<BF16>(pt ? h2hi(v) * gf : (h2lo(v) - dc) * gf);
                                }
                                e[jj] = lo | ((unsigned)hi << 16);
                            }
                            *reinterpret_cast<uint4 *>(dst + ks * 64 + pt * 32 + hh * 16) =
                                make_uint4(e[0], e[1], e[2], e[3]);
                        }
                }
            }
            if (tail == 8) {
#pragma unroll
                for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                    for (int hh = 0; hh < 2; ++hh) {
                        unsigned e[2];
#pragma unroll
                        for (int jj = 0; jj < 2; ++jj) {
                            unsigned short lo = 0, hi = 0;
                            // full16 <= 2 when R <= 40: ring indices below are static per full16
#pragma unroll
                            for (int f16 = 0; f16 <= 2; ++f16) {
                                if (f16 != full16) continue;
                                const int i0 = 16 * f16 + 4 * hh + 2 * jj;
                                if (i0 < kFragMaxRings && i0 < R) {
                                    const unsigned v = sp[i0][h];
                                    lo = frag16<BF16>(pt ? h2hi(v) * gf : (h2lo(v) - dc) * gf);
                                }
                                if (i0 + 1 < kFragMaxRings && i0 + 1 < R) {
                                    const unsigned v = sp[i0 + 1][h];
                                    hi = frag16<BF16>(pt ? h2hi(v) * gf : (h2lo(v) - dc) * gf);
                                }
                            }
                            e[jj] = lo | ((unsigned)hi << 16);
                        }
                        *reinterpret_cast<uint2 *>(dst + full16 * 64 + pt * 16 + hh * 8) =
                            make_uint2(e[0], e[1]);
                    }
            }
        }
    };

    // all rings of row j: sample position centre + shift + (i + 1)(cos, sin)
    auto row = [&](int j, float cx, float cy, auto inside_tag) __attribute__((always_inline)) {
        unsigned sp[kFragMaxRings][2];
        double sA = 0.0, sQ = 0.0;
#pragma unroll
        for (int i = 0; i < kFragMaxRings; i += 2) {
            if (i < R) {   // uniform
                const bool hb = (i + 1) < R;
                const float ra = (float)(i + 1), rb = (float)(i + 2);
                float va[4], vb[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // ring i + 2 of an odd R is sampled (inside the checked extent) and
                    // then zeroed, so the loop body has no branch per sample
                    va[q] = tap(fmaf(ra, cq[q], cx), fmaf(ra, sq[q], cy), inside_tag);
                    const float t = tap(fmaf(rb, cq[q], cx), fmaf(rb, sq[q], cy), inside_tag);
                    vb[q] = hb ? t : 0.0f;
                }
                ring_pair(i, va, vb, sp, sA, sQ);
            }
        }
        store_row(j, sp, sA, sQ);
    };

    for (int j = wave; j < n_rows; j += 4) {
        const int2 sh = shift_i[j];
        const float cx = (float)(D / 2 + kFragBorder + sh.x) + ax;
        const float cy = (float)(D / 2 + kFragBorder + sh.y) + ay;
        // uniform: every cell of the row's rings lies in the bordered copy (a
        // one-pixel margin covers the rounding of the positions)
        const float ext = (float)(R + 1), hi = (float)(W - 2);
        if (cx - ext >= 0.0f && cy - ext >= 0.0f && cx + ext <= hi && cy + ext <= hi)
            row(j, cx, cy, std::true_type{});
        else
            row(j, cx, cy, std::false_type{});
    }
}

// ------------------------------------------------------------------ stage B
// Psi transform: 256-point inverse FFTs, four per wavefront (16 lanes each, 16 points
// per lane).  The four radix-4 stages run in pairs inside a lane, so one exchange
// through LDS is left (a form with a transform spread over 64 lanes had three, and 36
// LDS instructions per transform against 12 here); the arithmetic of a stage (inputs,
// twiddles, operation order) is that of the Stockham stages above.
constexpr int kFftLd = 273;       // float2 per transform in LDS (odd mod 32: no bank conflicts
                                  // between transforms; 17 x 16 + 1 hold the padded exchange)
constexpr int kMirOff = 136;      // Z[k], k < 128, at k; Z[256 - k] at kMirOff + k (k = 1..128)
// First two stages.  In: x[m] = Z[u + 16 m], Z[64..127] (m = 4..7) without the row's
// scale gs, which the first butterflies apply in one rounding.  Out: x[4 k + q] is
// point 17 u + k + 4 q of the exchange.
__device__ __forceinline__ void ifft256_head(float2 (&x)[16], float gs) {
#pragma unroll
    for (int q2 = 0; q2 < 4; ++q2) {   // stage 1, butterfly u + 16 q2
        const float2 v0 = x[q2], v1 = x[q2 + 4], v2 = x[q2 + 8], v3 = x[q2 + 12];
        const float2 a0 = f2(v0.x + v2.x, v0.y + v2.y), a1 = f2(v0.x - v2.x, v0.y - v2.y);
        const float2 a2 = f2(fmaf(gs, v1.x, v3.x), fmaf(gs, v1.y, v3.y));
        const float2 a3 = f2(fmaf(gs, v1.x, -v3.x), fmaf(gs, v1.y, -v3.y));
        x[q2] = f2(a0.x + a2.x, a0.y + a2.y);
        x[q2 + 4] = f2(a1.x - a3.y, a1.y + a3.x);
        x[q2 + 8] = f2(a0.x - a2.x, a0.y - a2.y);
        x[q2 + 12] = f2(a1.x + a3.y, a1.y - a3.x);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {      // stage 2, butterfly 4 u + k
        float2 v[4] = {x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
        if (k > 0) {
#pragma unroll
            for (int q = 1; q < 4; ++q) v[q] = cmulc(v[q], stage2_tw(16 * q * k));
        }
        radix4<true>(v);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[4 * k + q] = v[q];
    }
}

__device__ __forceinline__ void ifft256_put(const float2 (&x)[16], float2 *xb, int u) {
    float2 *xw = xb + 17 * u;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) xw[k + 4 * q] = x[4 * k + q];
}

__device__ __forceinline__ void ifft256_get(float2 (&x)[16], const float2 *xb, int u) {
    const float2 *xr = xb + u;
#pragma unroll
    for (int a = 0; a < 16; ++a) x[a] = xr[17 * a];
}

// Z of one transform from LDS (positions of kMirOff) into lane u's 16 points
__device__ __forceinline__ void load_z(float2 (&x)[16], const float2 *xb, int u) {
    const float2 *lo = xb + u, *hi = xb + (kMirOff + 16 - u);
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = lo[16 * m];
#pragma unroll
    for (int m = 8; m < 16; ++m) x[m] = hi[16 * (15 - m)];
}

// Four transforms (lane row f's at xb, kFftLd float2 that are free to overwrite)
__device__ __forceinline__ void ifft256_rows4(float2 (&x)[16], float gs, float2 *xb, const float2 *tw, int u) {
    load_z(x, xb, u);
    ifft256_head(x, gs);
    wave_lds_sync();
    ifft256_put(x, xb, u);
    wave_lds_sync();
    ifft256_get(x, xb, u);
    fft256_tail<true>(x, tw, u);
}

// max over the 16 lanes of each lane row, then the wavefront's (uniform)
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, true)));
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// Running first maximum of one (particle, reference) over (mirror, shift, psi): value,
// flat index shift * 256 + psi sample, and (LDS) the seven samples around it.
struct PeakState {
    float bv[2];
    int bf[2];
    __device__ __forceinline__ void reset(float v, int f) {
        bv[0] = bv[1] = v;
        bf[0] = bf[1] = f;
    }
};

// Takes lane rows [f0, f0 + cnt) of a batch (lane row f holds the transform of shift
// s + f - f0) into the running maximum.  Rows arrive in increasing shift order, so a
// later equal value never displaces an earlier one, and the search for the position
// runs only when some lane beats the running maximum.  xb: the lane's transform
// buffer, free to overwrite.  SINGLE: the search starts from value 0 at index 0 like
// the reference's row argmax (cuda/gpu_aln_noref.cu:1638-1664), so when no value of
// the first shift is positive the record is that shift's sample 0.  MASKED: only the
// samples u + 16 m whose bit m (mirror 0) / 16 + m (mirror 1) of `allow` is set
// compete; the seven neighbours stay the unmasked values.
template <bool SINGLE, bool MASKED>
__device__ __forceinline__ void peak_update(PeakState &st, const float2 (&x)[16], int f0, int cnt, int s,
                                            int lane, float2 *xb, float (*nb)[8], unsigned allow) {
    const int f = lane >> 4, u = lane & 15;
    const bool in = f >= f0 && f < f0 + cnt;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        auto val = [&](int i) {
            const float v = m ? x[i].y : x[i].x;
            return (MASKED && !((allow >> (16 * m + i)) & 1u)) ? -INFINITY : v;
        };
        float lm = val(0);
#pragma unroll
        for (int i = 1; i < 16; ++i) lm = fmaxf(lm, val(i));
        lm = in ? lm : -INFINITY;
        const bool beats = __any(lm > st.bv[m]);
        const bool sentinel = SINGLE && m == 0 && s == 0 && !beats;
        if (!beats && !sentinel) continue;
        int fw = f0, t = 0;
        if (beats) {
            const float top = wave_max(lm);
            int tl = INT_MAX;
#pragma unroll
            for (int i = 15; i >= 0; --i)
                if (val(i) == top) tl = u + 16 * i;
            const unsigned long long hit = __ballot(in && lm == top);
            fw = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)hit) - 1) >> 4;   // smallest shift
            int tm = (f == fw && lm == top) ? tl : INT_MAX;
            tm = min(tm, __builtin_amdgcn_update_dpp(0, tm, 0x128, 0xf, 0xf, true));
            tm = min(tm, __builtin_amdgcn_update_dpp(0, tm, 0x124, 0xf, 0xf, true));
            tm = min(tm, __builtin_amdgcn_update_dpp(0, tm, 0x122, 0xf, 0xf, true));
            tm = min(tm, __builtin_amdgcn_update_dpp(0, tm, 0x121, 0xf, 0xf, true));
            t = __builtin_amdgcn_readlane(tm, fw * 16);
            st.bv[m] = top;
            st.bf[m] = (s + fw - f0) * kRingLen + t;
        }
        wave_lds_sync();
        float *zb = reinterpret_cast<float *>(xb);
        if (f == fw) {
#pragma unroll
            for (int i = 0; i < 16; ++i) zb[u + 16 * i] = m ? x[i].y : x[i].x;
        }
        wave_lds_sync();
        if (f == fw && u < 7) nb[m][u] = zb[(t + u - 3) & 255];
        wave_lds_sync();
    }
}

__device__ __forceinline__ void write_rec(PeakRec *o, const PeakState &st, const float (*nb)[8], int lane) {
    const int m = (st.bv[1] > st.bv[0]) ? 1 : 0;
    const bool none = st.bf[m] == INT_MAX;   // never updated: empty, or all values NaN
    const int f = none ? 0 : st.bf[m];
    if (lane == 0) {
        o->val = st.bv[m];
        o->m = m;
        o->s = f / kRingLen;
        o->t = f % kRingLen;
        o->pad = 0;
    }
    if (lane < 7) o->x[lane] = none ? 0.0f : nb[m][lane];
}

constexpr float kNoPeak = -3.40282e+38f;

// value of the neighbouring lane (lane ^ 1)
__device__ __forceinline__ float dpp_xor1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));
}

// A lane's 16 bytes of a ring row: one part (real in even lanes) of the four slots
// (lane >> 1 & 15) + 64 (lane >> 5) + 16 j.
__device__ __forceinline__ float4 load_part(const float2 *row, int lane) {
    return reinterpret_cast<const float4 *>(row)[lane];
}

// Products of one reference's lane part b with a row's a, summed over rings: own part in
// acc[0], the other one in acc[1].  Even lanes have P1 = rr sr and P3 = rr si of the four
// slots, odd lanes P2 = ri si and P4 = ri sr.
__device__ __forceinline__ void part_fma(float (&acc)[2][4], const float4 &b, const float4 &a) {
    const float bv[4] = {b.x, b.y, b.z, b.w}, av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        acc[0][j] = fmaf(bv[j], av[j], acc[0][j]);
        acc[1][j] = fmaf(bv[j], dpp_xor1(av[j]), acc[1][j]);
    }
}

// Z of one (shift row, reference) from the ring products, into LDS at the transform's
// positions: C0 = R conj S = (P1 + P2, P4 - P3), C1 = conj(R S) = (P1 - P2, -(P3 + P4));
// Z[k] = C0 + i C1 from even lanes, Z[256 - k] its Hermitian partner from odd ones; slot 0
// packs the real bins 0 (with the mean correction) and 128.  nm = (mu L, 1 / sd) scales the
// row, but for Z[64..127], which ifft256_head scales.
__device__ __forceinline__ void store_part_z(float2 *xb, const float (&acc)[2][4], float2 nm, float rs0, int lane) {
    const bool odd = lane & 1;
    const int k0 = ((lane >> 1) & 15) + 64 * (lane >> 5);
    const float gz = odd || lane < 32 ? nm.y : 1.0f;
    float2 *o = xb + (odd ? kMirOff : 0) + k0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float o0 = dpp_xor1(acc[0][j]), o1 = dpp_xor1(acc[1][j]);
        const float a = acc[0][j] + o0, e = acc[1][j] + o1;
        const float c = odd ? o0 - acc[0][j] : acc[0][j] - o0, b = odd ? acc[1][j] - o1 : o1 - acc[1][j];
        float2 z = odd ? f2(gz * (a - e), gz * (c - b)) : f2(gz * (a + e), gz * (b + c));
        if (j == 0 && lane < 2) {
            const float v = nm.y * (odd ? acc[0][0] : fmaf(-nm.x, rs0, acc[0][0]));
            xb[odd ? kMirOff + 128 : 0] = f2(v, v);
            continue;
        }
        o[16 * j] = z;
    }
}

// The value of the lane's row of 16 lanes.
__device__ __forceinline__ float lane_row_of(float r0, float r1, float r2, float r3, int lane) {
    const float lo = (lane & 16) ? r1 : r0, hi = (lane & 16) ? r3 : r2;
    return (lane & 32) ? hi : lo;
}

// One wavefront per particle, against its own reference ref_of[i * ref_stride]: four
// shift rows at a time (4 rows x 1 reference, two slots per lane), psi transforms of
// the four rows side by side.  The search starts from value 0 at index 0.
__global__ __launch_bounds__(256) void k_ccf_single(
    const float2 *__restrict__ spec, const float2 *__restrict__ norm,
    const float2 *__restrict__ rspec, const float *__restrict__ rsum0,
    const int *__restrict__ ref_of, int ref_stride, int n_items, int S, int R, int N,
    const float2 *__restrict__ twg, PeakRec *__restrict__ rec) {
    __shared__ float2 tw[kIfftTw];
    __shared__ float2 fbuf[4][4 * kFftLd];
    __shared__ float nbuf[4][2][8];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    fill_ifft_twiddles(tw, twg, tid, 256);
    __syncthreads();
    const int p = blockIdx.x * 4 + wave;
    if (p >= n_items) return;
    PeakState st;
    st.reset(0.0f, 0);
    // the host validates ref ids; the clamp keeps every read in bounds
    const int n = min(max(ref_of[(size_t)p * ref_stride], 0), N - 1);
    const float rs0 = rsum0[n];
    const float2 *rb0 = rspec + (size_t)n * R * kSlots;
    const size_t img_stride = (size_t)S * R * kSlots;
    float2 *xb = fbuf[wave] + (lane >> 4) * kFftLd;
    for (int s0 = 0; s0 < S; s0 += 4) {
        float acc[4][2][4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r][h][e] = 0.0f;
        const float2 *arow[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            arow[r] = spec + (size_t)p * img_stride + (size_t)min(s0 + r, S - 1) * R * kSlots;
        for (int i = 0; i < R; ++i) {
            const float4 b = load_part(rb0 + i * kSlots, lane);
            float4 a[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) a[r] = load_part(arow[r] + i * kSlots, lane);
            __builtin_amdgcn_sched_barrier(0);   // all of the ring's loads in flight before the FMAs
#pragma unroll
            for (int r = 0; r < 4; ++r) part_fma(acc[r], b, a[r]);
        }
        wave_lds_sync();
        float2 nm[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            nm[r] = norm[(size_t)p * S + min(s0 + r, S - 1)];
            store_part_z(fbuf[wave] + r * kFftLd, acc[r], nm[r], rs0, lane);
        }
        wave_lds_sync();
        float2 x[16];
        ifft256_rows4(x, lane_row_of(nm[0].y, nm[1].y, nm[2].y, nm[3].y, lane), xb, tw, lane & 15);
        peak_update<true, false>(st, x, 0, min(4, S - s0), s0, lane, xb, nbuf[wave], 0u);
    }
    write_rec(rec + p, st, nbuf[wave], lane);
}

// a b, rounded before any sum that takes it (not fused into it)
__device__ __forceinline__ float mul_rn(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

// Each image against its own reference ref_of[p * ref_stride], from the pixels: k_polar_spectra's
// workgroup and wavefronts (one image, four shift rows at a time, a ring pair at a time), but
// the spectra of a pair are contracted with the reference's at once, in the ring order and
// operation order of k_ccf_single, and are never written out; then the psi transforms of the
// four rows.  The wavefronts' first maxima are merged: larger value, then smaller shift.
// What bounds it: vector instructions, as k_polar_spectra without its stores, and scratch: 61
// of a lane's values do not fit the 128 registers of four wavefronts per SIMD.  5000 images
// of 76 x 76, 34 rings, 49 and 9 shifts in turn: 2.1 ms a search; the two passes, with 8.6 GB
// of spectra written and read at 49 shifts, took 3.3.  With the sums of a ring pair over
// its lanes at once 9 values spill, and pre-alignment of these images took 13.3 ms for 12.7.
__global__ __launch_bounds__(1024, 4) void k_polar_single(
    const float *__restrict__ imgs, int D, ShiftView acc, const int2 *__restrict__ shift_i, int S,
    const float2 *__restrict__ tmpl, int R, const float2 *__restrict__ twg, const float2 *__restrict__ rspec,
    const float *__restrict__ rsum0, const int *__restrict__ ref_of, int ref_stride, int N,
    PeakRec *__restrict__ rec) {
    extern __shared__ float4 smem4[];
    __shared__ float nbuf[16][2][8];
    __shared__ float pv[16][2];
    __shared__ int pf[16][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = blockDim.x >> 6, f = lane >> 4, u = lane & 15;
    const int p = blockIdx.x, W = D + 2;
    float2 *tw = reinterpret_cast<float2 *>(smem4);
    float *xb = reinterpret_cast<float *>(tw + kIfftTw) + (wave * 4 + f) * kXchLd;
    float *img = reinterpret_cast<float *>(tw + kIfftTw) + nw * 4 * kXchLd;
    load_bordered(img, imgs + (size_t)p * D * D, D);
    fill_ifft_twiddles(tw, twg, tid, blockDim.x);
    __syncthreads();
    const float ax = acc.base[(size_t)p * acc.stride], ay = acc.base[(size_t)p * acc.stride + 1];
    // the host validates ref ids; the clamp keeps every read in bounds
    const int n = min(max(ref_of[(size_t)p * ref_stride], 0), N - 1);
    const float rs0 = rsum0[n];
    const float4 *rb = reinterpret_cast<const float4 *>(rspec + (size_t)n * R * kSlots) + 2 * u;
    PeakState st;
    st.reset(0.0f, 0);
    for (int j0 = 4 * wave; j0 < S; j0 += 4 * nw) {
        const int2 si = shift_i[min(j0 + f, S - 1)];   // lanes past the last row repeat it
        const float cx = (float)(D / 2 + si.x) + ax, cy = (float)(D / 2 + si.y) + ay;
        double sA = 0.0, sQ = 0.0;
        float c[8][4];
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) c[m][e] = 0.0f;
        auto contract = [&](const float2 (&v)[8], int i) {
            const float4 *r = rb + (size_t)i * (kSlots / 2);
#pragma unroll
            for (int mh = 0; mh < 2; ++mh) {
                const float4 re4 = r[32 * mh], im4 = r[32 * mh + 1];
                const float re[4] = {re4.x, re4.y, re4.z, re4.w}, im[4] = {im4.x, im4.y, im4.z, im4.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int m = 4 * mh + k;
                    c[m][0] = fmaf(re[k], v[m].x, c[m][0]);
                    c[m][1] = fmaf(im[k], v[m].y, c[m][1]);
                    c[m][2] = fmaf(re[k], v[m].y, c[m][2]);
                    c[m][3] = fmaf(im[k], v[m].x, c[m][3]);
                }
            }
        };
        for (int i = 0; i < R; i += 2) {
            float2 a[8], b[8];
            const double2 t = ring_pair(img + W + 1, (float)W, (float)(D - 1), W, tmpl, i, R, cx, cy, u, xb, tw, a, b);
            sA += t.x;
            sQ += t.y;
            contract(a, i);
            if (i + 1 < R) contract(b, i + 1);
        }
        const float2 nm = ring_norm(row_sum(sA), row_sum(sQ), R);
        // Z as store_pair_z makes it; Z[256 - k] goes to lane (16 - u) & 15 through LDS
        float2 x[16];
        float2 *zb = reinterpret_cast<float2 *>(xb);
        wave_lds_sync();
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const float a = c[m][0] + c[m][1], e = c[m][2] + c[m][3];
            const float g = c[m][0] - c[m][1], b = c[m][3] - c[m][2];
            x[m] = m < 4 ? f2(mul_rn(nm.y, a + e), mul_rn(nm.y, b + g)) : f2(a + e, b + g);
            float2 y = f2(nm.y * (a - e), nm.y * (g - b));
            int ky = u + 16 * m;
            if (m == 0 && u == 0) {
                const float c0 = mul_rn(nm.y, fmaf(-nm.x, rs0, c[0][0]));
                const float cn = nm.y * c[0][1];
                x[0] = f2(c0, c0);
                y = f2(cn, cn);
                ky = 128;
            }
            zb[ky] = y;
        }
        wave_lds_sync();
#pragma unroll
        for (int m = 8; m < 16; ++m) x[m] = zb[128 - u - 16 * (m - 8)];
        ifft256_head(x, nm.y);
        row_exchange(x, xb, u);
        fft256_tail<true>(x, tw, u);
        peak_update<true, false>(st, x, 0, min(4, S - j0), j0, lane, zb, nbuf[wave], 0u);
    }
    if (lane < 2) {
        pv[wave][lane] = lane ? st.bv[1] : st.bv[0];
        pf[wave][lane] = lane ? st.bf[1] : st.bf[0];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        int w = 0;
#pragma unroll 1
        for (int k = 1; k < nw; ++k)
            if (pv[k][m] > st.bv[m] || (pv[k][m] == st.bv[m] && pf[k][m] < st.bf[m])) {
                st.bv[m] = pv[k][m];
                st.bf[m] = pf[k][m];
                w = k;
            }
        if (lane < 7) nbuf[0][m][lane] = nbuf[w][m][lane];   // where write_rec reads them
    }
    wave_lds_sync();
    write_rec(rec + p, st, nbuf[0], lane);
}

// Top-K references of every particle by approximate peak value (descending; ties
// to the lower reference index).  One thread per particle.
template <int K>
__global__ void k_topk(const PeakRec *__restrict__ rec, int n_img, int N, int *__restrict__ cand) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img) return;
    float v[K];
    int id[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = -INFINITY;
        id[k] = 0;
    }
    for (int n = 0; n < N; ++n) {
        const float x = rec[(size_t)p * N + n].val;
        if (!(x > v[K - 1])) continue;
        float cv = x;
        int ci = n;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (cv > v[k]) {
                const float tv = v[k];
                const int ti = id[k];
                v[k] = cv;
                id[k] = ci;
                cv = tv;
                ci = ti;
            }
        }
    }
    const int kk = min(K, N);
#pragma unroll
    for (int k = 0; k < K; ++k) cand[(size_t)p * K + k] = (k < kk) ? id[k] : id[0];
}

// Best exact candidate per particle: highest FP32 peak (ties to the lower
// reference index); flags a near-tie when the best distinct candidate is within
// tie_rel of it.  best[p] = candidate slot, second[p] = runner-up slot (-1 none).
__global__ void k_best_candidate(const PeakRec *__restrict__ rec, const int *__restrict__ cand,
                                 int n_img, int K, float tie_rel, int *__restrict__ best,
                                 int *__restrict__ second, int *__restrict__ tie) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img) return;
    int b = -1, s2 = -1;
    for (int k = 0; k < K; ++k) {
        const int n = cand[(size_t)p * K + k];
        bool dup = false;
        for (int j = 0; j < k; ++j) dup |= cand[(size_t)p * K + j] == n;
        if (dup) continue;
        const float x = rec[(size_t)p * K + k].val;
        if (b < 0) {
            b = k;
            continue;
        }
        const float xb = rec[(size_t)p * K + b].val;
        const int nb = cand[(size_t)p * K + b];
        if (x > xb || (x == xb && n < nb)) {
            s2 = b;
            b = k;
        } else if (s2 < 0) {
            s2 = k;
        } else {
            const float x2 = rec[(size_t)p * K + s2].val;
            const int n2 = cand[(size_t)p * K + s2];
            if (x > x2 || (x == x2 && n < n2)) s2 = k;
        }
    }
    best[p] = b;
    second[p] = s2;
    int t = 0;
    if (s2 >= 0) {
        const float xb = rec[(size_t)p * K + b].val, x2 = rec[(size_t)p * K + s2].val;
        t = (xb - x2) <= tie_rel * fabsf(xb);
    }
    tie[p] = t;
}

// Near-tie re-scoring in FP64: for a flagged particle, one wavefront per candidate
// (best, runner-up) recomputes C0/C1 over rings in double from the FP32 spectra
// and evaluates the psi CCF of its winning mirror / shift at t*-1, t*, t*+1 by
// direct summation: c[t] = C[0] + C[128] (-1)^t + 2 sum_k Re(C[k] e^{2 pi i k t/256}).
// val64[2p + j] = the largest of the three (j = 0 best, 1 runner-up).
__global__ __launch_bounds__(256) void k_rescore_f64(
    const float2 *__restrict__ spec, const float2 *__restrict__ norm,
    const float2 *__restrict__ rspec, const PeakRec *__restrict__ rec,
    const int *__restrict__ cand, const int *__restrict__ best, const int *__restrict__ second,
    const int *__restrict__ tie, int n_img, int K, int S, int R, int N, double *__restrict__ val64) {
    const int lane = threadIdx.x & 63;
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int p = w >> 1, j = w & 1;
    if (p >= n_img || !tie[p]) return;
    const int slot_k = j ? second[p] : best[p];
    if (slot_k < 0) return;
    const PeakRec r = rec[(size_t)p * K + slot_k];
    const int n = min(max(cand[(size_t)p * K + slot_k], 0), N - 1);
    const int s = min(max(r.s, 0), S - 1);
    const float2 nm = norm[(size_t)p * S + s];
    const double muL = nm.x, g = nm.y;
    double P[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    const float2 *a = spec + ((size_t)p * S + s) * R * kSlots;
    const float2 *b = rspec + (size_t)n * R * kSlots;
    for (int i = 0; i < R; ++i) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = lane + 64 * h;
            const float2 av = load_slot(a + i * kSlots, k), bv = load_slot(b + i * kSlots, k);
            const double x = ((k == 0) ? ((double)av.x - muL) : (double)av.x) * g;
            const double y = (double)av.y * g;
            P[h][0] += (double)bv.x * x;
            P[h][1] += (double)bv.y * y;
            P[h][2] += (double)bv.x * y;
            P[h][3] += (double)bv.y * x;
        }
    }
    double best_v = -INFINITY;
    for (int dt = -1; dt <= 1; ++dt) {
        const int t = (r.t + dt + 256) & 255;
        double sum = 0.0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = lane + 64 * h;
            const double c0r = P[h][0] + P[h][1], c0i = P[h][3] - P[h][2];
            const double c1r = P[h][0] - P[h][1], c1i = -(P[h][2] + P[h][3]);
            const double cr = r.m ? c1r : c0r, ci = r.m ? c1i : c0i;
            if (k == 0) {  // DC and Nyquist (slot 0 packs both)
                sum += P[h][0] + ((t & 1) ? -P[h][1] : P[h][1]);
            } else {
                double sn, cs;
                sincospi((double)(2 * k * t % 512) / 256.0, &sn, &cs);
                sum += 2.0 * (cr * cs - ci * sn);
            }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        best_v = fmax(best_v, sum);
    }
    if (lane == 0) val64[2 * p + j] = best_v;
}

// Swap best and runner-up of flagged particles when FP64 ranks them the other way
// (equal values: the lower reference index wins).
__global__ void k_resolve_ties(const int *__restrict__ cand, const double *__restrict__ val64,
                               const int *__restrict__ tie, int n_img, int K, int *__restrict__ best,
                               int *__restrict__ second) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img || !tie[p] || second[p] < 0) return;
    const double vb = val64[2 * p], vs = val64[2 * p + 1];
    const int nb = cand[(size_t)p * K + best[p]], ns = cand[(size_t)p * K + second[p]];
    if (vs > vb || (vs == vb && ns < nb)) {
        const int t = best[p];
        best[p] = second[p];
        second[p] = t;
    }
}

// Multi-reference search, FP32.  Workgroup = 8 references (a tile) x a run of consecutive
// (particle, shift) rows, sixteen wavefronts, one workgroup per CU.  Per block of 8 rows:
//  * ring contraction (wavefronts 0..7) on v_mfma_f32_16x16x1_f32 (four 16 x 16 blocks,
//    K = 1 ring): the four blocks are four spectrum slots, rows = 8 particle rows x (re,
//    im), columns = 8 references x (re, im), so one instruction adds P1..P4 of 64 pairs
//    in four slots.  Each step is one fused multiply-add, rings in order: the bits of an
//    fmaf chain.  A wavefront owns 16 slots (4 instructions a ring, 64 accumulators);
//    the operands of one ring are one 16-byte load per lane and side;
//  * the cross-spectra of the 64 pairs (128 KB) go through LDS to the psi transforms;
//  * psi transforms and search (wavefronts 8..15): one reference each, four rows side by
//    side, while the others contract the next block.
// The tiles of a run are neighbouring workgroups on one XCD and read its rows through
// one L2.
//
// Why this form: with both stages on the vector unit (an earlier kernel, 4 rows x 16
// references per workgroup at two wavefronts per SIMD) instruction issue bound the
// search, 115 ms for 20 000 x 100 at 76 px, 35 rings, 49 shifts; this one takes 65 ms.
// On this chip a SIMD's matrix and vector instructions do not overlap (4 matrix
// instructions of 32 cycles and 64 adds take the sum of their times, at 1, 2 and 4
// wavefronts), so the floor of a block is the sum: 8 960 matrix cycles at 35 rings and
// about 5 600 vector cycles, 36 ms in all.  What is left above it: 528 KB of operand
// loads a block (without them 53 ms; 8 KB a ring at 25-32 bytes per cycle and CU), the
// psi wavefronts' LDS round trips, and the two barriers.  Splitting the wavefronts by
// stage beat every form in which each does both (spills at 128 registers, or phases
// that leave the load path idle): 75 ms with two workgroups of 8 wavefronts per CU, 82 ms
// with one whose wavefronts keep 28 rings of the rows.
constexpr int kMrefPre = 4;       // rings of the rows in flight
constexpr int kRefPre = 2;        // and of the references' rings past the resident ones
// rings of the references kept in registers over a run: 4 096 x 100 at 76 px takes 14.9 ms
// with none, 13.5 with 4, 14.3 with 6, 15.0 with 8 (a wavefront has 128 registers)
constexpr int kMrefKeep = 4;

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// Loads through a job's pointers.  The queue kernel reads them from memory, where nothing
// says that they are global, and a flat load also holds the LDS counter.
#define GLOBAL_AS __attribute__((address_space(1)))
typedef GLOBAL_AS char global_char;
template <class T>
__device__ __forceinline__ T load_global(const T *p) {
    return *(const GLOBAL_AS T *)p;
}
__device__ __forceinline__ float2 load_global2(const float2 *p) {
    const f32x2_t v = *(const GLOBAL_AS f32x2_t *)p;
    return f2(v.x, v.y);
}

struct MrefLds {
    float2 z[64 * kFftLd];            // transform (reference n, row r) at n + 8 r
    float2 tw[kIfftTw];
    float nb[kMrefRefs][2][8];        // seven samples around the running maxima
};

// f(0), f(1), .., f(N - 1) with compile-time arguments
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// Reference of column c of tile g (negative: none).  LIST: the candidate form of MrefJob,
// list p0's K references.
template <bool LIST>
__device__ __forceinline__ int mref_ref_at(const MrefJob &j, int p0, int g, int c) {
    if (LIST) return c < j.K ? j.cand[(size_t)p0 * j.K + c] : -1;
    return kMrefRefs * g + c < j.N ? kMrefRefs * g + c : -1;
}

// Contraction wavefront w of a run.  KR: rings of the references kept in registers (at
// most R).
template <bool LIST, int KR>
__device__ __forceinline__ void mref_contract(const MrefJob &j, int w, int lane, int p0, int np, int g,
                                              MrefLds &sh) {
    const int S = j.S, R = j.R, N = j.N;
    const int f = lane >> 4, u = lane & 15;
    const int ps = (LIST && j.pidx) ? j.pidx[p0] : p0;   // spectra row of the first particle
    const int n_rows = np * S;
    const int n_blk = (n_rows + 7) / 8;

    // operand addresses.  Lane 16 b + i of an instruction: block b (slot), i = 2 t + part;
    // matrix row pair t holds shift row (t >> 1) + 4 (t & 1), so accumulators 0, 1 of a
    // block belong to row f and 2, 3 to row 4 + f (f = lane row); columns 2 t + part.
    const int part = u & 1, t = u >> 1, ar = (t >> 1) + 4 * (t & 1);
    const unsigned row_bytes = (unsigned)R * (kSlots * 8);
    const unsigned ring_off = (unsigned)(w * 8 + f * 2 + part) * 16u;   // in a ring row
    const char *ab = reinterpret_cast<const char *>(j.spec) + (size_t)ps * S * row_bytes;
    const float sgn = part ? -1.0f : 1.0f;
    // the host validates candidate ids; the clamp keeps every read in bounds
    const int ref = min(max(mref_ref_at<LIST>(j, p0, g, t), 0), N - 1);
    const global_char *bp = (const global_char *)j.rspec + (size_t)ref * row_bytes + ring_off;
    const float rs0 = load_global<float>(j.rsum0 + ref);

    // LDS positions: this lane's Z values (reference t, row f or 4 + f; even lanes Z[k],
    // odd lanes Z[256 - k]) of its wavefront's slots 16 (4 mh + jj) + 4 uq + b, w = 4 mh + uq
    float2 *zw = sh.z + (t + 8 * f) * kFftLd + part * kMirOff + 64 * (w >> 2) + 4 * (w & 3);

    const char *ablk = ab;   // the block's rows, and this lane's row among them
    unsigned aoff = (unsigned)min(ar, n_rows - 1) * row_bytes + ring_off;
    f32x4_t keep[KR > 0 ? KR : 1], rb[kRefPre], ra[kMrefPre];
    auto load_b = [&](int i) {
        return *(const GLOBAL_AS f32x4_t *)(bp + (size_t)(unsigned)min(i, R - 1) * (kSlots * 8));
    };
    auto load_a = [&](int i) {
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(ablk), (short)0, -1, 0x00020000);
        return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                               rs, aoff, (unsigned)min(i, R - 1) * (kSlots * 8), 0));
    };
    static_for<KR>([&](auto ic) { keep[decltype(ic)::value] = load_b(decltype(ic)::value); });
    static_for<kMrefPre>([&](auto dc) { ra[decltype(dc)::value] = load_a(decltype(dc)::value); });
    for (int blk = 0; blk < n_blk; ++blk) {
        float2 nm[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
            nm[hh] = load_global2(j.norm + ((size_t)ps * S + 8 * (size_t)blk + min(4 * hh + f, n_rows - 1 - 8 * blk)));
        static_for<kRefPre>([&](auto dc) { rb[decltype(dc)::value] = load_b(KR + decltype(dc)::value); });

        f32x16_t acc[4] = {};
        auto step = [&](const f32x4_t &a, const f32x4_t &b) {
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
                acc[jj] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[jj], b[jj], acc[jj], 0, 0, 0);
        };
        static_for<KR>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            step(ra[i % kMrefPre], keep[i]);
            ra[i % kMrefPre] = load_a(i + kMrefPre);
            __builtin_amdgcn_sched_barrier(0);   // keeps the loads ahead of their use
        });
        int i0 = KR;
        for (; i0 + kMrefPre <= R; i0 += kMrefPre)
            static_for<kMrefPre>([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                step(ra[(KR + d) % kMrefPre], rb[d % kRefPre]);
                rb[d % kRefPre] = load_b(i0 + d + kRefPre);
                ra[(KR + d) % kMrefPre] = load_a(i0 + d + kMrefPre);
                __builtin_amdgcn_sched_barrier(0);
            });
        static_for<kMrefPre - 1>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            if (i0 + d < R) {   // uniform
                if constexpr (d < kRefPre) step(ra[(KR + d) % kMrefPre], rb[d]);
                else step(ra[(KR + d) % kMrefPre], load_b(i0 + d));
            }
        });
        // the next block's first rings load while this one's cross-spectra go to LDS
        if (blk + 1 < n_blk) {
            ablk += 8 * (size_t)row_bytes;
            aoff = (unsigned)min(ar, n_rows - 9 - 8 * blk) * row_bytes + ring_off;
        }
        static_for<kMrefPre>([&](auto dc) { ra[decltype(dc)::value] = load_a(decltype(dc)::value); });

        __syncthreads();   // the transforms of the previous block are done
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const float gs = nm[hh].y;
            const float gw = (w >= 4 && !part) ? 1.0f : gs;   // Z[64..127] is scaled by the transform
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    // even lanes hold (sr, si) rr = P1, P3 and odd lanes (sr, si) ri = P4, P2 of
                    // a slot; with the neighbour's values both form C0 and C1:
                    // Z[k] = (s + t', d + e) in even lanes, Z[256 - k] = (t' - s, e - d) in odd
                    const float x0 = acc[jj][4 * b + 2 * hh], x1 = acc[jj][4 * b + 2 * hh + 1];
                    const float y0 = dpp_xor1(x0), y1 = dpp_xor1(x1);
                    const float ss = x0 + y1, tt = x1 + y0, dd = x0 - y1, ee = y0 - x1;
                    zw[32 * hh * kFftLd + 16 * jj + b] = f2(gw * fmaf(sgn, ss, tt), gw * fmaf(sgn, dd, ee));
                }
            if (w == 0) {   // slot 0 packs the real bins 0 (mean-corrected) and 128
                const float x0 = acc[0][2 * hh], x1 = acc[0][2 * hh + 1];
                const float c = gs * (part ? x1 : fmaf(-nm[hh].x, rs0, x0));
                wave_lds_sync();
                sh.z[(t + 8 * (4 * hh + f)) * kFftLd + part * (kMirOff + 128)] = f2(c, c);
            }
        }
        __syncthreads();
    }
}

// Psi wavefront c of a run: column c of the tile.
template <bool LIST>
__device__ __forceinline__ void mref_psi(const MrefJob &j, int c, int lane, int p0, int np, int g, MrefLds &sh) {
    const int S = j.S;
    const int f = lane >> 4, u = lane & 15;
    const int ps = (LIST && j.pidx) ? j.pidx[p0] : p0;
    const int n_rows = np * S;
    const int n_blk = (n_rows + 7) / 8;
    const int ref = mref_ref_at<LIST>(j, p0, g, c);
    PeakState st;
    st.reset(kNoPeak, INT_MAX);
    int p = 0, s = 0;   // particle and shift of the next row
    for (int blk = 0; blk < n_blk; ++blk) {
        const int rows = min(8, n_rows - 8 * blk);
        const size_t row0 = (size_t)ps * S + 8 * (size_t)blk;
        const float gs0 = load_global2(j.norm + (row0 + min(f, rows - 1))).y;
        const float gs1 = load_global2(j.norm + (row0 + min(4 + f, rows - 1))).y;
        __syncthreads();   // the contraction of this block is done
        __syncthreads();   // and its cross-spectra are in LDS
        if (ref < 0) continue;   // uniform over the wavefront
        float2 *xb = sh.z + (c + 8 * f) * kFftLd;
        for (int hh = 0; 4 * hh < rows; ++hh, xb += 32 * kFftLd) {
            float2 x[16];
            ifft256_rows4(x, hh ? gs1 : gs0, xb, sh.tw, u);
            // the rows may end a particle and begin the next
            for (int f0 = 0; f0 < min(4, rows - 4 * hh);) {
                const int cnt = min(min(4, rows - 4 * hh) - f0, S - s);
                peak_update<false, false>(st, x, f0, cnt, s, lane, xb, sh.nb[c], 0u);
                f0 += cnt;
                s += cnt;
                if (s == S) {
                    wave_lds_sync();
                    write_rec(LIST ? j.rec + (size_t)p0 * j.K + c : j.rec + (size_t)(p0 + p) * j.N + ref, st, sh.nb[c],
                              lane);
                    wave_lds_sync();
                    st.reset(kNoPeak, INT_MAX);
                    s = 0;
                    ++p;
                }
            }
        }
    }
    // an empty slot of a list: an empty record
    if (LIST && ref < 0 && c < j.K) write_rec(j.rec + (size_t)p0 * j.K + c, st, sh.nb[c], lane);
}

// Work of one workgroup: reference tile g against particles p0 .. p0 + np - 1 of job j (the
// twiddles must be in sh.tw by the first barrier).  LIST: list p0 (np = 1), its K
// references against its particle; every slot of the list gets a record, and each listed
// reference's record is the one the exhaustive form computes for it.
template <bool LIST, int KR>
__device__ __forceinline__ void mref_run(const MrefJob &j, int tid, int p0, int np, int g, MrefLds &sh) {
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    if (w < 8) mref_contract<LIST, KR>(j, w, lane, p0, np, g, sh);
    else mref_psi<LIST>(j, w - 8, lane, p0, np, g, sh);
}

// Logical block = run of cp particles x reference tile (fastest).
template <int KR>
__global__ __launch_bounds__(kMrefWaves * 64, 4) void k_ccf_mref(MrefJob j, int cp,
                                                                 const float2 *__restrict__ twg) {
    __shared__ MrefLds sh;
    fill_ifft_twiddles(sh.tw, twg, threadIdx.x, kMrefWaves * 64);
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int ng = (j.N + kMrefRefs - 1) / kMrefRefs;
    const int p0 = lb / ng * cp;
    if (p0 >= j.n_img) return;  // uniform over the workgroup
    mref_run<false, KR>(j, threadIdx.x, p0, min(cp, j.n_img - p0), lb % ng, sh);
}

// Candidate re-scoring (the candidate form of MrefJob) by the exhaustive kernel's
// workgroup code, so every record equals k_ccf_mref's for that (particle, reference).
template <int KR>
__global__ __launch_bounds__(kMrefWaves * 64, 4) void k_ccf_cand(MrefJob j, const float2 *__restrict__ twg) {
    __shared__ MrefLds sh;
    fill_ifft_twiddles(sh.tw, twg, threadIdx.x, kMrefWaves * 64);
    mref_run<true, KR>(j, threadIdx.x, blockIdx.x, 1, 0, sh);
}

// Persistent form over many jobs (batched subsets): work items (job, first particle,
// reference tile, particles) sit in 8 queues, one per XCD (the tiles of a run share a
// queue, so its spectra stay in one L2); each workgroup takes items from the queue of
// the XCD it runs on (blockIdx % 8) until the queue is exhausted.  The claim is a vector
// atomic by one lane, broadcast through LDS.  Every workgroup leaves the loop once its
// queue is empty.
template <int KR>
__global__ __launch_bounds__(kMrefWaves * 64, 4) void k_ccf_mref_queue(
    const MrefJob *__restrict__ jobs, const int4 *__restrict__ items, const int *__restrict__ qbeg,
    int *__restrict__ counters, const float2 *__restrict__ twg) {
    __shared__ MrefLds sh;
    __shared__ int claim;
    fill_ifft_twiddles(sh.tw, twg, threadIdx.x, kMrefWaves * 64);
    const int q = blockIdx.x & 7;
    const int q0 = qbeg[q], q1 = qbeg[q + 1];
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) claim = atomicAdd(&counters[q], 1);
        __syncthreads();
        const int idx = q0 + __builtin_amdgcn_readfirstlane(claim);   // scalar, and what follows from it
        if (idx >= q1) break;
        const int4 it = items[idx];
        const MrefJob j = jobs[it.x];
        // what follows from the lane is computed again for each item: kept over the loop it
        // takes the registers of the resident rings
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        mref_run<false, KR>(j, tid, it.y, it.w, it.z, sh);
    }
}

__global__ void k_reset_counters(int *__restrict__ c, int n) {
    const int i = threadIdx.x;
    if (i < n) c[i] = 0;
}

// ------------------------------------------------------------------ decode
// Angle of a multi-reference peak, as the reference wizard computes it
// (cuda/gpu_aln_noref.cu:1777-1793): float coefficients from double
// expressions, the offset in double, the angle stored as float.
__device__ __forceinline__ float wizard_angle(const PeakRec &r) {
    const float *x = r.x;
    const float c2 = (float)(49. * x[0] + 6. * x[1] - 21. * x[2] - 32. * x[3] - 27. * x[4] -
                             6. * x[5] + 31. * x[6]);
    const float c3 = (float)(5. * x[0] - 3. * x[2] - 4. * x[3] - 3. * x[4] + 5. * x[6]);
    const float step = (float)(360.0 / (double)kRingLen);
    float angle = step * (float)r.t;
    if (c3 != 0.0f) angle = (float)((double)angle + (double)step * ((double)c2 / (2.0 * (double)c3) - 4.0));
    angle = (float)(360.0 - (double)angle);
    if (r.m == 1) angle = (float)((double)angle + 180.0);
    if (angle >= 360.0f) angle = (float)((double)angle - 360.0);
    return angle;
}

// ------------------------------------------------------------------ narrowed search
// Proposals (ref, mirror, psi bin, shift) -> work items.  Proposals with the
// same (ref, shift) share one item whose mask is the union of their (mirror,
// psi) windows: bit m*256 + t for the psi samples t within psi_half degrees of
// the bin centre (b + 0.5) * 360 / n_bins.  smask[p] marks every shift inside
// the (2 hw + 1)^2 windows (for the masked polar pass).  Invalid proposals
// (ref or shift out of range) are dropped.  One thread per particle.
__global__ void k_prop_items(const int4 *__restrict__ prop, int n_img, int K, int N, int nx,
                             int ny, int hw, int n_bins, float psi_half, PropItem *__restrict__ items,
                             unsigned long long *__restrict__ smask) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img) return;
    PropItem it[kMaxProposals];
    int cnt = 0;
    unsigned long long mk = 0ull;
    const double step = 360.0 / (double)kRingLen, bw = 360.0 / (double)n_bins;
    for (int k = 0; k < K; ++k) {
        const int4 q = prop[(size_t)p * K + k];
        const int ref = q.x, m = q.y, b = q.z, sh = q.w;
        if (ref < 0 || ref >= N || m < 0 || m > 1 || b < 0 || b >= n_bins || sh < 0 || sh >= nx * ny)
            continue;
        int j = 0;
        while (j < cnt && !(it[j].ref == ref && it[j].s == sh)) ++j;
        if (j == cnt) {
            it[j].ref = ref;
            it[j].s = sh;
            for (int w = 0; w < 16; ++w) it[j].mask[w] = 0u;
            ++cnt;
        }
        const double c = ((double)b + 0.5) * bw;
        const int t0 = (int)ceil((c - (double)psi_half) / step);
        const int t1 = (int)floor((c + (double)psi_half) / step);
        for (int t = t0; t <= t1 && t < t0 + kRingLen; ++t) {
            const int tt = ((t % kRingLen) + kRingLen) % kRingLen;
            const int bit = m * kRingLen + tt;
            it[j].mask[bit >> 5] |= 1u << (bit & 31);
        }
        const int ix0 = sh / ny, iy0 = sh % ny;
        for (int ix = max(0, ix0 - hw); ix <= min(nx - 1, ix0 + hw); ++ix)
            for (int iy = max(0, iy0 - hw); iy <= min(ny - 1, iy0 + hw); ++iy)
                mk |= 1ull << (ix * ny + iy);
    }
    for (int j = 0; j < K; ++j) {
        PropItem o;
        if (j < cnt) {
            o = it[j];
        } else {
            o.ref = -1;
            o.s = 0;
            for (int w = 0; w < 16; ++w) o.mask[w] = 0u;
        }
        items[(size_t)p * K + j] = o;
    }
    smask[p] = mk;
}

// One wavefront per item: the shifts of the item's (2 hw + 1)^2 window (in
// increasing grid order) NROW at a time against its reference, with exactly
// the arithmetic of the exhaustive kernels (ring contraction, psi FFT), the
// maximum taken over the item's (mirror, psi) mask only.  Workgroup = one
// particle's K <= 8 items (K wavefronts), so the spectrum rows its windows share
// are read through one CU and one L2.
// What bounds it: the loads of the contraction, one 16-byte load a row and ring (10 000 x 8
// items of 76 x 76, 9 shifts, 34 rings: 2.97 ms; two 8-byte loads 3.22), and the vector work
// of the psi transforms; LDS for K items only lets more workgroups share a CU where they are
// few (10 000 x 1 item of one shift: 0.46 -> 0.11 ms, with NROW = 1 for windows of one shift).
template <int NROW>
__global__ __launch_bounds__(512) void k_ccf_prop(
    const float2 *__restrict__ spec, const float2 *__restrict__ norm,
    const float2 *__restrict__ rspec, const float *__restrict__ rsum0,
    const PropItem *__restrict__ items, int K, int n_items, int S, int R, int N, int nx, int ny,
    int hw, const float2 *__restrict__ twg, PeakRec *__restrict__ rec) {
    extern __shared__ float4 smem4[];
    float2 (*fbuf)[4 * kFftLd] = reinterpret_cast<float2 (*)[4 * kFftLd]>(smem4);   // [K]
    __shared__ float2 tw[kIfftTw];
    __shared__ float nbuf[kMaxProposals][2][8];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    fill_ifft_twiddles(tw, twg, tid, blockDim.x);
    __syncthreads();
    const int item = blockIdx.x * K + wave;
    if (item >= n_items) return;
    const int p = item / K;
    const PropItem &it = items[item];
    PeakState st;
    st.reset(kNoPeak, INT_MAX);
    const int n = it.ref;
    if (n >= 0 && n < N) {
        const int u = lane & 15;
        unsigned allow = 0u;   // bit 16 m + i: sample u + 16 i of mirror m
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                allow |= ((it.mask[m * 8 + (i >> 1)] >> (u + 16 * (i & 1))) & 1u) << (16 * m + i);
        // window rows j = 0..nr-1 in increasing grid order
        const int ix0 = it.s / ny, iy0 = it.s % ny;
        const int ixa = max(0, ix0 - hw), ixb = min(nx - 1, ix0 + hw);
        const int iya = max(0, iy0 - hw), iyb = min(ny - 1, iy0 + hw);
        const int wy = iyb - iya + 1, nr = (ixb - ixa + 1) * wy;
        auto row = [&](int j) { return (ixa + j / wy) * ny + iya + j % wy; };
        const float rs0 = rsum0[n];
        const float2 *rb0 = rspec + (size_t)n * R * kSlots;
        const size_t img_stride = (size_t)S * R * kSlots;
        float2 *xb = fbuf[wave] + (lane >> 4) * kFftLd;
        for (int r0 = 0; r0 < nr; r0 += NROW) {
            float acc[NROW][2][4];
#pragma unroll
            for (int r = 0; r < NROW; ++r)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[r][h][e] = 0.0f;
            const float2 *arow[NROW];
#pragma unroll
            for (int r = 0; r < NROW; ++r)
                arow[r] = spec + (size_t)p * img_stride + (size_t)row(min(r0 + r, nr - 1)) * R * kSlots;
            for (int i = 0; i < R; ++i) {
                const float4 b = load_part(rb0 + i * kSlots, lane);
                float4 a[NROW];
#pragma unroll
                for (int r = 0; r < NROW; ++r) a[r] = load_part(arow[r] + i * kSlots, lane);
                __builtin_amdgcn_sched_barrier(0);   // all of the ring's loads in flight before the FMAs
#pragma unroll
                for (int r = 0; r < NROW; ++r) part_fma(acc[r], b, a[r]);
            }
            wave_lds_sync();
            float2 nm[NROW];
#pragma unroll
            for (int r = 0; r < NROW; ++r) {
                nm[r] = norm[(size_t)p * S + row(min(r0 + r, nr - 1))];
                store_part_z(fbuf[wave] + r * kFftLd, acc[r], nm[r], rs0, lane);
            }
            wave_lds_sync();
            float2 x[16];
            ifft256_rows4(x, lane_row_of(nm[0].y, nm[NROW / 2].y, nm[NROW - 1].y, 0.0f, lane), xb, tw, u);
            // a window's rows are consecutive shifts up to the end of its column
            for (int r = 0; r < min(NROW, nr - r0);) {
                const int cnt = min(min(NROW, nr - r0) - r, wy - (r0 + r) % wy);
                peak_update<false, true>(st, x, r, cnt, row(r0 + r), lane, xb, nbuf[wave], allow);
                r += cnt;
            }
        }
    }
    write_rec(rec + item, st, nbuf[wave], lane);
}

// Is (m, s, t) of reference `ref` admitted by one of the particle's items?
__device__ __forceinline__ bool admitted(const PropItem *it, int K, int ref, int m, int s, int t,
                                         int ny, int hw) {
    const int ix = s / ny, iy = s % ny;
    const int bit = m * kRingLen + t;
    for (int k = 0; k < K; ++k) {
        if (it[k].ref != ref) continue;
        const int cx = it[k].s / ny, cy = it[k].s % ny;
        if (abs(ix - cx) <= hw && abs(iy - cy) <= hw && ((it[k].mask[bit >> 5] >> (bit & 31)) & 1u))
            return true;
    }
    return false;
}

// Edge test of a maximum (m, s, t) of reference `ref`: true when one of its
// neighbours (psi sample t +- 1, or the next shift in x or y inside the grid) is
// admitted by no item of that reference, i.e. the windows may have cut the
// search short.
__device__ __forceinline__ bool on_edge(const PropItem *it, int K, int ref, int m, int s, int t,
                                        int nx, int ny, int hw) {
    const int ix = s / ny, iy = s % ny;
    bool in = admitted(it, K, ref, m, s, (t + 1) & (kRingLen - 1), ny, hw) &&
              admitted(it, K, ref, m, s, (t + kRingLen - 1) & (kRingLen - 1), ny, hw);
    if (ix > 0) in = in && admitted(it, K, ref, m, s - ny, t, ny, hw);
    if (ix < nx - 1) in = in && admitted(it, K, ref, m, s + ny, t, ny, hw);
    if (iy > 0) in = in && admitted(it, K, ref, m, s - 1, t, ny, hw);
    if (iy < ny - 1) in = in && admitted(it, K, ref, m, s + 1, t, ny, hw);
    return !in;
}

__device__ __forceinline__ void decode_best(const PeakRec &r, int ref, int p, ShiftView acc,
                                            const float2 *shifts_f, int n_shift, size_t pp,
                                            int *best_ref, float *best_val, float *best_peak) {
    float ax = 0.0f, ay = 0.0f;
    if (acc.base) {
        ax = acc.base[(size_t)p * acc.stride];
        ay = acc.base[(size_t)p * acc.stride + 1];
    }
    const float2 sh = shifts_f[min(max(r.s, 0), n_shift - 1)];
    best_ref[pp] = ref;
    best_val[pp] = r.val;
    best_peak[4 * pp + 0] = wizard_angle(r);
    best_peak[4 * pp + 1] = ax + sh.x;
    best_peak[4 * pp + 2] = ay + sh.y;
    best_peak[4 * pp + 3] = r.m ? 1.0f : 0.0f;
}

// Best item per particle (value, then lower reference, mirror, shift, psi
// sample), decoded like the multi-reference wizard into the outputs at p_off + p;
// edge[p] = 1 when it failed the edge test (with edge_test) or no item had a
// valid sample.
__global__ void k_best_prop(const PeakRec *__restrict__ rec, const PropItem *__restrict__ items,
                            int n_img, int K, int nx, int ny, int hw, int edge_test, ShiftView acc,
                            const float2 *__restrict__ shifts_f, int n_shift, int p_off,
                            int *__restrict__ best_ref, float *__restrict__ best_val,
                            float *__restrict__ best_peak, int *__restrict__ edge) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img) return;
    int bk = -1;
    for (int k = 0; k < K; ++k) {
        const PropItem &it = items[(size_t)p * K + k];
        const PeakRec &r = rec[(size_t)p * K + k];
        if (it.ref < 0 || !(r.val > -3.40282e+38f)) continue;
        if (bk < 0) {
            bk = k;
            continue;
        }
        const PeakRec &b = rec[(size_t)p * K + bk];
        const int br = items[(size_t)p * K + bk].ref;
        const bool better = r.val > b.val ||
                            (r.val == b.val &&
                             (it.ref < br || (it.ref == br && (r.m < b.m || (r.m == b.m &&
                              (r.s < b.s || (r.s == b.s && r.t < b.t)))))));
        if (better) bk = k;
    }
    const size_t pp = (size_t)p_off + p;
    if (bk < 0) {
        best_ref[pp] = -1;
        best_val[pp] = -3.40282e+38f;
        best_peak[4 * pp] = best_peak[4 * pp + 1] = best_peak[4 * pp + 2] = best_peak[4 * pp + 3] = 0.0f;
        edge[p] = 1;
        return;
    }
    PeakRec r = rec[(size_t)p * K + bk];
    r.m = min(max(r.m, 0), 1);
    r.s = min(max(r.s, 0), n_shift - 1);
    r.t &= kRingLen - 1;
    const PropItem *it = items + (size_t)p * K;
    const int ref = it[bk].ref;
    decode_best(r, ref, p, acc, shifts_f, n_shift, pp, best_ref, best_val, best_peak);
    edge[p] = (edge_test && on_edge(it, K, ref, r.m, r.s, r.t, nx, ny, hw)) ? 1 : 0;
}

// Second level: the distinct valid references among particle idx[j]'s
// proposals -> cand[j][0..K), padded with -1 (reference 0 if none is valid).
__global__ void k_prop_refs(const int4 *__restrict__ prop, const int *__restrict__ idx, int n, int K,
                            int N, int *__restrict__ cand) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int p = idx[j];
    int c[kMaxProposals];
    int cnt = 0;
    for (int k = 0; k < K; ++k) {
        const int r = prop[(size_t)p * K + k].x;
        if (r < 0 || r >= N) continue;
        bool seen = false;
        for (int q = 0; q < cnt; ++q) seen = seen || c[q] == r;
        if (!seen) c[cnt++] = r;
    }
    if (cnt == 0) c[cnt++] = 0;
    for (int k = 0; k < K; ++k) cand[(size_t)j * K + k] = k < cnt ? c[k] : -1;
}

// Second-level shifts of a batch: for the particles flagged 1 (flag[p]), every
// shift the first level did not compute (done[p]); none for the others.
__global__ void k_level2_mask(const int *__restrict__ flag, int n, int S,
                              const unsigned long long *__restrict__ done,
                              unsigned long long *__restrict__ smask) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const unsigned long long full = S >= 64 ? ~0ull : ((1ull << S) - 1ull);
    smask[p] = flag[p] == 1 ? (full & ~done[p]) : 0ull;
}

// Best of the second-level records rec[j][K] (value, then lower reference) of
// batch particle idx[j], decoded into its outputs at p_off + idx[j];
// fallback = value below threshold.
__global__ void k_best_refs_level2(const PeakRec *__restrict__ rec, const int *__restrict__ cand,
                                   int n, int K, ShiftView acc,
                                   const float2 *__restrict__ shifts_f, int n_shift,
                                   const int *__restrict__ idx, int p_off, float threshold,
                                   int *__restrict__ best_ref, float *__restrict__ best_val,
                                   float *__restrict__ best_peak, int *__restrict__ fallback) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    int bk = 0;   // entry 0 always holds a reference
    for (int k = 1; k < K; ++k) {
        if (cand[(size_t)j * K + k] < 0) continue;
        const float v = rec[(size_t)j * K + k].val, bv = rec[(size_t)j * K + bk].val;
        if (v > bv || (v == bv && cand[(size_t)j * K + k] < cand[(size_t)j * K + bk])) bk = k;
    }
    const PeakRec r = rec[(size_t)j * K + bk];
    const int p = idx[j];
    float2 a = f2(0.0f, 0.0f);
    if (acc.base) a = f2(acc.base[(size_t)p * acc.stride], acc.base[(size_t)p * acc.stride + 1]);
    const float2 sh = shifts_f[min(max(r.s, 0), n_shift - 1)];
    const size_t pp = (size_t)p_off + p;
    best_ref[pp] = cand[(size_t)j * K + bk];
    best_val[pp] = r.val;
    best_peak[4 * pp + 0] = wizard_angle(r);
    best_peak[4 * pp + 1] = a.x + sh.x;
    best_peak[4 * pp + 2] = a.y + sh.y;
    best_peak[4 * pp + 3] = r.m ? 1.0f : 0.0f;
    fallback[pp] = (r.val >= threshold) ? 0 : 1;
}

// fallback = 2 when the proposal confidence is below conf_min (straight to the
// exhaustive search), else 1 for an edge maximum or a value below the threshold
// (NaN included), else 0.
__global__ void k_fallback_flags(const float *__restrict__ best_val, const int *__restrict__ edge,
                                 const float *__restrict__ conf, float conf_min, int n_img,
                                 float threshold, int p_off, int *__restrict__ fallback) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img) return;
    const size_t pp = (size_t)p_off + p;
    int f = (edge[p] || !(best_val[pp] >= threshold)) ? 1 : 0;
    if (conf && !(conf[pp] >= conf_min)) f = 2;
    fallback[pp] = f;
}

// Indices of the particles whose flag lies in [lo, hi] (any order).
__global__ void k_compact(const int *__restrict__ flag, int n, int lo, int hi, int *__restrict__ idx,
                          int *__restrict__ count) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || flag[p] < lo || flag[p] > hi) return;
    idx[atomicAdd(count, 1)] = p;
}

// Copies the images (and accumulated shifts) of the listed particles.
__global__ void k_gather(const float *__restrict__ imgs, int D, ShiftView acc,
                         const int *__restrict__ idx, int n, float *__restrict__ out,
                         float2 *__restrict__ out_acc) {
    const int j = blockIdx.x;
    if (j >= n) return;
    const int p = idx[j];
    const float *src = imgs + (size_t)p * D * D;
    float *dst = out + (size_t)j * D * D;
    for (int i = threadIdx.x; i < D * D; i += blockDim.x) dst[i] = src[i];
    if (threadIdx.x == 0)
        out_acc[j] = acc.base ? f2(acc.base[(size_t)p * acc.stride], acc.base[(size_t)p * acc.stride + 1])
                              : f2(0.0f, 0.0f);
}

// Exhaustive records rec[j][N] of gathered particle j -> best reference (first
// maximum over references), decoded into the outputs of particle idx[j0 + j].
__global__ void k_best_refs_scatter(const PeakRec *__restrict__ rec, int n, int N,
                                    const float2 *__restrict__ acc, const float2 *__restrict__ shifts_f,
                                    int n_shift, const int *__restrict__ idx, int *__restrict__ best_ref,
                                    float *__restrict__ best_val, float *__restrict__ best_peak) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    int bn = 0;
    for (int k = 1; k < N; ++k)
        if (rec[(size_t)j * N + k].val > rec[(size_t)j * N + bn].val) bn = k;
    const PeakRec r = rec[(size_t)j * N + bn];
    const float2 a = acc[j];
    const float2 sh = shifts_f[min(max(r.s, 0), n_shift - 1)];
    const size_t pp = (size_t)idx[j];
    best_ref[pp] = bn;
    best_val[pp] = r.val;
    best_peak[4 * pp + 0] = wizard_angle(r);
    best_peak[4 * pp + 1] = a.x + sh.x;
    best_peak[4 * pp + 2] = a.y + sh.y;
    best_peak[4 * pp + 3] = r.m ? 1.0f : 0.0f;
}

// Best candidate per particle -> reference index, peak value, {angle, sx, sy, mirror}.
__global__ void k_decode_best(const PeakRec *__restrict__ rec, const int *__restrict__ cand,
                              const int *__restrict__ best, const int *__restrict__ tie, int n_img,
                              int K, ShiftView acc, const float2 *__restrict__ shifts_f,
                              int n_shift, int p_off, int *__restrict__ best_ref,
                              float *__restrict__ best_val, float *__restrict__ best_peak,
                              int *__restrict__ tie_out, const int *__restrict__ idx) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_img) return;
    const int k = max(best[p], 0);
    const PeakRec r = rec[(size_t)p * K + k];
    float ax = 0.0f, ay = 0.0f;
    if (acc.base) {
        ax = acc.base[(size_t)p * acc.stride];
        ay = acc.base[(size_t)p * acc.stride + 1];
    }
    const float2 sh = shifts_f[min(max(r.s, 0), n_shift - 1)];
    // output slot: p_off + p, or idx[p_off + p] (a scatter to the caller's particles)
    const size_t pp = idx ? (size_t)idx[(size_t)p_off + p] : (size_t)p_off + p;
    best_ref[pp] = cand[(size_t)p * K + k];
    best_val[pp] = r.val;
    best_peak[4 * pp + 0] = wizard_angle(r);
    best_peak[4 * pp + 1] = ax + sh.x;
    best_peak[4 * pp + 2] = ay + sh.y;
    best_peak[4 * pp + 3] = r.m ? 1.0f : 0.0f;
    if (tie_out) tie_out[pp] = tie[p];
}

// Multi-reference decode (reference wizard, cuda/gpu_aln_noref.cu:1758-1793, with
// its float/double mix) and output scatter (:517-540).
__global__ void k_decode_mref(const PeakRec *__restrict__ rec, int n_img, int N, ShiftView acc,
                              const float2 *__restrict__ shifts_f, int n_shift, float *__restrict__ peak,
                              int peak_row, int p_off, float *__restrict__ d, int d_pitch) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_img * N) return;
    const int p = idx / N, n = idx % N;
    const PeakRec r = rec[idx];
    const float angle = wizard_angle(r);
    float ax = 0.0f, ay = 0.0f;
    if (acc.base) {
        ax = acc.base[(size_t)p * acc.stride];
        ay = acc.base[(size_t)p * acc.stride + 1];
    }
    const float2 sh = shifts_f[min(max(r.s, 0), n_shift - 1)];
    const size_t pp = (size_t)p_off + p;
    d[(size_t)n * d_pitch + pp] = r.val;
    float *pk = peak + (size_t)n * peak_row + 4 * pp;
    pk[0] = angle;
    pk[1] = ax + sh.x;
    pk[2] = ay + sh.y;
    pk[3] = r.m ? 1.0f : 0.0f;
}

// Pre-align / reference-free decode (cuda/gpu_aln_noref.cu:2486-2519, FP64
// parabola :2558-2581).
__global__ void k_decode_single(const PeakRec *__restrict__ rec, int cnt, DevParam *__restrict__ prm,
                                const float2 *__restrict__ shifts_f, int n_shift, float lim) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cnt) return;
    const PeakRec r = rec[i];
    DevParam q = prm[i];
    double x[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) x[k] = (double)r.x[k];
    const double c2 = 49. * x[0] + 6. * x[1] - 21. * x[2] - 32. * x[3] - 27. * x[4] - 6. * x[5] + 31. * x[6];
    const double c3 = 5. * x[0] - 3. * x[2] - 4. * x[3] - 3. * x[4] + 5. * x[6];
    const double step = 360.0 / (double)kRingLen;
    double interp = step * (double)r.t;
    if (c3 != 0.0) interp = interp + step * (c2 / (2.0 * c3) - 4.0);
    q.mirror = (r.m == 1);
    const float2 sh = shifts_f[min(max(r.s, 0), n_shift - 1)];
    q.shift_x += sh.x;
    q.shift_y += sh.y;
    q.shift_x = fminf(fmaxf(q.shift_x, -lim), lim);
    q.shift_y = fminf(fmaxf(q.shift_y, -lim), lim);
    q.angle = (float)(360.0 - interp);
    if (q.mirror) {
        q.angle = (float)((double)q.angle + 180.0);
        if (q.angle >= 360.0f) q.angle = (float)((double)q.angle - 360.0);
    }
    prm[i] = q;
}

// ------------------------------------------------- averages of transformed images
// Pixel (x, y) of image p after the transform of cu_transform_batch
// (cuda/gpu_aln_noref.cu:1558-1588): mirror (x -> D - x), rotate by +angle about D / 2,
// add the accumulated shift.  t = (cos, sin, shift_x, shift_y).
__device__ __forceinline__ Quad transformed_quad(const float *imgs, int D, int p, int x, int y, float4 t, int mir) {
    const float c = (float)(D / 2);
    float sx = mir ? (float)(D - x) : (float)x;
    float sy = (float)y;
    sx -= c;
    sy -= c;
    const float tx = sx;
    sx = tx * t.x - sy * t.y;
    sy = tx * t.y + sy * t.x;
    sx += c;
    sy += c;
    return load_quad(imgs + (size_t)p * D * D, D, sx + t.z, sy + t.w);
}

// Sum over j in [a, b), in that order, of pixel (x, y) of the transformed images members[j]
// (j itself without a list).  What bounds it is the latency of the list, the parameters
// and the pixels, so eight members are loaded at once and added in order, and the cache
// lines a wavefront's taps touch (average_tile).  20000 images of 76 x 76 in 100 classes
// (0.46 GB): 244 us; 434 with lines of 64 pixels a wavefront, 614 with one member at a time.
__device__ __forceinline__ float transformed_sum(const float *__restrict__ imgs, int D, int x, int y, int a, int b,
                                                 const int *__restrict__ members, const float4 *__restrict__ tp,
                                                 const int *__restrict__ mir) {
    float s = 0.0f;
    int j = a;
    for (; j + 8 <= b; j += 8) {
        Quad q[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int i = members ? members[j + n] : j + n;
            q[n] = transformed_quad(imgs, D, i, x, y, tp[i], mir[i]);
        }
#pragma unroll
        for (int n = 0; n < 8; ++n) s += mix_quad(q[n], D);
    }
    for (; j < b; ++j) {
        const int i = members ? members[j] : j;
        s += mix_quad(transformed_quad(imgs, D, i, x, y, tp[i], mir[i]), D);
    }
    return s;
}

// Block (16 x 16 pixels, group), 8 x 8 pixels a wavefront: a rotated square of 64 pixels
// lies in about 11 rows of the image, a rotated line of 64 in up to 64.  All tiles of a
// group run on one XCD, whose L2 then fetches each image once for them.
struct AverageTile {
    int x, y, group;
};
__device__ __forceinline__ AverageTile average_tile(int D) {
    const int nt = (D + 15) >> 4;
    const int b = xcd_remap(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int t = b % (nt * nt), l = threadIdx.x;
    return {(t % nt) * 16 + ((l >> 6) & 1) * 8 + (l & 7), (t / nt) * 16 + (l >> 7) * 8 + ((l >> 3) & 7), b / (nt * nt)};
}
static dim3 average_grid(int D, int groups) { return dim3(((D + 15) / 16) * ((D + 15) / 16), groups); }

// Class averages of the transformed images of particles [cid_idx[k], cid_idx[k + 1])
// (cu_average_batch, cuda/gpu_aln_noref.cu:1605-1621); an empty class keeps its reference.
// 3000 images of 76 x 76, 30 classes: 52 us; 800 when a pass wrote the transformed images
// and a workgroup per class added them.
__global__ __launch_bounds__(256) void k_class_average(const float *__restrict__ imgs, int D,
                                                       const int *__restrict__ cid_idx,
                                                       const float4 *__restrict__ tp, const int *__restrict__ mir,
                                                       float *__restrict__ refs) {
    const AverageTile t = average_tile(D);
    const int k = t.group, a = cid_idx[k], b = cid_idx[k + 1];
    if (t.x >= D || t.y >= D || b <= a) return;
    refs[((size_t)k * D + t.y) * D + t.x] =
        transformed_sum(imgs, D, t.x, t.y, a, b, nullptr, tp, mir) / (float)(b - a);
}

// ------------------------------------------------------ pre-alignment loop
// The average of every particle transformed with its current parameters (the
// image transform of transformed_quad), without materialising the transformed stack:
// per particle the rotation (cos, sin), shifts and mirror; partial sums over
// chunks of kPreChunk particles per pixel; then the chunks in order, divided by P.
constexpr int kPreChunk = 256;

__global__ __launch_bounds__(256) void k_pre_tp(const DevParam *__restrict__ prm, int P,
                                                float4 *__restrict__ tp, int *__restrict__ mir) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const DevParam q = prm[p];
    const float ang = (3.141592653589793f / 180.0f) * q.angle;
    tp[p] = make_float4(cosf(ang), sinf(ang), q.shift_x, q.shift_y);
    mir[p] = q.mirror ? 1 : 0;
}

__global__ __launch_bounds__(256) void k_pre_partial(const float *__restrict__ imgs, int D, int P,
                                                     const float4 *__restrict__ tp,
                                                     const int *__restrict__ mir,
                                                     float *__restrict__ part) {
    const AverageTile t = average_tile(D);
    const int c = t.group;
    if (t.x >= D || t.y >= D) return;
    part[((size_t)c * D + t.y) * D + t.x] =
        transformed_sum(imgs, D, t.x, t.y, c * kPreChunk, min((c + 1) * kPreChunk, P), nullptr, tp, mir);
}

__global__ __launch_bounds__(256) void k_pre_finish(const float *__restrict__ part, int D, int P,
                                                    int n_chunks, float *__restrict__ avg) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= D * D) return;
    double s = 0.0;
    for (int c = 0; c < n_chunks; ++c) s += (double)part[(size_t)c * D * D + idx];
    avg[idx] = (float)(s / (double)P);
}

// Centring shift of the average from the particles' shifts after the driver's
// rotation (bin/sp_isac_applications.py:1664-1690): sx_sum = sum of +-shift_x'
// (minus for mirrored particles), sy_sum = sum of shift_y'; the average is then
// moved by (-sx_sum / P, -sy_sum / P) (:1547-1552).  One workgroup, FP64 sums.
__global__ __launch_bounds__(256) void k_pre_center(const DevParam *__restrict__ prm, int P,
                                                    float2 *__restrict__ shift) {
    __shared__ double rx[256], ry[256];
    double sx = 0.0, sy = 0.0;
    for (int p = threadIdx.x; p < P; p += blockDim.x) {
        const DevParam q = prm[p];
        const double a = (double)q.angle * (M_PI / 180.0);
        const double c = cos(a), sn = -sin(a);
        const double nx = -(double)q.shift_x, ny = -(double)q.shift_y;
        const double px = nx * c - ny * sn, py = nx * sn + ny * c;
        sx += q.mirror ? -px : px;
        sy += py;
    }
    rx[threadIdx.x] = sx;
    ry[threadIdx.x] = sy;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            rx[threadIdx.x] += rx[threadIdx.x + o];
            ry[threadIdx.x] += ry[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) shift[0] = make_float2((float)(-rx[0] / P), (float)(-ry[0] / P));
}

// ------------------------------------------------------- reference update
// Device form of the multi-reference driver's reference update
// (bin/sp_isac2_gpu.py:1146-1232): every particle is transformed with the
// parameters of its class's peak and added to that class's average, the average
// shift of each class centres the new reference, and each particle's shifts are
// re-expressed about that centre.

// Per particle i of class k = cls[i]: the peak (angle, sx, sy, mirror) of
// peak_list[k][4i..4i+3] as the library writes it.  tp[i] = (cos, sin, sx, sy) for
// the image transform of transformed_quad; post[i] = the shifts after the driver's
// rotation (bin/sp_isac2_gpu.py:1016-1022, in FP32 like the driver's numpy code).
// A class id outside [0, N) sets *bad and gives the particle neutral values.
__global__ void k_upd_params(const float *__restrict__ peak, int P, int N,
                             const int *__restrict__ cls, float4 *__restrict__ tp,
                             int *__restrict__ mir, float2 *__restrict__ post,
                             float4 *__restrict__ raw, int *__restrict__ bad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    const int k = cls[i];
    if (k < 0 || k >= N) {
        atomicOr(bad, 1);
        tp[i] = make_float4(1.0f, 0.0f, 0.0f, 0.0f);
        mir[i] = 0;
        post[i] = f2(0.0f, 0.0f);
        raw[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const float *q = peak + (size_t)k * 4 * P + 4 * (size_t)i;
    const float a = q[0], sx = q[1], sy = q[2], m = q[3];
    const float ang = (3.141592653589793f / 180.0f) * a;   // as k_pre_tp
    tp[i] = make_float4(cosf(ang), sinf(ang), sx, sy);
    mir[i] = (m != 0.0f) ? 1 : 0;
    raw[i] = make_float4(a, sx, sy, m);
    const float rad = a * (float)(3.141592653589793 / 180.0);
    const float c = cosf(rad), sn = -sinf(rad);
    const float sxn = -sx, syn = -sy;
    post[i] = f2(sxn * c - syn * sn, sxn * sn + syn * c);
}

// Block k: the particles of class k in ascending order.  pass 0 counts them into
// cnt[k]; pass 1 writes them to members[off[k] ...].  A chain of two barriers a chunk:
// chunks of 1024 particles (20000 x 100: 13 us a pass, 27 in chunks of 256).
template <int PASS>
__global__ __launch_bounds__(1024) void k_class_members(const int *__restrict__ cls, int P,
                                                       int *__restrict__ cnt,
                                                       const int *__restrict__ off,
                                                       int *__restrict__ members) {
    __shared__ int wsum[16];
    const int k = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int base = PASS ? off[k] : 0;
    for (int p0 = 0; p0 < P; p0 += 1024) {
        const int i = p0 + tid;
        const bool hit = i < P && cls[i] == k;
        const unsigned long long m = __ballot(hit);
        if (lane == 0) wsum[w] = __popcll(m);
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            before += (v < w) ? wsum[v] : 0;
            total += wsum[v];
        }
        if (PASS && hit) {
            const unsigned long long lt = (lane == 0) ? 0ull : (m & (~0ull >> (64 - lane)));
            members[base + before + __popcll(lt)] = i;
        }
        base += total;
        __syncthreads();
    }
    if (!PASS && tid == 0) cnt[k] = base;
}

// Exclusive scan of cnt[0..N) into off[0..N] (one block).
__global__ void k_scan_counts(const int *__restrict__ cnt, int N, int *__restrict__ off) {
    if (threadIdx.x != 0) return;
    int s = 0;
    for (int k = 0; k < N; ++k) {
        off[k] = s;
        s += cnt[k];
    }
    off[N] = s;
}

// One wavefront per class: the shift sums of the driver (mirrored particles enter
// with -sx), summed in double in ascending particle order, rounded to float as the
// driver's MPI_FLOAT reduction does, divided by the member count in double.
// neg[k] = -(avg_x, avg_y) (the centring shift of the new reference); avg_out and
// members_out (either may be NULL) receive (avg_x, avg_y) as floats and the counts.
// 64 members are loaded at once; lane 0 adds the x in order, lane 1 the y (20000 x 100:
// 6 us; 85 with a thread per class).
__global__ __launch_bounds__(64) void k_class_shift(const int *__restrict__ off, const int *__restrict__ members,
                                                    int N, const float2 *__restrict__ post,
                                                    const int *__restrict__ mir, double2 *__restrict__ avg,
                                                    float2 *__restrict__ neg, float2 *__restrict__ avg_out,
                                                    int *__restrict__ members_out) {
    __shared__ double v[2][64];
    const int k = blockIdx.x, lane = threadIdx.x;
    const int a = off[k], b = off[k + 1];
    double s = 0.0;
    for (int j = a; j < b; j += 64) {
        if (j + lane < b) {
            const int i = members[j + lane];
            const float2 q = post[i];
            v[0][lane] = mir[i] ? -(double)q.x : (double)q.x;
            v[1][lane] = (double)q.y;
        }
        wave_lds_sync();
        if (lane < 2) {
            const int n = min(64, b - j);
#pragma unroll 8
            for (int m = 0; m < n; ++m) s += v[lane][m];
        }
        wave_lds_sync();
    }
    const double sx = s, sy = __shfl(s, 1, kWave);
    if (lane != 0) return;
    double ax = 0.0, ay = 0.0;
    if (b > a) {
        ax = (double)(float)sx / (double)(b - a);
        ay = (double)(float)sy / (double)(b - a);
    }
    avg[k] = make_double2(ax, ay);
    neg[k] = f2((float)-ax, (float)-ay);
    if (avg_out) avg_out[k] = f2((float)ax, (float)ay);
    if (members_out) members_out[k] = b - a;
}

// Per particle: (angle, sx -/+ avg_x, sy - avg_y, mirror) in the driver's
// convention (bin/sp_isac2_gpu.py:1200-1208).
__global__ void k_upd_params_out(const int *__restrict__ cls, int P, int N,
                                 const float4 *__restrict__ raw, const float2 *__restrict__ post,
                                 const int *__restrict__ mir, const double2 *__restrict__ avg,
                                 float4 *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    const int k = cls[i];
    if (k < 0 || k >= N) {
        out[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const double2 g = avg[k];
    const float2 q = post[i];
    const double x = mir[i] ? (double)q.x + g.x : (double)q.x - g.x;
    out[i] = make_float4(raw[i].x, (float)x, (float)((double)q.y - g.y), raw[i].w);
}

// Block (tile, k): pixels of class k's average.  Each member image is transformed
// (transformed_quad) and added in ascending particle order; the sum is scaled
// by 1 / members (a class without members gives zeros).
__global__ __launch_bounds__(256) void k_class_transform_average(
    const float *__restrict__ imgs, int D, const int *__restrict__ off,
    const int *__restrict__ members, const float4 *__restrict__ tp, const int *__restrict__ mir,
    float *__restrict__ refs) {
    const AverageTile t = average_tile(D);
    if (t.x >= D || t.y >= D) return;
    const int k = t.group, a = off[k], b = off[k + 1];
    const float s = transformed_sum(imgs, D, t.x, t.y, a, b, members, tp, mir);
    refs[((size_t)k * D + t.y) * D + t.x] = (b > a) ? s * (1.0f / (float)(b - a)) : 0.0f;
}

// Tangent filter, three separable passes over a half-plane spectrum
// F[n][ky][kx], kx = 0..D/2 (cuda/gpu_aln_noref.cu:1007-1037, :2203-2266).
__global__ void k_row_dft(const float *__restrict__ refs, int D, float2 *__restrict__ F,
                          const float2 *__restrict__ tw) {
    const int n = blockIdx.y, y = blockIdx.x, Dh = D / 2 + 1;
    const float *row = refs + ((size_t)n * D + y) * D;
    for (int kx = threadIdx.x; kx < Dh; kx += blockDim.x) {
        float re = 0.0f, im = 0.0f;
        for (int x = 0; x < D; ++x) {
            const float2 w = tw[(x * kx) % D];
            re += row[x] * w.x;
            im += row[x] * w.y;
        }
        F[((size_t)n * D + y) * Dh + kx] = f2(re, im);
    }
}

// Column pass: forward DFT over y, the tanh low-pass, and (shift != NULL) the phase
// ramp exp(-2 pi i (kx dx + ky dy) / D) that moves image n's content by
// shift[n] = (dx, dy) (signed ky; ky = D/2 taken as +D/2), then the inverse DFT.
// abs_freq = 0: the reference's frequency coordinates (x = kx / (D/2+1) / 2,
// y = min(ky, D-ky) / D); 1: absolute frequency in cycles per pixel
// (x = kx / D, y = min(ky, D-ky) / D).
__global__ void k_col_filter(float2 *__restrict__ F, int D, const float2 *__restrict__ tw,
                             float cutoff, float falloff, const float2 *__restrict__ shift,
                             int abs_freq) {
    extern __shared__ float2 col[];
    const int n = blockIdx.y, kx = blockIdx.x, Dh = D / 2 + 1;
    float2 *base = F + (size_t)n * D * Dh + kx;
    const float cc = 3.141592653589793f / (2.0f * falloff * cutoff);
    const float xx = abs_freq ? (float)kx / (float)D : (float)kx / (float)Dh * 0.5f;
    const float half = (float)D / 2.0f;
    const float2 sh = shift ? shift[n] : f2(0.0f, 0.0f);
    for (int ky = threadIdx.x; ky < D; ky += blockDim.x) {
        float re = 0.0f, im = 0.0f;
        for (int y = 0; y < D; ++y) {
            const float2 v = base[(size_t)y * Dh];
            const float2 w = tw[(y * ky) % D];
            re += v.x * w.x - v.y * w.y;
            im += v.x * w.y + v.y * w.x;
        }
        float yy = ((float)ky < half) ? (float)ky : (float)(D - ky);
        yy = yy / half * 0.5f;
        const float dd = sqrtf(xx * xx + yy * yy);
        // cutoff <= 0: no low-pass (the phase ramp alone)
        const float h = cutoff > 0.0f ? 0.5f * (tanhf(cc * (dd + cutoff)) - tanhf(cc * (dd - cutoff)))
                                      : 1.0f;
        re *= h;
        im *= h;
        if (shift) {
            const int kys = (2 * ky > D) ? ky - D : ky;
            float t = ((float)kx * sh.x + (float)kys * sh.y) / (float)D;   // turns
            t -= rintf(t);
            float sn, cs;
            sincospif(-2.0f * t, &sn, &cs);
            const float r2 = re * cs - im * sn;
            im = re * sn + im * cs;
            re = r2;
        }
        col[ky] = f2(re, im);
    }
    __syncthreads();
    for (int y = threadIdx.x; y < D; y += blockDim.x) {
        float re = 0.0f, im = 0.0f;
        for (int ky = 0; ky < D; ++ky) {
            const float2 v = col[ky];
            const float2 w = tw[(y * ky) % D];  // conj for the inverse
            re += v.x * w.x + v.y * w.y;
            im += v.y * w.x - v.x * w.y;
        }
        base[(size_t)y * Dh] = f2(re, im);
    }
}

// Row C2R.  gain > 0 scales every image by gain; otherwise the reference's
// scaling: 1 / (D*D)^2 for image 0 only (quirk of cuda/gpu_aln_noref.cu:2235-2262).
__global__ void k_row_c2r(float *__restrict__ refs, int D, const float2 *__restrict__ F,
                          const float2 *__restrict__ tw, float gain_all) {
    const int n = blockIdx.y, y = blockIdx.x, Dh = D / 2 + 1;
    const float2 *row = F + ((size_t)n * D + y) * Dh;
    const float dd = (float)D * (float)D;
    const float gain = gain_all > 0.0f ? gain_all : ((n == 0) ? 1.0f / (dd * dd) : 1.0f);
    for (int x = threadIdx.x; x < D; x += blockDim.x) {
        float s = 0.0f;
        for (int kx = 0; kx < Dh; ++kx) {
            const float2 v = row[kx];
            const float2 w = tw[(x * kx) % D];  // e^{+i}: (w.x, -w.y)
            const float re = v.x * w.x + v.y * w.y;
            const bool edge = (kx == 0) || ((D % 2 == 0) && kx == D / 2);
            s += edge ? re : 2.0f * re;
        }
        refs[((size_t)n * D + y) * D + x] = s * gain;
    }
}

}  // namespace

// ---------------------------------------------------------------- launchers

// Launch shape of the polar pass.  A workgroup's wavefronts take the row groups (four
// shifts each) in equal passes: 13 groups run as 2 x 7, not 8 + 5.  Up to 8 wavefronts
// where two workgroups fit in a CU's LDS, up to 16 where only one does.  With fewer
// groups than the chip has wavefront slots (16 per CU), a workgroup takes one group, its
// ring pairs spread over the wavefronts: 24 images of 64 x 64, 9 shifts, 29 rings take 21 us
// instead of 77.
struct PolarShape {
    int waves, rows, spread;
};
static int polar_wave_cap(int img_dim) {
    return 2 * polar_lds_floats(img_dim, 8) * sizeof(float) <= 160 * 1024 - 4096 ? 8 : 16;
}
static int polar_waves(int n_shift, int img_dim) {
    const int g = (n_shift + 3) / 4;
    const int cap = polar_wave_cap(img_dim);
    const int passes = (g + cap - 1) / cap;
    return (g + passes - 1) / passes;
}
// Cost of an image's n ring pairs of wavefronts by workgroups of nw wavefronts of which busy
// have any: the vector unit's time, and more where fewer than nine of a CU's are busy (seven
// of 128 x 128, 25 shifts: 11.6 ns a pair, nine to sixteen 9.4 to 9.9, three 21).
static double polar_cost(int img_dim, int nw, int busy, double n) {
    const int fit = (int)(160 * 1024 / (polar_lds_floats(img_dim, nw) * sizeof(float) + 512));
    return n / std::min(1.0, busy * std::max(1, std::min(fit, 16 / nw)) / 9.0);
}
// Wavefronts of the spread form of n_rows rows, or 0 where `plain` unspread ones are the better
// form: a spread pair costs 6 to 12 % more, by 25 and 49 shifts of 76 x 76.
static int polar_spread(int n_rows, int img_dim, int n_ring, int plain) {
    const long long pairs = (n_ring + 1) / 2, g = (n_rows + 3) / 4, tasks = n_rows * pairs;
    int nw = 4;   // the smallest workgroup of which a CU holds 16 wavefronts
    while (nw < 16 && 16 / nw * (polar_lds_floats(img_dim, nw) * sizeof(float) + 512) > 160 * 1024) nw *= 2;
    if (tasks < 4 * nw) nw = tasks <= 16 ? (int)(tasks + 3) / 4 : (int)(tasks + 15) / 16 * 4;
    const double spread = 1.06 * ((tasks + 4 * nw - 1) / (4 * nw) * nw);
    return polar_cost(img_dim, nw, nw, spread) <
                   0.95 * polar_cost(img_dim, plain, (int)std::min<long long>(g, plain), (double)(g * pairs))
               ? nw
               : 0;
}
static PolarShape polar_shape(long long n_img, int n_shift, int img_dim, int n_ring) {
    const int g = (n_shift + 3) / 4, pairs = (n_ring + 1) / 2;
    const long long fill = 4096 / (n_img * g);
    if (fill >= 2 && pairs >= 2) {
        const int split = (int)std::min<long long>({fill, (std::min(n_shift, 4) * pairs + 3) / 4, 16});
        return {split, 4, 1};
    }
    const int plain = polar_waves(n_shift, img_dim), nw = polar_spread(n_shift, img_dim, n_ring, plain);
    return {nw ? nw : plain, n_shift, nw > 0};
}

constexpr int kPropLds = 4 * kFftLd * sizeof(float2);   // of k_ccf_prop, a proposal

hipError_t prepare_launches() {
    static bool lds_raised = false;
    if (!lds_raised) {
        const int lds = (int)(polar_lds_floats(kMaxImgDim, 16) * sizeof(float));
        hipError_t e = hipFuncSetAttribute((const void *)k_ref_spectra, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)(polar_lds_floats(kMaxImgDim, 16) * sizeof(float)));
        if (e != hipSuccess) return e;
        e = hipFuncSetAttribute((const void *)k_polar_single, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        for (const void *fn : {(const void *)k_polar_spectra<false, false>, (const void *)k_polar_spectra<false, true>,
                               (const void *)k_polar_spectra<true, false>, (const void *)k_polar_spectra<true, true>}) {
            e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess) return e;
        }
        for (const void *fn : {(const void *)k_ccf_prop<1>, (const void *)k_ccf_prop<3>}) {
            e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxProposals * kPropLds);
            if (e != hipSuccess) return e;
        }
        const int lds_frag = (int)((256 + 4 * 512) * sizeof(float2) +
                                   (kMaxImgDim + 2 * kFragBorder) * (kMaxImgDim + 2 * kFragBorder) *
                                       sizeof(float));
        e = hipFuncSetAttribute((const void *)k_polar_frag<false>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_frag);
        if (e != hipSuccess) return e;
        e = hipFuncSetAttribute((const void *)k_polar_frag<true>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_frag);
        if (e != hipSuccess) return e;
        lds_raised = true;
    }
    return hipSuccess;
}

hipError_t launch_polar_spectra(const float *imgs, int n_img, int img_dim, ShiftView acc,
                                const int2 *shift_i, int n_shift, const float2 *tmpl, int n_ring,
                                const float2 *twiddle, float2 *spec, float2 *norm,
                                hipStream_t st) {
    if (n_img <= 0 || n_shift <= 0) return hipSuccess;
    if (hipError_t e = prepare_launches()) return e;
    const PolarShape ps = polar_shape(n_img, n_shift, img_dim, n_ring);
    const size_t lds = polar_lds_floats(img_dim, ps.waves) * sizeof(float);
    const auto kernel = ps.spread ? k_polar_spectra<false, true> : k_polar_spectra<false, false>;
    hipLaunchKernelGGL(kernel, dim3(n_img, (n_shift + ps.rows - 1) / ps.rows), dim3(64 * ps.waves), lds, st, imgs,
                       img_dim, acc, shift_i, n_shift, tmpl, n_ring, twiddle, spec, norm, nullptr, ps.rows);
    return hipGetLastError();
}

bool polar_frag_supported(int n_ring) { return n_ring >= 1 && n_ring <= kFragMaxRings; }

hipError_t launch_polar_frag(const float *imgs, int n_img, int img_dim, ShiftView acc,
                             const int2 *shift_i, int n_shift, int n_ring, bool bf16,
                             const float2 *twiddle, void *frag, hipStream_t st) {
    if (n_img <= 0 || n_shift <= 0) return hipSuccess;
    if (!polar_frag_supported(n_ring)) return hipErrorInvalidValue;
    const GemmLayout L = gemm_layout(n_ring);
    const int S_pad = gemm_rows_per_particle(n_shift);
    const size_t lds = (256 + 4 * 512) * sizeof(float2) +
                       (size_t)(img_dim + 2 * kFragBorder) * (img_dim + 2 * kFragBorder) * sizeof(float);
    if (hipError_t e = prepare_launches()) return e;
    const dim3 grid((unsigned)((n_img + 15) / 16 * 16));
    if (bf16)
        hipLaunchKernelGGL(k_polar_frag<true>, grid, dim3(256), lds, st, imgs, n_img, img_dim, acc,
                           shift_i, n_shift, S_pad, n_ring, L.full16, L.tail, L.slot_bytes, L.cp,
                           twiddle, (unsigned char *)frag);
    else
        hipLaunchKernelGGL(k_polar_frag<false>, grid, dim3(256), lds, st, imgs, n_img, img_dim, acc,
                           shift_i, n_shift, S_pad, n_ring, L.full16, L.tail, L.slot_bytes, L.cp,
                           twiddle, (unsigned char *)frag);
    return hipGetLastError();
}

hipError_t launch_polar_spectra_masked(const float *imgs, int n_img, int img_dim, ShiftView acc,
                                       const int2 *shift_i, int n_shift, const float2 *tmpl,
                                       int n_ring, const float2 *twiddle, float2 *spec,
                                       float2 *norm, const unsigned long long *smask,
                                       int n_rows, hipStream_t st) {
    if (n_img <= 0 || n_shift <= 0) return hipSuccess;
    if (n_shift > 64) return hipErrorInvalidValue;
    if (hipError_t e = prepare_launches()) return e;
    // as many wavefronts as fit: how many of a particle's shifts are set is not known here,
    // and about 30 of 49 (8 windows) are one pass of 8 wavefronts but two of 7 (10 000 images
    // of 76 x 76: 3.9 ms against 4.1).  About 9 (one window) spread: 1.20 ms, unspread 1.73
    const int plain = std::min((n_shift + 3) / 4, polar_wave_cap(img_dim));
    const int nw = polar_spread(n_rows, img_dim, n_ring, plain);
    const PolarShape ps{nw ? nw : plain, n_shift, nw > 0};
    const size_t lds = polar_lds_floats(img_dim, ps.waves) * sizeof(float);
    const auto kernel = ps.spread ? k_polar_spectra<true, true> : k_polar_spectra<true, false>;
    hipLaunchKernelGGL(kernel, dim3(n_img), dim3(64 * ps.waves), lds, st, imgs, img_dim, acc, shift_i, n_shift, tmpl,
                       n_ring, twiddle, spec, norm, smask, n_shift);
    return hipGetLastError();
}

hipError_t launch_ref_spectra(const float *imgs, int n_ref, int img_dim, const float2 *tmpl, int n_ring,
                              const float2 *twiddle, float2 *rspec, float *rsum0, hipStream_t st) {
    if (n_ref <= 0) return hipSuccess;
    if (hipError_t e = prepare_launches()) return e;
    const int nw = (n_ring + 7) / 8;   // wavefronts of four ring pairs
    hipLaunchKernelGGL(k_ref_spectra, dim3(n_ref), dim3(64 * nw), polar_lds_floats(img_dim, nw) * sizeof(float), st,
                       imgs, img_dim, tmpl, n_ring, twiddle, rspec, rsum0);
    return hipGetLastError();
}

// Particles per workgroup of the search, 1, 2, 4 or 8: a run of cp particles fills
// ceil(cp S / 8) row blocks (8 particles fill S without a partial block), and the
// device holds one workgroup per CU at a time.  The count with the fewest block steps
// (rounds of workgroups x blocks of each) wins, at equal cost the larger run.  4 096 x
// 100 at 76 px, 49 shifts: 13.5 ms with 8, 14.3 with 4, 15.5 with 1 (7 blocks for 6.1);
// small searches take 1, so that every CU has work.
static int particles_per_workgroup(int n_img, int S, int N) {
    const long long ng = (N + kMrefRefs - 1) / kMrefRefs, cus = 256;
    int best = 1;
    long long best_cost = LLONG_MAX;
    for (int cp = 1; cp <= 8; cp *= 2) {
        const long long wgs = ((long long)n_img + cp - 1) / cp * ng;
        const long long cost = (wgs + cus - 1) / cus * (((long long)cp * S + 7) / 8);
        if (cost <= best_cost) {
            best_cost = cost;
            best = cp;
        }
    }
    return best;
}

hipError_t launch_ccf_mref(const float2 *spec, const float2 *norm, const float2 *rspec,
                           const float *rsum0, int n_img, int n_shift, int n_ring, int n_ref,
                           const float2 *twiddle, PeakRec *rec, hipStream_t st) {
    if (n_img <= 0 || n_ref <= 0) return hipSuccess;
    const int cp = particles_per_workgroup(n_img, n_shift, n_ref);
    const long long ng = (n_ref + kMrefRefs - 1) / kMrefRefs;
    const dim3 wg(kMrefWaves * 64);
    const long long step = std::max(1ll, kGridItems / wg.x / ng) * cp;
    for (long long p = 0; p < n_img; p += step) {
        const int n = (int)std::min(step, n_img - p);
        const size_t row = (size_t)p * n_shift;
        const MrefJob j = mref_job(spec + row * n_ring * kSlots, norm + row, rspec, rsum0, rec + (size_t)p * n_ref, n,
                                   n_shift, n_ring, n_ref);
        const dim3 grid((unsigned)((n + cp - 1) / cp * ng));
        if (n_ring >= kMrefKeep) hipLaunchKernelGGL(k_ccf_mref<kMrefKeep>, grid, wg, 0, st, j, cp, twiddle);
        else hipLaunchKernelGGL(k_ccf_mref<0>, grid, wg, 0, st, j, cp, twiddle);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

MrefJob mref_job(const float2 *spec, const float2 *norm, const float2 *rspec, const float *rsum0,
                 PeakRec *rec, int n_img, int n_shift, int n_ring, int n_ref) {
    MrefJob j;
    j.spec = spec;
    j.norm = norm;
    j.rspec = rspec;
    j.rsum0 = rsum0;
    j.rec = rec;
    j.n_img = n_img;
    j.S = n_shift;
    j.R = n_ring;
    j.N = n_ref;
    return j;
}

int mref_queue_blocks_per_cu() {
    int n = 0;
    const hipError_t e =
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_ccf_mref_queue<kMrefKeep>, kMrefWaves * 64, 0);
    return e == hipSuccess ? n : 0;
}

hipError_t launch_ccf_mref_queue(const MrefJob *jobs, const int4 *items, const int *qbeg,
                                 int *counters, int blocks, int min_ring, const float2 *twiddle,
                                 hipStream_t st) {
    hipLaunchKernelGGL(k_reset_counters, dim3(1), dim3(64), 0, st, counters, 8);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid(blocks), wg(kMrefWaves * 64);
    if (min_ring >= kMrefKeep)
        hipLaunchKernelGGL(k_ccf_mref_queue<kMrefKeep>, grid, wg, 0, st, jobs, items, qbeg, counters, twiddle);
    else
        hipLaunchKernelGGL(k_ccf_mref_queue<0>, grid, wg, 0, st, jobs, items, qbeg, counters, twiddle);
    return hipGetLastError();
}

hipError_t launch_ccf_single(const float2 *spec, const float2 *norm, const float2 *rspec,
                             const float *rsum0, const int *ref_of, int ref_stride, int n_img,
                             int n_shift, int n_ring, int n_ref, const float2 *twiddle,
                             PeakRec *rec, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ccf_single, dim3((n_img + 3) / 4), dim3(256), 0, st, spec, norm, rspec, rsum0,
                       ref_of, ref_stride, n_img, n_shift, n_ring, n_ref, twiddle, rec);
    return hipGetLastError();
}

hipError_t launch_polar_single(const float *imgs, int n_img, int img_dim, ShiftView acc, const int2 *shift_i,
                               int n_shift, const float2 *tmpl, int n_ring, const float2 *twiddle,
                               const float2 *rspec, const float *rsum0, const int *ref_of, int ref_stride, int n_ref,
                               PeakRec *rec, hipStream_t st) {
    if (n_img <= 0 || n_shift <= 0) return hipSuccess;
    if (hipError_t e = prepare_launches()) return e;
    const int nw = polar_waves(n_shift, img_dim);
    const size_t lds = polar_lds_floats(img_dim, nw) * sizeof(float);
    const long long step = kGridItems / (64 * nw);
    for (long long p = 0; p < n_img; p += step) {
        const ShiftView a{acc.base + (size_t)p * acc.stride, acc.stride};
        const dim3 grid((unsigned)std::min(step, n_img - p));
        hipLaunchKernelGGL(k_polar_single, grid, dim3(64 * nw), lds, st, imgs + (size_t)p * img_dim * img_dim, img_dim,
                           a, shift_i, n_shift, tmpl, n_ring, twiddle, rspec, rsum0, ref_of + (size_t)p * ref_stride,
                           ref_stride, n_ref, rec + p);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

// One pass does a group of four shifts in one wavefront; two passes spread the rings of few
// groups over wavefronts.  Pre-alignment of 76 x 76 images, 34 rings, three iterations, one
// pass / two (us): 49 shifts, 5 images 512 / 585, 155 images 662 / 1145, 5000 images 12700 /
// 18900; 9 shifts, 30 images 340 / 292, 150 images 455 / 457, 600 images 776 / 898; 1 shift,
// 600 images 759 / 634.  Two iterations of 25 shifts: 600 images of 76 x 76 1494 / 1985, 3000
// of 128 x 128 8729 / 8952.  Where a CU holds one workgroup of the few wavefronts of 4 to 12
// shifts, the spread form is the better one for all but few images: 128 x 128, 9 shifts, 500
// images 2064 / 2310, 600 2581 / 2557, 800 3160 / 2250, 2000 5764 / 3855; with two a CU they
// are within 7 % (118 x 118, 1500 images 2843 / 2853).
bool polar_single_fills(int n_img, int n_shift, int img_dim) {
    const long long groups = (long long)n_img * ((n_shift + 3) / 4);
    const bool two = 2 * (polar_lds_floats(img_dim, polar_waves(n_shift, img_dim)) * sizeof(float) + 4096) <= 160 * 1024;
    return n_shift > 12 || (n_shift >= 4 && groups >= 1024 && (two || groups < 2048));
}

hipError_t launch_ccf_candidates(const float2 *spec, const float2 *norm, const float2 *rspec,
                                 const float *rsum0, const int *cand, int K, int n_img,
                                 int n_shift, int n_ring, int n_ref, const float2 *twiddle,
                                 PeakRec *rec, hipStream_t st, const int *pidx) {
    if (n_img <= 0 || K <= 0) return hipSuccess;
    if (K > kMrefRefs) return hipErrorInvalidValue;
    MrefJob j = mref_job(spec, norm, rspec, rsum0, rec, n_img, n_shift, n_ring, n_ref);
    j.cand = cand;
    j.pidx = pidx;
    j.K = K;
    const dim3 grid((unsigned)n_img), wg(kMrefWaves * 64);
    if (n_ring >= kMrefKeep) hipLaunchKernelGGL(k_ccf_cand<kMrefKeep>, grid, wg, 0, st, j, twiddle);
    else hipLaunchKernelGGL(k_ccf_cand<0>, grid, wg, 0, st, j, twiddle);
    return hipGetLastError();
}

hipError_t launch_topk(const PeakRec *rec, int n_img, int n_ref, int K, int *cand, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    if (K != 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_topk<8>, dim3((n_img + 127) / 128), dim3(128), 0, st, rec, n_img, n_ref, cand);
    return hipGetLastError();
}

hipError_t launch_best_candidate(const PeakRec *rec, const int *cand, int n_img, int K,
                                 float tie_rel, int *best, int *second, int *tie, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_best_candidate, dim3((n_img + 127) / 128), dim3(128), 0, st, rec, cand,
                       n_img, K, tie_rel, best, second, tie);
    return hipGetLastError();
}

hipError_t launch_rescore_f64(const float2 *spec, const float2 *norm, const float2 *rspec,
                              const PeakRec *rec, const int *cand, int *best, int *second,
                              const int *tie, int n_img, int K, int n_shift, int n_ring,
                              int n_ref, double *val64, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    const int waves = 2 * n_img;
    hipLaunchKernelGGL(k_rescore_f64, dim3((waves + 3) / 4), dim3(256), 0, st, spec, norm, rspec,
                       rec, cand, best, second, tie, n_img, K, n_shift, n_ring, n_ref, val64);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_resolve_ties, dim3((n_img + 127) / 128), dim3(128), 0, st, cand, val64,
                       tie, n_img, K, best, second);
    return hipGetLastError();
}

hipError_t launch_decode_best(const PeakRec *rec, const int *cand, const int *best,
                              const int *tie, int n_img, int K, ShiftView acc,
                              const float2 *shifts_f, int n_shift, int p_off, int *best_ref,
                              float *best_val, float *best_peak, int *tie_out, hipStream_t st,
                              const int *idx) {
    if (n_img <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_decode_best, dim3((n_img + 127) / 128), dim3(128), 0, st, rec, cand, best,
                       tie, n_img, K, acc, shifts_f, n_shift, p_off, best_ref, best_val, best_peak,
                       tie_out, idx);
    return hipGetLastError();
}

hipError_t launch_decode_mref(const PeakRec *rec, int n_img, int n_ref, ShiftView acc,
                              const float2 *shifts_f, int n_shift, float *peak, int peak_row,
                              int p_off, float *d, int d_pitch, hipStream_t st) {
    const long long n = (long long)n_img * n_ref;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_decode_mref, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rec,
                       n_img, n_ref, acc, shifts_f, n_shift, peak, peak_row, p_off, d, d_pitch);
    return hipGetLastError();
}

hipError_t launch_decode_single(const PeakRec *rec, int cnt, DevParam *prm,
                                const float2 *shifts_f, int n_shift, float shift_limit,
                                hipStream_t st) {
    if (cnt <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_decode_single, dim3((cnt + 255) / 256), dim3(256), 0, st, rec, cnt, prm,
                       shifts_f, n_shift, shift_limit);
    return hipGetLastError();
}

size_t pre_average_scratch_floats(int P, int D) {
    return (size_t)((P + kPreChunk - 1) / kPreChunk) * D * D;
}

hipError_t launch_pre_average(const float *imgs, int P, int D, const DevParam *prm, float4 *tp,
                              int *mir, float *part, float *avg, hipStream_t st) {
    if (P <= 0) return hipSuccess;
    const int nc = (P + kPreChunk - 1) / kPreChunk;
    hipLaunchKernelGGL(k_pre_tp, dim3((P + 255) / 256), dim3(256), 0, st, prm, P, tp, mir);
    hipLaunchKernelGGL(k_pre_partial, average_grid(D, nc), dim3(256), 0, st, imgs, D, P,
                       tp, mir, part);
    hipLaunchKernelGGL(k_pre_finish, dim3((D * D + 255) / 256), dim3(256), 0, st, part, D, P, nc,
                       avg);
    return hipGetLastError();
}

hipError_t launch_pre_center(const DevParam *prm, int P, float2 *shift, hipStream_t st) {
    hipLaunchKernelGGL(k_pre_center, dim3(1), dim3(256), 0, st, prm, P, shift);
    return hipGetLastError();
}

hipError_t launch_class_average(const float *imgs, int P, int img_dim, const DevParam *prm, const int *cid_idx,
                                int n_cls, float4 *tp, int *mir, float *refs, hipStream_t st) {
    if (P <= 0 || n_cls <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pre_tp, dim3((P + 255) / 256), dim3(256), 0, st, prm, P, tp, mir);
    hipLaunchKernelGGL(k_class_average, average_grid(img_dim, n_cls), dim3(256), 0, st, imgs,
                       img_dim, cid_idx, tp, mir, refs);
    return hipGetLastError();
}

static hipError_t filter_passes(float *refs, int n, int D, float cutoff, float falloff,
                                const float2 *shift, int abs_freq, float gain, float2 *work,
                                const float2 *tw_d, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const int Dh = D / 2 + 1;
    hipLaunchKernelGGL(k_row_dft, dim3(D, n), dim3(128), 0, st, refs, D, work, tw_d);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_col_filter, dim3(Dh, n), dim3(128), D * sizeof(float2), st, work, D,
                       tw_d, cutoff, falloff, shift, abs_freq);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_row_c2r, dim3(D, n), dim3(128), 0, st, refs, D, work, tw_d, gain);
    return hipGetLastError();
}

hipError_t launch_tanl_filter(float *refs, int n, int img_dim, float cutoff, float falloff,
                              float2 *work, const float2 *tw_d, hipStream_t st) {
    return filter_passes(refs, n, img_dim, cutoff, falloff, nullptr, 0, -1.0f, work, tw_d, st);
}

hipError_t launch_filter_shift(float *refs, int n, int img_dim, float cutoff, float falloff,
                               const float2 *shift, float2 *work, const float2 *tw_d,
                               hipStream_t st) {
    const float dd = (float)img_dim * (float)img_dim;
    return filter_passes(refs, n, img_dim, cutoff, falloff, shift, 1, 1.0f / dd, work, tw_d, st);
}

hipError_t launch_update_references(const float *imgs, int P, int D, const float *peak,
                                   const int *cls, int N, float cutoff, float falloff,
                                   UpdateScratch w, float *refs, float4 *params, hipStream_t st) {
    if (P <= 0 || N <= 0) return hipSuccess;
    const int gp = (P + 255) / 256;
    hipLaunchKernelGGL(k_upd_params, dim3(gp), dim3(256), 0, st, peak, P, N, cls, w.tp, w.mir,
                       w.post, w.raw, w.bad);
    hipLaunchKernelGGL(k_class_members<0>, dim3(N), dim3(1024), 0, st, cls, P, w.cnt, w.off,
                       w.members);
    hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(64), 0, st, w.cnt, N, w.off);
    hipLaunchKernelGGL(k_class_members<1>, dim3(N), dim3(1024), 0, st, cls, P, w.cnt, w.off,
                       w.members);
    hipLaunchKernelGGL(k_class_shift, dim3(N), dim3(64), 0, st, w.off, w.members, N,
                       w.post, w.mir, w.avg, w.neg, w.avg_out, w.members_out);
    hipLaunchKernelGGL(k_upd_params_out, dim3(gp), dim3(256), 0, st, cls, P, N, w.raw, w.post,
                       w.mir, w.avg, params);
    hipLaunchKernelGGL(k_class_transform_average, average_grid(D, N), dim3(256), 0, st,
                       imgs, D, w.off, w.members, w.tp, w.mir, refs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_filter_shift(refs, N, D, cutoff, falloff, w.neg, w.work, w.tw, st);
}

hipError_t launch_prop_items(const int *prop, int n_img, int K, int N, int nx, int ny, int hw,
                             int n_bins, float psi_half, PropItem *items,
                             unsigned long long *smask, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    if (K < 1 || K > kMaxProposals || nx * ny > 64 || hw < 0 || hw > 2) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_prop_items, dim3((n_img + 127) / 128), dim3(128), 0, st,
                       reinterpret_cast<const int4 *>(prop), n_img, K, N, nx, ny, hw, n_bins, psi_half,
                       items, smask);
    return hipGetLastError();
}

hipError_t launch_ccf_prop(const float2 *spec, const float2 *norm, const float2 *rspec,
                           const float *rsum0, const PropItem *items, int K, int n_img, int n_shift,
                           int n_ring, int n_ref, int nx, int ny, int hw, const float2 *twiddle,
                           PeakRec *rec, hipStream_t st) {
    const int n_items = n_img * K;
    if (n_items <= 0) return hipSuccess;
    if (K < 1 || K > kMaxProposals) return hipErrorInvalidValue;
    if (hipError_t e = prepare_launches()) return e;
    hipLaunchKernelGGL(hw > 0 ? k_ccf_prop<3> : k_ccf_prop<1>, dim3(n_img), dim3(64 * K), K * kPropLds, st, spec, norm,
                       rspec, rsum0, items, K, n_items, n_shift, n_ring, n_ref, nx, ny, hw, twiddle, rec);
    return hipGetLastError();
}

hipError_t launch_best_prop(const PeakRec *rec, const PropItem *items, int n_img, int K, int nx,
                            int ny, int hw, int edge_test, ShiftView acc, const float2 *shifts_f,
                            int n_shift, int p_off, int *best_ref, float *best_val,
                            float *best_peak, int *edge, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    if (nx * ny != n_shift || ny < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_best_prop, dim3((n_img + 127) / 128), dim3(128), 0, st, rec, items, n_img, K,
                       nx, ny, hw, edge_test, acc, shifts_f, n_shift, p_off, best_ref, best_val,
                       best_peak, edge);
    return hipGetLastError();
}

hipError_t launch_prop_refs(const int *prop, const int *idx, int n, int K, int N, int *cand,
                            hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (K < 1 || K > kMaxProposals) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_prop_refs, dim3((n + 127) / 128), dim3(128), 0, st,
                       reinterpret_cast<const int4 *>(prop), idx, n, K, N, cand);
    return hipGetLastError();
}

hipError_t launch_level2_mask(const int *flag, int n, int S, const unsigned long long *done,
                              unsigned long long *smask, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (S > 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_level2_mask, dim3((n + 255) / 256), dim3(256), 0, st, flag, n, S, done, smask);
    return hipGetLastError();
}

hipError_t launch_best_refs_level2(const PeakRec *rec, const int *cand, int n, int K, ShiftView acc,
                                   const float2 *shifts_f, int n_shift, const int *idx, int p_off,
                                   float threshold, int *best_ref, float *best_val,
                                   float *best_peak, int *fallback, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_best_refs_level2, dim3((n + 127) / 128), dim3(128), 0, st, rec, cand, n, K,
                       acc, shifts_f, n_shift, idx, p_off, threshold, best_ref, best_val, best_peak,
                       fallback);
    return hipGetLastError();
}

hipError_t launch_fallback_flags(const float *best_val, const int *edge, const float *conf,
                                 float conf_min, int n_img, float threshold, int p_off,
                                 int *fallback, hipStream_t st) {
    if (n_img <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fallback_flags, dim3((n_img + 255) / 256), dim3(256), 0, st, best_val, edge,
                       conf, conf_min, n_img, threshold, p_off, fallback);
    return hipGetLastError();
}

hipError_t launch_compact(const int *flag, int n, int lo, int hi, int *idx, int *count,
                          hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reset_counters, dim3(1), dim3(64), 0, st, count, 1);
    hipLaunchKernelGGL(k_compact, dim3((n + 255) / 256), dim3(256), 0, st, flag, n, lo, hi, idx, count);
    return hipGetLastError();
}

hipError_t launch_gather(const float *imgs, int D, ShiftView acc, const int *idx, int n, float *out,
                         float2 *out_acc, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather, dim3(n), dim3(256), 0, st, imgs, D, acc, idx, n, out, out_acc);
    return hipGetLastError();
}

hipError_t launch_best_refs_scatter(const PeakRec *rec, int n, int N, const float2 *acc,
                                    const float2 *shifts_f, int n_shift, const int *idx,
                                    int *best_ref, float *best_val, float *best_peak,
                                    hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_best_refs_scatter, dim3((n + 127) / 128), dim3(128), 0, st, rec, n, N, acc,
                       shifts_f, n_shift, idx, best_ref, best_val, best_peak);
    return hipGetLastError();
}

}  // namespace isac
