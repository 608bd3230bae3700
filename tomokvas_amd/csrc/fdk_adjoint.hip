// fdk_adjoint.hip -- adjoint of the backprojector: voxel-driven transposed-bilinear
// forward projection with atomic detector splats (gfx950).
//
// The backprojector (fdk_backproject.hip, reference FBPConeKernel/fQ3D,
// FBPG/kernel.cu:68-177) computes x = s * sum_beta U^2 * bilinear(Q_beta; u, v).
// Its transpose scatters every voxel value, weighted by s * U^2 and the same
// four bilinear weights, onto the detector samples that the voxel reads:
//   y(iv,   iu)   += s U^2 (1-fu)(1-fv) x      y(iv,   iu+1) += s U^2 fu (1-fv) x
//   y(iv+1, iu)   += s U^2 (1-fu) fv   x      y(iv+1, iu+1) += s U^2 fu fv     x
// with the same zero-outside-detector rule.
//
// FP32 (fp_lds_kernel): per angle, a workgroup's splats land in an LDS copy of
// its detector footprint box (as the one the backprojector stages,
// fdk_box.hpp) through integer LDS atomics, with the lanes of a wave along z;
// the box is then added to the detector with one coalesced global atomic per
// touched sample and cleared, which cuts global atomics from four per
// voxel-update to about a tenth.  Angles of ordinary footprints are summed in 32
// bits, those of wide ones in 64 by a second launch.  FP64 (fp_kernel) splats straight into HBM with
// hardware double atomics, one (x, y) column and a z-run per thread.
#include "fdk_internal.hpp"
#include "fdk_box.hpp"

#include <algorithm>
#include <type_traits>

namespace tkv {

template <typename R>
struct FPArgs {
    const R *vol;
    R *sino;                     // [Nv][nang][Nu]
    const R *ang, *ax, *ay, *az;
    int Nu, Nv, nang, Nx, Ny, Nz;
    R cX, cZ, D, umax, vmax, out_scale;
    double maskR2;
    int tiles_x, tiles_xy, tiles_z;
    // FP32, see FPLaunch:
    int splits;                  // angle splits of a tile, each a workgroup
    int wide;                    // the wide kernel takes the angles of wide footprints
    float fx_tile, fx_block, fx_count, umax_cyl;
};

template <typename R>
__device__ __forceinline__ R rfl(R x);
template <>
__device__ __forceinline__ float rfl(float x) { return floorf(x); }
template <>
__device__ __forceinline__ double rfl(double x) { return floor(x); }

template <typename R>
__device__ __forceinline__ R rfm(R a, R b, R c);
template <>
__device__ __forceinline__ float rfm(float a, float b, float c) { return fmaf(a, b, c); }
template <>
__device__ __forceinline__ double rfm(double a, double b, double c) { return fma(a, b, c); }

template <typename R>
__device__ __forceinline__ void splat(R *p, R v)
{
    unsafeAtomicAdd(p, v);
}

template <typename R, int ZR>
__global__ void __launch_bounds__(256) fp_kernel(FPArgs<R> a)
{
    const int lb = blockIdx.x;
    const int zr = lb / a.tiles_xy;
    const int tile = lb - zr * a.tiles_xy;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int x = tx * 16 + (wave & 1) * 8 + (lane & 7);
    const int y = ty * 16 + (wave >> 1) * 8 + (lane >> 3);
    const int z0 = zr * ZR;
    if (x >= a.Nx || y >= a.Ny) return;
    const R aX = a.ax[x], aY = a.ay[y];
    if (!((double)aX * (double)aX + (double)aY * (double)aY < a.maskR2)) return;

    R val[ZR], az[ZR];
    const size_t plane = (size_t)a.Nx * a.Ny;
    bool any = false;
#pragma unroll
    for (int k = 0; k < ZR; ++k) {
        int z = z0 + k;
        val[k] = z < a.Nz ? a.vol[(size_t)z * plane + (size_t)y * a.Nx + x] * a.out_scale : (R)0;
        az[k] = a.az[z0 + k];
        any = any || val[k] != (R)0;
    }
    if (!any) return;

    const size_t rstride = (size_t)a.nang * a.Nu;   // one detector row to the next
    for (int b = 0; b < a.nang; ++b) {
        const R c = a.ang[2 * b], s = a.ang[2 * b + 1];
        R S = rfm(aX, c, aY * s);
        R T = rfm(aY, c, -(aX * s));
        R U = a.D / (a.D - S);
        R u = rfm(T, U, a.cX);
        if (!(u >= (R)0 && u <= a.umax)) continue;
        R fl = rfl(u);
        const int iu = (int)fl;
        const R fu = u - fl;
        const R W = U * U;
        const R w1 = W * fu, w0 = W - W * fu;
        const bool has_u1 = iu + 1 < a.Nu;
        R *col = a.sino + (size_t)b * a.Nu + iu;
#pragma unroll
        for (int k = 0; k < ZR; ++k) {
            if (val[k] == (R)0) continue;
            R v = rfm(az[k], U, a.cZ);
            if (!(v >= (R)0 && v <= a.vmax)) continue;
            R fv0 = rfl(v);
            const int iv = (int)fv0;
            const R fv = v - fv0;
            const R x0 = val[k] * (1 - fv), x1 = val[k] * fv;
            R *r0 = col + (size_t)iv * rstride;
            splat(r0, w0 * x0);
            if (has_u1) splat(r0 + 1, w1 * x0);
            if (iv + 1 < a.Nv) {
                splat(r0 + rstride, w0 * x1);
                if (has_u1) splat(r0 + rstride + 1, w1 * x1);
            }
        }
    }
}

// Columns and slices whose footprints decide how an angle is summed: 32-bit sums
// where the footprint of every such block of a tile is below NARROW_W x NARROW_H
// samples, 64-bit sums elsewhere.
constexpr int FP_BLOCK = 16;
constexpr int FP_ZR = 64;                       // slices per workgroup: one per lane
constexpr int NARROW_W = 64, NARROW_H = 128;
constexpr int FP_WAVES = 16;
constexpr int FP_THREADS = 64 * FP_WAVES;
constexpr int FP_WORDS = 2 * 109 * 160;         // LDS of the boxes: 136 of a CU's 160 KiB

// Tile edge in columns, type of a sum, columns and rows of the LDS box.  The pitch
// is one more, odd: the rows of one column fall in distinct LDS banks.
template <bool WIDE>
struct FPTile {
    // 32 x 32 columns cover up to 32 sqrt 2 columns times pitch and magnification;
    // two boxes
    using Cell = int;
    static constexpr int T = 32, W = 108, H = 160;
};
template <>
struct FPTile<true> {
    // 16 x 16 columns of up to 2 samples at a magnification of 1.4, 64 slices of 2 at
    // up to 1.9; one box
    using Cell = unsigned long long;
    static constexpr int T = 16, W = 68, H = 252;
};
static_assert(2 * (FPTile<false>::W + 1) * FPTile<false>::H <= FP_WORDS &&
              2 * (FPTile<true>::W + 1) * FPTile<true>::H <= FP_WORDS, "boxes beyond the LDS");
// 32-bit sums whose blocks' footprints are narrow and whose tile's is beyond one box
// take the memory of both as one of 136 x 254
constexpr int FP_W2 = 136, FP_P2 = FP_W2 + 1, FP_H2 = FP_WORDS / FP_P2;
constexpr int BOX_LARGE = 0x40000;              // flag beside such a footprint's width
static_assert(FP_BLOCK * FP_ZR * (FPTile<false>::T + 1) <= FP_WORDS,
              "voxel transposition beyond the boxes");

// floor(x + 1/2), one instruction
__device__ __forceinline__ int round_half_up(float x)
{
    int r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// x (|x| < 2^51) rounded to the nearest integer: the low bits of x + 1.5 2^52
__device__ __forceinline__ unsigned long long round_i64(float x)
{
    const double d = (double)x + 0x1.8p52;
    return (unsigned long long)(unsigned)(__double2hiint(d) - 0x43380000) << 32 |
           (unsigned)__double2loint(d);
}

__device__ __forceinline__ float lane_f32(float x, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// first and last coordinate of each of the 2 x 2 blocks of 32 x 32 columns (blocks past
// the volume repeat the last column's)
struct BlockEdges {
    float x0[2], x1[2], y0[2], y1[2];
    __device__ __forceinline__ BlockEdges(const FPArgs<float> &a, int X0, int Y0)
    {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            x0[h] = a.ax[min(X0 + h * FP_BLOCK, a.Nx - 1)];
            x1[h] = a.ax[min(X0 + (h + 1) * FP_BLOCK, a.Nx) - 1];
            y0[h] = a.ay[min(Y0 + h * FP_BLOCK, a.Ny - 1)];
            y1[h] = a.ay[min(Y0 + (h + 1) * FP_BLOCK, a.Ny) - 1];
        }
    }
    // whether the footprints of all blocks are narrow
    __device__ inline bool narrow(const FPArgs<float> &a, float c, float s, float azlo,
                                  float azhi) const
    {
        bool all = true;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            all = footprint(c, s, x0[q & 1], x1[q & 1], y0[q >> 1], y1[q >> 1], azlo, azhi, a.cX,
                            a.cZ, a.D, a.Nu, a.Nv, NARROW_H, NARROW_W).z >= 0 && all;
        return all;
    }
};

// Lanes run along z: in each splat instruction the 64 lanes of a wave are the
// 64 slices of one (x, y) column, so their taps share the column and sit on
// distinct detector rows.  A wave owns NC of the tile's columns in both roles:
// lane l computes the angle's S, T, U, u and weights of column l once, and the
// splat loop takes column j's from lane j into scalar registers (v_readlane),
// with no LDS traffic and no barrier between the two.
//
// The box accumulates in fixed point with integer LDS atomics: float LDS atomics
// (ds_add_f32) measured 46x slower than ds_add_u32 (193 against 4.2 cycles per wave
// instruction and CU; ds_add_u64 6 to 8).
//
// 32-bit sums (WIDE false): the scale is the largest power of two that keeps every
// sample of the box below 2^31 (from the bound on the sum of a tile's bilinear
// weights), so the sums are exact.  A voxel's two column splats are rounded to the
// nearest unit (halves to even); the lower row takes its part, rounded, and the
// upper row the integer rest, so a column's sum over the rows is that of its
// rounded splats.  The flush converts back.  (Rounding by adding 3 * 2^22 needs two
// vector instructions less but limits a splat to 22 bits, and measured 3 % faster
// with larger errors on smooth volumes.)  A scale set by one large voxel must not
// coarsen the sums of the voxels around it: the unit of every 16 x 16 x 64 block is
// at most 2^-30 of the block's own bound (its largest voxel times the number of its
// voxels that reach one sample), and blocks whose largest voxels differ by more than
// that allows, about eightfold, are splatted in passes of their own.
//
// 64-bit sums (WIDE true), for footprints whose many rows per voxel leave 32 bits too
// few: the splats are the FP32 products of the direct splats below, rounded to
// 2^-K with K about 49 of a tile whose largest voxel is scaled to [1/2, 1): within
// 2^-26 of the voxel's weight down to 2^(25 - K) of the largest voxel, with exact sums.
//
// Voxels that fixed point can't hold -- infinities, NaN, and the largest (32 bits) or
// the relatively smallest (64 bits) -- are splatted straight into HBM in a pass of
// their own, and so are the angles whose footprint is beyond the box.
//
// What bounds it: a splat costs 22 vector instructions (about 1.1 issue cycles
// of the CU each; plain FP32 and integer adds and multiplies 0.75) beside 16
// cycles of LDS atomics.  The flush costs one global atomic per touched sample,
// 0.1 per voxel-update (0.25, and 0.86 of 3.8 ms, with tiles of 16 x 16
// columns; 384 x 384 x 320 voxels, 90 projections, 3.92 ms before and 3.16
// ms now).  The one workgroup of 16 waves fills a CU, so there are two boxes and
// one barrier per angle, and odd waves flush the last angle's box after this
// angle's splats, even waves before them: the flush's LDS and memory latency
// then overlaps other waves' splats.  An angle whose footprint needs the memory of
// both boxes, and every angle of 64-bit sums, has its splats and its flush one after
// the other.  332 x 326 x 164 voxels, 35 projections at two samples per voxel and
// magnifications up to 1.22: 1.3 ms with 64-bit sums, 66 straight into HBM; 14 ms where
// the volume falls off by 2^-80 within it, as voxels below 2^-24 of their block's
// largest go straight into HBM.  A second pass of a tile costs its angles' set-up and
// flush again: 384 x 384 x 320 voxels above, 3.2 ms with normal or smooth voxels, 3.75
// with one voxel in 33000 300 times as large, 3.95 where every tile takes four passes.
template <bool WIDE>
__global__ void __launch_bounds__(FP_THREADS) fp_lds_kernel(FPArgs<float> a)
{
    using Cell = typename FPTile<WIDE>::Cell;
    constexpr int T = FPTile<WIDE>::T, W = FPTile<WIDE>::W, H = FPTile<WIDE>::H, P = W + 1;
    constexpr int NC = T * T / FP_WAVES;             // columns of a wave
    constexpr int HALVES = T / FP_BLOCK, NB = HALVES * HALVES;   // blocks of a tile
    constexpr int XP = T + 1;                        // row pitch of the voxel transposition
    // block of column j (see the column role)
    constexpr auto block_of = [](int j) { return WIDE ? 0 : (j & 1) | (j >> 5) << 1; };
    extern __shared__ __align__(16) int fp_mem[];
    Cell *const box = (Cell *)fp_mem;     // H x P, twice for 32-bit sums
    int4 *boxes = (int4 *)(fp_mem + FP_WORDS);
    float2 *angs = (float2 *)(boxes + 64);
    float *wmax = (float *)(angs + 64);   // [FP_WAVES][NB]
    // Workgroups i, i + 8, ... of 8 * splits consecutive ones share a tile, so an
    // XCD's L2 (workgroups are dealt to the 8 XCDs in turn) serves the tile's
    // voxels to all its angle splits; tiles are skewed so that a compact
    // non-zero part of the volume spreads over the XCDs.
    const int per = 8 * a.splits;
    const int lb = blockIdx.x / per * 8 + (blockIdx.x & 7);
    const int sp = (blockIdx.x % per) >> 3;
    if (lb >= a.tiles_xy * a.tiles_z) return;
    const int zr = lb / a.tiles_xy;
    const int tile = lb - zr * a.tiles_xy;
    const int ty = tile / a.tiles_x;
    const int tx = (tile - ty * a.tiles_x + 3 * ty + 5 * zr) % a.tiles_x;
    const int b0 = (int)((long long)a.nang * sp / a.splits);
    const int b1 = (int)((long long)a.nang * (sp + 1) / a.splits);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int z0 = zr * FP_ZR;
    const int xa = tx * T, ya = ty * T;
    const float az0 = a.az[z0], az1 = a.az[z0 + FP_ZR - 1];
    const float azlo = fminf(az0, az1), azhi = fmaxf(az0, az1);
    const BlockEdges edges(a, xa & ~31, ya & ~31);
    if (a.wide) {
        // any angle of this kernel's kind?
        bool mine = false;
        for (int b = b0 + threadIdx.x; b < b1; b += FP_THREADS)
            mine = mine || edges.narrow(a, a.ang[2 * b], a.ang[2 * b + 1], azlo, azhi) != WIDE;
        if (!__syncthreads_or(mine)) return;
    }

    // column role: lane l of wave w owns column x = w + 16 (l & 1), y = l >> 1 of
    // the tile (every wave owns a part of each row: rim tiles stay balanced), or
    // x = w, y = l of a tile of 16 x 16
    const int x = xa + wave + (lane & (HALVES - 1)) * FP_BLOCK, y = ya + lane / HALVES;
    const bool valid = lane < NC && x < a.Nx && y < a.Ny;
    const float aX = valid ? a.ax[x] : 0.f, aY = valid ? a.ay[y] : 0.f;
    const bool inside =
        valid && ((double)aX * (double)aX + (double)aY * (double)aY < a.maskR2);
    const uint64_t columns = __ballot(inside);   // of this wave, bit = lane

    // slice role: lane = slice z0 + lane, val[j] its voxel of column j.  The tile
    // is read along x, 16 of its rows at a time with all of a thread's loads in
    // flight together, and turned through LDS.
    const float azl = a.az[z0 + lane];    // the z table is padded past Nz
    const bool in_z = z0 + lane < a.Nz;
    const size_t plane = (size_t)a.Nx * a.Ny;
    float val[NC];
    uint64_t live = 0;                    // columns with a voxel that is not zero
    float *turn = (float *)fp_mem;        // [16 y][64 z][XP]
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
        // row r = (y, z) of the half tile, STEP rows apart
        constexpr int STEP = FP_THREADS / T, ROWS = FP_BLOCK * FP_ZR / STEP;
        const int lx = threadIdx.x & (T - 1), r0 = threadIdx.x / T;
        const int gx = xa + lx;
        const float *src = a.vol + min(gx, a.Nx - 1);
        float q[ROWS];
        // unconditional loads (clamped into the volume; columns and slices
        // beyond it are masked below), so none waits for another
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int r = r0 + i * STEP;
            const int gy = ya + h * FP_BLOCK + r / FP_ZR, gz = z0 + r % FP_ZR;
            q[i] = src[(size_t)min(gz, a.Nz - 1) * plane + (size_t)min(gy, a.Ny - 1) * a.Nx];
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) turn[(r0 + i * STEP) * XP + lx] = q[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FP_BLOCK * HALVES; ++i) {
            const int j = FP_BLOCK * HALVES * h + i;
            const float t = turn[((i / HALVES) * FP_ZR + lane) * XP + wave + (i % HALVES) * FP_BLOCK];
            val[j] = ((columns >> j) & 1) && in_z ? t * a.out_scale : 0.f;
            if (__any(val[j] != 0.f)) live |= 1ull << j;
        }
        __syncthreads();
    }
    // the barriers below are workgroup-wide: skip only whole workgroups
    if (!__syncthreads_or(live != 0)) return;

    // the largest |voxel| of each block, of those that fixed point can hold
    constexpr float TOP = WIDE ? __builtin_inff() : 0x1p100f;
    bool odd = false;
    {
        float m[NB];
#pragma unroll
        for (int q = 0; q < NB; ++q) m[q] = 0.f;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const float g = fabsf(val[j]);
            const bool fits = g < TOP;
            odd = odd || !fits;
            m[block_of(j)] = fmaxf(m[block_of(j)], fits ? g : 0.f);
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) m[q] = fmaxf(m[q], __shfl_xor(m[q], o));
            if (lane == 0) wmax[wave * NB + q] = m[q];
        }
    }
    for (int i = threadIdx.x; i < FP_WORDS; i += FP_THREADS) fp_mem[i] = 0;
    __syncthreads();
    float qmax[NB];
    unsigned rest = 0;                    // blocks to be splatted
    {
        float t = wmax[lane & (FP_WAVES * NB - 1)];
#pragma unroll
        for (int o = NB; o < FP_WAVES * NB; o <<= 1) t = fmaxf(t, __shfl_xor(t, o));
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            qmax[q] = lane_f32(t, q);
            if (qmax[q] > 0.f) rest |= 1u << q;
        }
    }
    // U is at most D / (D - r) at radius r, r the tile's farthest column or the
    // cylinder's edge
    const float ex = fmaxf(fabsf(a.ax[xa]), fabsf(a.ax[min(xa + T, a.Nx) - 1]));
    const float ey = fmaxf(fabsf(a.ay[ya]), fabsf(a.ay[min(ya + T, a.Ny) - 1]));
    const float den = a.D - sqrtf(ex * ex + ey * ey);
    const float umax = fminf(den > 0.01f * a.D ? a.D / den : 100.f, a.umax_cyl);
    const float W2 = umax * umax;
    // exponent of the largest scale that keeps a sum of at most `bound` below 2^bits
    auto scale_of = [](float bound, float bits) { return (int)(bits - ceilf(log2f(bound) + 0.01f)); };
    // 64-bit sums: voxels as multiples of 2^val_exp, units of 2^(val_exp - K); smaller
    // voxels than `least` go straight to HBM (2^-26 of their weight is below half a unit)
    int val_exp = 0, K = 0;
    float least = 0.f;
    if constexpr (WIDE) {
        val_exp = __builtin_amdgcn_frexp_expf(qmax[0]);
        K = min(scale_of(W2, 50.f), scale_of(a.fx_block * W2, 62.f));
        least = ldexpf(1.f, val_exp + 25 - K);
#pragma unroll
        for (int j = 0; j < NC; ++j) odd = odd || (val[j] != 0.f && fabsf(val[j]) < least);
    }
    // beyond this magnification K would leave too few bits
    const bool steep = WIDE && umax > 4.f;
    auto straight = [&](float g) { return g != 0.f && !(fabsf(g) >= least && fabsf(g) < TOP); };
    // only voxels for fixed point are left
    auto settle = [&]() {
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            val[j] = straight(val[j]) ? 0.f : val[j];
            if constexpr (WIDE) val[j] = ldexpf(val[j], -val_exp);
        }
    };
    bool direct = __syncthreads_or(odd);  // a pass straight into HBM comes first
    if (WIDE && !direct) settle();

    const size_t rstride = (size_t)a.nang * a.Nu;   // one detector row to the next
    // constants of the splat loop in vector registers: an instruction reads one
    // scalar register, and that is the column's
    float czv = a.cZ;
    unsigned rowb = (unsigned)sizeof(Cell) * P;
    asm("" : "+v"(czv), "+v"(rowb));
    Cell *cur = box;                      // the box of this angle
    // the last angle splatted and not yet flushed (fb < 0: none): its box, first
    // column and row, columns (taps reach one past the last) and cells
    int fb = -1, fu0 = 0, fv0 = 0, fw = 1, fn = 0, fpitch = P;
    Cell *fbox = box;
    int unit = 0;                         // exponent of a unit of the sums
    // flush and clear: one global atomic per touched sample; the waves take
    // 64 consecutive cells of the box's used columns in turn, four at a time
    auto flush = [&]() {
        if (fb < 0) return;
        float *out = a.sino + (size_t)fb * a.Nu;
        const float winv = 1.f / (float)fw;
        const float funit = WIDE ? 0.f : ldexpf(1.f, unit);
        for (int q0 = wave * 64 + lane; q0 - lane < fn; q0 += 4 * FP_THREADS) {
            Cell t[4];
            int rr[4], cc[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int q = q0 + i * FP_THREADS;      // < 2^16: exact in float
                rr[i] = (int)(((float)q + 0.5f) * winv);
                cc[i] = q - rr[i] * fw;
                t[i] = q < fn ? fbox[rr[i] * fpitch + cc[i]] : 0;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (t[i] == 0) continue;
                fbox[rr[i] * fpitch + cc[i]] = 0;
                const int vr = fv0 + rr[i], uc = fu0 + cc[i];
                float sum;
                if constexpr (WIDE) sum = (float)ldexp((double)(long long)t[i], unit);
                else sum = (float)t[i] * funit;
                if (vr < a.Nv && uc < a.Nu) splat(out + (size_t)vr * rstride + uc, sum);
            }
        }
    };

    while (direct || rest) {
        // the blocks of this pass, and the scale of its sums
        unsigned group = (1u << NB) - 1;
        int fx = 0;
        if (WIDE) {
            fx = K;
            unit = val_exp - K;
        } else if (!direct) {
            // the block of the largest voxel, and those that the tile's scale serves
            int top = 0;
            float g = 0.f;
#pragma unroll
            for (int q = 0; q < NB; ++q)
                if ((rest >> q & 1) && qmax[q] > g) {
                    g = qmax[q];
                    top = q;
                }
            fx = min(scale_of(a.fx_tile * W2 * g, 31.f), 126);
            group = 0;
#pragma unroll
            for (int q = 0; q < NB; ++q)
                if ((rest >> q & 1) &&
                    min((int)(30.f - ceilf(log2f(a.fx_count * qmax[q]))), 126) <= fx)
                    group |= 1u << q;
            if (!(group >> top & 1) || !(group & (group - 1))) {
                group = 1u << top;
                fx = min(scale_of(a.fx_block * W2 * g, 31.f), 126);
            }
            unit = -fx;
        }
        const float fxs = ldexpf(1.f, fx);
        // the group's columns and corners
        uint64_t sel = ~0ull;
        int gx0 = xa, gx1 = xa + T, gy0 = ya, gy1 = ya + T;
        if constexpr (!WIDE) {
            const uint64_t even = 0x55555555ull;
            sel = (group & 1 ? even : 0) | (group & 2 ? even << 1 : 0) |
                  (group & 4 ? even << 32 : 0) | (group & 8 ? even << 33 : 0);
            if (!(group & 5)) gx0 += FP_BLOCK;
            if (!(group & 10)) gx1 -= FP_BLOCK;
            if (!(group & 3)) gy0 += FP_BLOCK;
            if (!(group & 12)) gy1 -= FP_BLOCK;
        }
        const float cx0 = a.ax[gx0], cx1 = a.ax[min(gx1, a.Nx) - 1];
        const float cy0 = a.ay[gy0], cy1 = a.ay[min(gy1, a.Ny) - 1];

        for (int b = b0; b < b1; ++b) {
            if (((b - b0) & 63) == 0) {
                __syncthreads();
                if (wave == 0 && b + lane < b1) {
                    const float c = a.ang[2 * (b + lane)], s = a.ang[2 * (b + lane) + 1];
                    int4 q = footprint(c, s, cx0, cx1, cy0, cy1, azlo, azhi, a.cX, a.cZ, a.D, a.Nu,
                                       a.Nv, H, W);
                    const bool narrow = !a.wide || edges.narrow(a, c, s, azlo, azhi);
                    if (narrow == WIDE) {
                        q.z = 0;          // the other kernel's
                    } else if (WIDE) {
                        if (q.z > 0 && (direct || steep)) q.z = -1;
                    } else if (direct) {
                        if (q.z != 0) q.z = -1;
                    } else if (q.z < 0) {
                        q = footprint(c, s, cx0, cx1, cy0, cy1, azlo, azhi, a.cX, a.cZ, a.D, a.Nu,
                                      a.Nv, FP_H2, FP_W2);
                        if (q.z > 0) q.z |= BOX_LARGE;
                    }
                    boxes[lane] = q;
                    angs[lane] = make_float2(c, s);
                }
                __syncthreads();
            }
            const int4 bx = boxes[(b - b0) & 63];
            const float2 cs = angs[(b - b0) & 63];
            const int bw = __builtin_amdgcn_readfirstlane(bx.z);
            if (bw == 0) continue;   // the block misses the detector at this angle
            const int bu0 = __builtin_amdgcn_readfirstlane(bx.x);
            const int bv0 = __builtin_amdgcn_readfirstlane(bx.y);
            const int bh = __builtin_amdgcn_readfirstlane(bx.w);

            // column role: the reference's S, T, U, u and the two column weights
            const float S = fmaf(aX, cs.x, aY * cs.y);
            const float Tc = fmaf(aY, cs.x, -(aX * cs.y));
            const float U = a.D / (a.D - S);
            const float u = fmaf(Tc, U, a.cX);
            const bool act = inside && u >= 0.f && u <= a.umax;
            const float fl = floorf(u);
            const int iu = (int)fl;
            const float fu = u - fl;
            const float Wc = U * U;
            const float w1 = Wc * fu, w0 = Wc - Wc * fu;
            const uint64_t todo = __ballot(act) & live & sel;
            const unsigned todo_lo = (unsigned)todo, todo_hi = (unsigned)(todo >> 32);

            if (bw > 0) {
                // splat into the LDS box; taps with zero weight past the
                // detector's last row or column land inside the box and are
                // dropped at the flush
                const bool inner = bw & BOX_INNER_V, large = !WIDE && (bw & BOX_LARGE);
                if (large) {
                    flush();
                    __syncthreads();          // both boxes are clear
                    cur = box;
                }
                char *lds = (char *)cur;
                // LDS byte offset of the column's sample in detector row 0; the
                // weights in units of the sums
                const int cb = (iu - bu0) * (int)sizeof(Cell) -
                               bv0 * (int)sizeof(Cell) * (large ? FP_P2 : P);
                const float ws0 = w0 * fxs, ws1 = w1 * fxs;
                auto splats = [&](auto inner_tag, auto pitch_tag) {
                    constexpr bool INNER = decltype(inner_tag)::value;
                    constexpr int PP = decltype(pitch_tag)::value;
#pragma unroll
                    for (int j = 0; j < NC; ++j) {
                        if (!((j < 32 ? todo_lo : todo_hi) & (1u << (j & 31)))) continue;   // scalar
                        const float v = fmaf(azl, lane_f32(U, j), czv);
                        const float ws0j = lane_f32(ws0, j), ws1j = lane_f32(ws1, j);
                        const int cbj = __builtin_amdgcn_readlane(cb, j);
                        if (INNER || (v >= 0.f && v <= a.vmax)) {
                            const float fv = __builtin_amdgcn_fractf(v);
                            Cell *p0 = (Cell *)(lds + (int)__umul24((unsigned)(int)v,
                                                                    PP == P ? rowb : sizeof(Cell) * PP) +
                                                cbj);
                            if constexpr (WIDE) {
                                const float x1 = val[j] * fv, x0 = val[j] - x1;
                                atomicAdd(p0, round_i64(ws0j * x0));
                                atomicAdd(p0 + 1, round_i64(ws1j * x0));
                                atomicAdd(p0 + PP, round_i64(ws0j * x1));
                                atomicAdd(p0 + PP + 1, round_i64(ws1j * x1));
                            } else {
                                const float s0 = val[j] * ws0j, s1 = val[j] * ws1j;
                                const int t0 = round_half_up(s0 * fv), t1 = round_half_up(s1 * fv);
                                atomicAdd(p0, __float2int_rn(s0) - t0);
                                atomicAdd(p0 + 1, __float2int_rn(s1) - t1);
                                atomicAdd(p0 + PP, t0);
                                atomicAdd(p0 + PP + 1, t1);
                            }
                        }
                    }
                };
                using pitch_t = std::integral_constant<int, P>;
                if (WIDE) {
                    if (inner) splats(std::true_type{}, pitch_t{});
                    else splats(std::false_type{}, pitch_t{});
                } else if (large) {
                    splats(std::false_type{}, std::integral_constant<int, FP_P2>{});
                } else {
                    if (!(wave & 1)) flush();
                    if (inner) splats(std::true_type{}, pitch_t{});
                    else splats(std::false_type{}, pitch_t{});
                    if (wave & 1) flush();
                }
                // the box splatted last is complete and the other one clear
                __syncthreads();
                fb = b;
                fbox = cur;
                fu0 = bu0;
                fv0 = bv0;
                fw = (bw & 0xffff) + 1;
                fn = fw * (bh + 1);
                if (WIDE || large) {
                    if (large) fpitch = FP_P2;
                    flush();
                    __syncthreads();          // all boxes are clear again
                    fpitch = P;
                    fb = -1;
                } else {
                    cur = cur == box ? box + H * P : box;
                }
            } else {
                // splat straight into HBM
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    if (!((todo >> j) & 1)) continue;
                    const float v = fmaf(azl, lane_f32(U, j), a.cZ);
                    const int iuj = __builtin_amdgcn_readlane(iu, j);
                    const float w0j = lane_f32(w0, j), w1j = lane_f32(w1, j);
                    float g = val[j];
                    if (g == 0.f || !(v >= 0.f && v <= a.vmax)) continue;
                    if (direct && !straight(g)) continue;
                    if constexpr (WIDE)
                        if (!direct) g = ldexpf(g, val_exp);
                    const float fv0 = floorf(v);
                    const int iv = (int)fv0;
                    const float fv = v - fv0;
                    const float x1 = g * fv, x0 = g - x1;
                    float *r0 = a.sino + (size_t)b * a.Nu + iuj + (size_t)iv * rstride;
                    const bool has_u1 = iuj + 1 < a.Nu;
                    splat(r0, w0j * x0);
                    if (has_u1) splat(r0 + 1, w1j * x0);
                    if (iv + 1 < a.Nv) {
                        splat(r0 + rstride, w0j * x1);
                        if (has_u1) splat(r0 + rstride + 1, w1j * x1);
                    }
                }
            }
        }
        flush();
        fb = -1;
        if (direct) {
            direct = false;
            settle();
        } else {
            rest &= ~group;
        }
    }
}

// Angle splits of every tile.  A workgroup fills a CU (of 256), and only tiles
// with a voxel that is not zero do any work (the gradient of a loss over a
// crop), so the angles are split until even 1/64 of the tiles gives the CUs two
// workgroups each, down to 24 angles.  Beyond that, the split that leaves the
// fewest angles in series when every tile works: rounds of 256 workgroups times
// the angles of one, reading the tile counted as two angles (24 us against 12 us
// measured for a full tile).  75 tiles x 40 angles of 1.5 samples per voxel: one
// split is 42 angles in series on 75 CUs, three are 16 on 225.
static int fp_splits(long long tiles, int nang)
{
    const long long least = std::max<long long>(
        1, std::min<long long>(nang / 24, (512 * 64 + tiles - 1) / tiles));
    long long best = least, cost = -1;
    for (long long s = least; s == least || (s <= nang / 2 && s <= 8 * least + 256); ++s) {
        const long long c = (tiles * s + 255) / 256 * ((nang + s - 1) / s + 2);
        if (cost < 0 || c < cost) {
            best = s;
            cost = c;
        }
    }
    return (int)best;
}

// Whether the footprint of a block with a column in the cylinder may be wide: bounds
// on its rows and columns at the cylinder's edge nearest to the source, with a sample
// to spare (U varies over a block, 15 sqrt 2 voxels across, by at most U^2/D per unit
// of S; a box has 7 rows and 10 columns beyond the span of the block's taps).
static bool may_be_wide(const FPLaunch &L)
{
    const double across = 21.3 * L.scale, r = std::sqrt(L.maskR2) + across;
    if (L.D <= r) return true;
    const double U = L.D / (L.D - r);
    const double rows = (FP_ZR - 1) * L.scale * U + L.az_max * across * U * U / L.D + 8.;
    const double cols = across * (U + r * U * U / L.D) + 11.;
    return rows >= NARROW_H || cols >= NARROW_W;
}

template <bool WIDE>
static int launch_fp_lds(FPArgs<float> a, hipStream_t st)
{
    constexpr int T = FPTile<WIDE>::T;
    a.tiles_x = (a.Nx + T - 1) / T;
    a.tiles_xy = a.tiles_x * ((a.Ny + T - 1) / T);
    a.tiles_z = (a.Nz + FP_ZR - 1) / FP_ZR;
    const long long tiles = (long long)a.tiles_xy * a.tiles_z;
    a.splits = fp_splits(tiles, a.nang);
    const long long nb = (tiles + 7) / 8 * 8 * a.splits;
    if (!grid_fits(nb, FP_THREADS))
        return fail(FDK_ERR_UNSUPPORTED, "forward_project: volume too large");
    const size_t lds = sizeof(int) * FP_WORDS + (sizeof(int4) + sizeof(float2)) * 64 +
                       sizeof(float) * FP_WAVES * 4;
    TKV_HIP(hipFuncSetAttribute((const void *)fp_lds_kernel<WIDE>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(fp_lds_kernel<WIDE>, dim3((unsigned)nb), dim3(FP_THREADS), lds, st, a);
    TKV_HIP(hipGetLastError());
    return FDK_OK;
}

template <typename R>
static int launch_fp_t(const FPLaunch &L, hipStream_t st)
{
    constexpr int ZR = 8;
    FPArgs<R> a;
    a.vol = (const R *)L.vol;
    a.sino = (R *)L.sino;
    a.ang = (const R *)L.ang;
    a.ax = (const R *)L.ax;
    a.ay = (const R *)L.ay;
    a.az = (const R *)L.az;
    a.Nu = L.Nu;
    a.Nv = L.Nv;
    a.nang = L.nang;
    a.Nx = L.Nx;
    a.Ny = L.Ny;
    a.Nz = L.Nz;
    a.cX = (R)L.cX;
    a.cZ = (R)L.cZ;
    a.D = (R)L.D;
    a.umax = (R)(L.Nu - 1);
    a.vmax = (R)(L.Nv - 1);
    a.out_scale = (R)L.out_scale;
    a.maskR2 = L.maskR2;
    if (L.Nx < 1 || L.Ny < 1 || L.Nz < 1 || L.nang == 0) return FDK_OK;
    if constexpr (sizeof(R) == 4) {
        a.fx_tile = (float)L.fx_tile;
        a.fx_block = (float)L.fx_block;
        a.fx_count = (float)L.fx_count;
        a.umax_cyl = (float)L.umax_cyl;
        a.wide = may_be_wide(L);
        int rc = launch_fp_lds<false>(a, st);
        if (!rc && a.wide) rc = launch_fp_lds<true>(a, st);
        return rc;
    } else {
        // 16 x 16 columns and 8 slices
        a.tiles_x = (L.Nx + 15) / 16;
        a.tiles_xy = a.tiles_x * ((L.Ny + 15) / 16);
        a.tiles_z = (L.Nz + ZR - 1) / ZR;
        const long long tiles = (long long)a.tiles_xy * a.tiles_z;
        if (!grid_fits(tiles, 256))
            return fail(FDK_ERR_UNSUPPORTED, "forward_project: volume too large");
        hipLaunchKernelGGL((fp_kernel<R, ZR>), dim3((unsigned)tiles), dim3(256), 0, st, a);
        TKV_HIP(hipGetLastError());
        return FDK_OK;
    }
}

int launch_forward_project(int real_bytes, const FPLaunch &a, hipStream_t st)
{
    return real_bytes == 8 ? launch_fp_t<double>(a, st) : launch_fp_t<float>(a, st);
}

}  // namespace tkv
