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
// voxel-update to about a tenth.  FP64 (fp_kernel) splats straight into HBM with
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
    int splits;                  // FP32: angle splits of a tile, each a workgroup
    float fx_bound;              // FP32: see FPLaunch::fx_bound
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

constexpr int FP_T = 32;                        // tile edge, columns
constexpr int FP_ZR = 64;                       // slices per workgroup: one per lane
constexpr int FP_WAVES = FP_T * FP_T / 64;      // a wave owns 64 columns
// LDS box: a tile of 32 x 32 columns x 64 slices covers up to 32 sqrt 2 columns
// and 64 rows of detector samples times pitch and magnification, so 108 x 160
// samples serve two samples per voxel; two boxes fill 136 of a CU's 160 KiB
constexpr int FP_W = 108;
constexpr int FP_H = 160;
constexpr int FP_P = FP_W + 1;                  // odd pitch: the rows of one column
                                                // fall in distinct LDS banks
// a footprint beyond that takes the memory of both boxes as one of 136 x 254
constexpr int FP_W2 = 136, FP_P2 = FP_W2 + 1, FP_H2 = 2 * FP_P * FP_H / FP_P2;
constexpr int BOX_LARGE = 0x40000;              // flag beside such a footprint's width
constexpr int FP_XP = FP_T + 1;                 // row pitch of the voxel transposition
static_assert(FP_T / 2 * FP_ZR * FP_XP <= 2 * FP_P * FP_H, "voxel transposition beyond the boxes");

// floor(x + 1/2), one instruction
__device__ __forceinline__ int round_half_up(float x)
{
    int r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

__device__ __forceinline__ float lane_f32(float x, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// Lanes run along z: in each splat instruction the 64 lanes of a wave are the
// 64 slices of one (x, y) column, so their taps share the column and sit on
// distinct detector rows.  A wave owns 64 of the tile's columns in both roles:
// lane l computes the angle's S, T, U, u and weights of column l once, and the
// splat loop takes column j's from lane j into scalar registers (v_readlane),
// with no LDS traffic and no barrier between the two.
//
// The box accumulates in 32-bit fixed point with integer LDS atomics: float
// LDS atomics (ds_add_f32) measured 46x slower than ds_add_u32 (193 against 4.2
// cycles per wave instruction and CU).  The workgroup's scale fxs is the largest
// power of two that keeps every sample of the box below 2^31 (from the bound on
// the sum of a tile's bilinear weights), so the sums are exact.  A voxel's
// two column splats are rounded to the nearest multiple of 1/fxs (halves to
// even); the lower row takes its part, rounded, and the upper row the integer
// rest, so a column's sum over the rows is that of its rounded splats.  The
// flush converts back.  (Rounding by adding 3 * 2^22 needs two vector
// instructions less but limits a splat to 22 bits, and measured 3 % faster with
// larger errors on smooth volumes.)
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
// both boxes has its splats and its flush one after the other; straight into HBM
// its splats cost 12 times as much (332 x 326 x 164 voxels, 35 projections at two
// samples per voxel and magnifications up to 1.22: 0.69 ms, 8.1 with those in HBM).
__global__ void __launch_bounds__(64 * FP_WAVES) fp_lds_kernel(FPArgs<float> a)
{
    extern __shared__ __align__(16) int fp_mem[];
    int *box = fp_mem;                    // 2 x FP_H x FP_P, units of 1/fxs
    int4 *boxes = (int4 *)(fp_mem + 2 * FP_H * FP_P);
    float2 *angs = (float2 *)(boxes + 64);
    unsigned *wmax = (unsigned *)(angs + 64);
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
    const int xa = tx * FP_T, ya = ty * FP_T;

    // column role: lane l of wave w owns column x = w + 16 (l & 1), y = l >> 1 of
    // the tile (every wave owns a part of each row: rim tiles stay balanced)
    const int x = xa + wave + (lane & 1) * (FP_T / 2), y = ya + (lane >> 1);
    const bool valid = x < a.Nx && y < a.Ny;
    const float aX = valid ? a.ax[x] : 0.f, aY = valid ? a.ay[y] : 0.f;
    const bool inside =
        valid && ((double)aX * (double)aX + (double)aY * (double)aY < a.maskR2);
    const uint64_t columns = __ballot(inside);   // of this wave, bit = lane

    // slice role: lane = slice z0 + lane, val[j] its voxel of column j.  The tile
    // is read along x, half of its rows at a time with all of a thread's loads in
    // flight together, and turned through LDS.
    const float azl = a.az[z0 + lane];    // the z table is padded past Nz
    const bool in_z = z0 + lane < a.Nz;
    const size_t plane = (size_t)a.Nx * a.Ny;
    float val[64];
    uint64_t live = 0;                    // columns with a voxel that is not zero
    float *turn = (float *)box;           // [16 y][64 z][FP_XP]
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // row r = (y, z) of the half tile, 32 rows apart: slice z alternates
        // between two per thread, y steps every second row
        constexpr int STEP = 64 * FP_WAVES / FP_T, ROWS = FP_T / 2 * FP_ZR / STEP;
        const int lx = threadIdx.x & (FP_T - 1), r0 = threadIdx.x / FP_T;
        const int gx = xa + lx;
        const float *src = a.vol + min(gx, a.Nx - 1);
        float q[ROWS];
        // unconditional loads (clamped into the volume; columns and slices
        // beyond it are masked below), so none waits for another
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int r = r0 + i * STEP;
            const int gy = ya + h * (FP_T / 2) + r / FP_ZR, gz = z0 + r % FP_ZR;
            q[i] = src[(size_t)min(gz, a.Nz - 1) * plane + (size_t)min(gy, a.Ny - 1) * a.Nx];
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) turn[(r0 + i * STEP) * FP_XP + lx] = q[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const int j = 32 * h + i;
            const float x = turn[((i >> 1) * FP_ZR + lane) * FP_XP + wave + (i & 1) * (FP_T / 2)];
            val[j] = ((columns >> j) & 1) && in_z ? x * a.out_scale : 0.f;
            if (__any(val[j] != 0.f)) live |= 1ull << j;
        }
        __syncthreads();
    }
    // the barriers below are workgroup-wide: skip only whole workgroups
    if (!__syncthreads_or(live != 0)) return;

    // the workgroup's largest |x| sets the fixed-point scale
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 64; ++j) m = fmaxf(m, fabsf(val[j]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) wmax[wave] = __float_as_uint(m);
    for (int i = threadIdx.x; i < 2 * FP_P * FP_H; i += 64 * FP_WAVES) box[i] = 0;
    __syncthreads();
    float gmax = 0.f;
#pragma unroll
    for (int w = 0; w < FP_WAVES; ++w) gmax = fmaxf(gmax, __uint_as_float(wmax[w]));
    const int xb = min(xa + FP_T - 1, a.Nx - 1), yb = min(ya + FP_T - 1, a.Ny - 1);
    const float cx0 = a.ax[xa], cx1 = a.ax[xb], cy0 = a.ay[ya], cy1 = a.ay[yb];
    // fixed-point scale: the largest power of two (exact in the weights and in
    // the flush) with fxs * bound * gmax below 2^31, room left for the splats'
    // rounding, one unit each; U is at most D / (D - r) at radius r, r the tile's
    // farthest column (capped so fxs stays finite)
    const float ux = fmaxf(fabsf(cx0), fabsf(cx1)), uy = fmaxf(fabsf(cy0), fabsf(cy1));
    const float den = a.D - sqrtf(ux * ux + uy * uy);
    const float umax = den > 0.01f * a.D ? a.D / den : 100.f;
    const float bound = a.fx_bound * (umax * umax) * gmax;
    const float fxs = exp2f(fminf(31.f - ceilf(log2f(bound) + 0.01f), 126.f));
    const float fxinv = 1.f / fxs;
    const float az0 = a.az[z0], az1 = a.az[z0 + FP_ZR - 1];
    const float azlo = fminf(az0, az1), azhi = fmaxf(az0, az1);
    const size_t rstride = (size_t)a.nang * a.Nu;   // one detector row to the next
    // constants of the splat loop in vector registers: an instruction reads one
    // scalar register, and that is the column's
    float czv = a.cZ;
    unsigned rowb = 4u * FP_P;
    asm("" : "+v"(czv), "+v"(rowb));
    int *cur = box;                       // the box of this angle
    // the last angle splatted and not yet flushed (fb < 0: none): its box, first
    // column and row, columns (taps reach one past the last) and cells
    int fb = -1, fu0 = 0, fv0 = 0, fw = 1, fn = 0, fpitch = FP_P;
    int *fbox = box;
    // flush and clear: one global atomic per touched sample; the waves take
    // 64 consecutive cells of the box's used columns in turn, four at a time
    auto flush = [&]() {
        if (fb < 0) return;
        float *out = a.sino + (size_t)fb * a.Nu;
        const float winv = 1.f / (float)fw;
        for (int q0 = wave * 64 + lane; q0 - lane < fn; q0 += 4 * 64 * FP_WAVES) {
            int t[4], rr[4], cc[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int q = q0 + i * 64 * FP_WAVES;   // < 2^16: exact in float
                rr[i] = (int)(((float)q + 0.5f) * winv);
                cc[i] = q - rr[i] * fw;
                t[i] = q < fn ? fbox[rr[i] * fpitch + cc[i]] : 0;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (t[i] == 0) continue;
                fbox[rr[i] * fpitch + cc[i]] = 0;
                const int vr = fv0 + rr[i], uc = fu0 + cc[i];
                if (vr < a.Nv && uc < a.Nu)
                    splat(out + (size_t)vr * rstride + uc, (float)t[i] * fxinv);
            }
        }
    };

    for (int b = b0; b < b1; ++b) {
        if (((b - b0) & 63) == 0) {
            __syncthreads();
            if (wave == 0 && b + lane < b1) {
                const float c = a.ang[2 * (b + lane)], s = a.ang[2 * (b + lane) + 1];
                int4 q = footprint(c, s, cx0, cx1, cy0, cy1, azlo, azhi, a.cX, a.cZ, a.D, a.Nu,
                                   a.Nv, FP_H, FP_W);
                if (q.z < 0) {
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
        const float T = fmaf(aY, cs.x, -(aX * cs.y));
        const float U = a.D / (a.D - S);
        const float u = fmaf(T, U, a.cX);
        const bool act = inside && u >= 0.f && u <= a.umax;
        const float fl = floorf(u);
        const int iu = (int)fl;
        const float fu = u - fl;
        const float W = U * U;
        const float w1 = W * fu, w0 = W - W * fu;
        const uint64_t todo = __ballot(act) & live;
        const unsigned todo_lo = (unsigned)todo, todo_hi = (unsigned)(todo >> 32);

        if (bw > 0) {
            // splat into the LDS box; taps with zero weight past the
            // detector's last row or column land inside the box and are
            // dropped at the flush
            const bool inner = bw & BOX_INNER_V, large = bw & BOX_LARGE;
            if (large) {
                flush();
                __syncthreads();          // both boxes are clear
                cur = box;
            }
            char *lds = (char *)cur;
            // LDS byte offset of the column's sample in detector row 0; the
            // weights in units of 1/fxs
            const int cb = (iu - bu0) * 4 - bv0 * 4 * (large ? FP_P2 : FP_P);
            const float ws0 = w0 * fxs, ws1 = w1 * fxs;
            auto splats = [&](auto inner_tag, auto pitch_tag) {
                constexpr bool INNER = decltype(inner_tag)::value;
                constexpr int P = decltype(pitch_tag)::value;
#pragma unroll
                for (int j = 0; j < 64; ++j) {
                    if (!((j < 32 ? todo_lo : todo_hi) & (1u << (j & 31)))) continue;   // scalar
                    const float v = fmaf(azl, lane_f32(U, j), czv);
                    const float s0 = val[j] * lane_f32(ws0, j), s1 = val[j] * lane_f32(ws1, j);
                    const int cbj = __builtin_amdgcn_readlane(cb, j);
                    if (INNER || (v >= 0.f && v <= a.vmax)) {
                        const float fv = __builtin_amdgcn_fractf(v);
                        int *p0 = (int *)(lds + (int)__umul24((unsigned)(int)v,
                                                              P == FP_P ? rowb : 4u * P) + cbj);
                        const int t0 = round_half_up(s0 * fv), t1 = round_half_up(s1 * fv);
                        atomicAdd(p0, __float2int_rn(s0) - t0);
                        atomicAdd(p0 + 1, __float2int_rn(s1) - t1);
                        atomicAdd(p0 + P, t0);
                        atomicAdd(p0 + P + 1, t1);
                    }
                }
            };
            using pitch_t = std::integral_constant<int, FP_P>;
            if (large) {
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
            if (large) {
                fpitch = FP_P2;
                flush();
                __syncthreads();          // both boxes are clear again
                fpitch = FP_P;
                fb = -1;
            } else {
                cur = cur == box ? box + FP_H * FP_P : box;
            }
        } else {
            // box beyond the LDS tile: splat straight into HBM
#pragma unroll
            for (int j = 0; j < 64; ++j) {
                if (!((todo >> j) & 1)) continue;
                const float v = fmaf(azl, lane_f32(U, j), a.cZ);
                const int iuj = __builtin_amdgcn_readlane(iu, j);
                const float w0j = lane_f32(w0, j), w1j = lane_f32(w1, j);
                const float g = val[j];
                if (g == 0.f || !(v >= 0.f && v <= a.vmax)) continue;
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
    a.fx_bound = (float)L.fx_bound;
    // 16 x 16 columns and 8 slices in FP64
    const int edge = sizeof(R) == 4 ? FP_T : 16, zrun = sizeof(R) == 4 ? FP_ZR : ZR;
    a.tiles_x = (L.Nx + edge - 1) / edge;
    a.tiles_xy = a.tiles_x * ((L.Ny + edge - 1) / edge);
    a.tiles_z = (L.Nz + zrun - 1) / zrun;
    a.splits = 1;
    const long long tiles = (long long)a.tiles_xy * a.tiles_z;
    if (tiles == 0 || L.nang == 0) return FDK_OK;
    if constexpr (sizeof(R) == 4) {
        a.splits = fp_splits(tiles, L.nang);
        const long long nb = (tiles + 7) / 8 * 8 * a.splits;
        if (!grid_fits(nb, 64 * FP_WAVES))
            return fail(FDK_ERR_UNSUPPORTED, "forward_project: volume too large");
        const size_t lds = sizeof(int) * 2 * FP_H * FP_P + (sizeof(int4) + sizeof(float2)) * 64 +
                           sizeof(unsigned) * FP_WAVES;
        TKV_HIP(hipFuncSetAttribute((const void *)fp_lds_kernel,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(fp_lds_kernel, dim3((unsigned)nb), dim3(64 * FP_WAVES), lds, st, a);
    } else {
        if (!grid_fits(tiles, 256))
            return fail(FDK_ERR_UNSUPPORTED, "forward_project: volume too large");
        hipLaunchKernelGGL((fp_kernel<R, ZR>), dim3((unsigned)tiles), dim3(256), 0, st, a);
    }
    TKV_HIP(hipGetLastError());
    return FDK_OK;
}

int launch_forward_project(int real_bytes, const FPLaunch &a, hipStream_t st)
{
    return real_bytes == 8 ? launch_fp_t<double>(a, st) : launch_fp_t<float>(a, st);
}

}  // namespace tkv
