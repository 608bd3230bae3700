// fdk_backproject.hip -- voxel-driven cone-beam backprojection for gfx950.
//
// Reference: FBPConeKernel + fQ3D (FBPG/kernel.cu:68-177): per voxel
//   a = scale*(idx - centre) (sign flips), inside iff |(aX,aY)| < Nu/2,
//   sum over beta of U^2 * bilinear(Q_beta; T*U + cX, aZ*U + cZ),
//   S = aX cos + aY sin, T = aY cos - aX sin, U = D/(D - S), times delta_f/p;
//   samples outside [0,Nu-1] x [0,Nv-1] contribute 0.
//
// MI355X design:
//  * a workgroup owns a block of 16x16 columns x ZR slices; a thread owns one
//    (x,y) column and its ZR slices in registers: S, T, U, u = T*U + cX and U^2
//    depend only on (x, y, beta) and are paid once per ZR updates.  Smaller
//    volumes take shorter runs, and G groups of threads that share a block's
//    angles (bp_shape);
//  * per angle, the block's detector footprint -- a box of samples that the
//    workgroup derives from its corner columns (u and U are linear-fractional
//    in (aX, aY), so their extremes over the block sit at the corners) -- is
//    staged from HBM into LDS with coalesced loads; every bilinear gather of
//    the angle then reads LDS, so L2/HBM carry about one stored sample per two
//    voxel-updates instead of four taps per update;
//  * the stored stack is plain and angle-major ([beta][v][pitch]) in the
//    storage type: FP32, FP16 with a per-projection scale, or BF16; FP16 and
//    BF16 halve the staging bytes.  The box in LDS holds FP32 samples, widened
//    exactly when they are staged, so for every storage type the interpolation
//    weights, lerps and accumulation are FP32 and a low-precision volume is the
//    FP32 arithmetic on the decoded samples.  (FP16 pairs in the box, widened by
//    mixed-precision FMAs, halve the LDS reads, but those FMAs issue at 1.1
//    cycles per wave instruction and CU where plain FP32 arithmetic on vector
//    registers takes 0.66: they are used for the highest boxes only.)
//    FDK_F16_PACKED (opt-in) keeps FP16 pairs (q[c], q[c+1]) per 32-bit word,
//    lerps in packed FP16 and weights with v_dot2 (FP16 fraction and column
//    weights): faster, outside the precision form;
//  * z-runs that project entirely inside the detector for every active lane of
//    a wave (the common case) skip the per-slice range test;
//  * workgroup ids are remapped so the workgroups an XCD runs together cover a
//    compact part of the volume and share detector rows in that XCD's L2;
//  * boxes larger than the LDS tile (extreme magnification, blocks near the
//    source) and the FP64 instantiation gather straight from HBM with the same
//    arithmetic.
#include "fdk_internal.hpp"
#include "fdk_box.hpp"

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <cmath>
#include <type_traits>

// Tuning knobs (defaults chosen by measurement on MI355X, 1024^3 from
// 1800 x 2048^2):
//   TKV_BP_ZR_F32 / _F16 / _BF16 / _F16P  slices per thread (register z-run)
//                                  per storage type (FP64 uses 8)
//   TKV_BP_BOXP_F32 / _F16P        LDS row pitch of the staged box in 32-bit
//                                  words (>= 64, multiple of 4): rows of one
//                                  column fall in different banks (FP32 samples;
//                                  FP16 pairs)
#ifndef TKV_BP_ZR_F32
#define TKV_BP_ZR_F32 24
#endif
#ifndef TKV_BP_ZR_F16
#define TKV_BP_ZR_F16 32
#endif
#ifndef TKV_BP_ZR_BF16
#define TKV_BP_ZR_BF16 32
#endif
#ifndef TKV_BP_ZR_F16P
#define TKV_BP_ZR_F16P 32
#endif
#ifndef TKV_BP_BOXP_F32
#define TKV_BP_BOXP_F32 80
#endif
#ifndef TKV_BP_BOXP_F16P
#define TKV_BP_BOXP_F16P 72
#endif

namespace tkv {

static_assert(box_rows<64>() <= STACK_TAIL_ROWS, "stored stack tail shorter than a box");

static_assert(STACK_PAD >= BOX_W + BOX_ALIGN, "stored rows padded by less than a box");

template <typename R>
struct BPArgs {
    const char *stack;
    size_t angle_bytes;           // bytes per projection of the stack
    uint32_t row_bytes;           // bytes per detector row of the stack
    const R *ang;                 // (cos, sin) per angle
    const R *scales;              // per angle dequantisation factor
    const R *ax, *ay, *az;
    R *vol;
    int Nx, Ny, Nz, Nu, Nv, nang;
    R cX, cZ, D, umax, vmax, out_scale;
    R one;                        // 1, at run time: see LdsGather
    double maskR2;
    int accumulate;
    int tiles_x, tiles_xy, nblocks;
    int box_h;                    // rows of the LDS box, a multiple of 16
};

// ---- storage types ----------------------------------------------------------------
// PAIRS: the LDS box holds FP16 sample pairs, interpolated in packed FP16 or, MIX,
// with FP32 fractions and weights in mixed-precision FMAs (else FP32 samples)
struct st_f32;
struct st_f16;
struct st_bf16;
struct st_f16p;
struct st_f16m;
struct st_f64;
template <typename S>
struct Store;
template <>
struct Store<st_f32> {
    using R = float;
    static constexpr int BYTES = 4;
    static constexpr bool STAGED = true;
    static constexpr int ZR = TKV_BP_ZR_F32;
    static constexpr int P = TKV_BP_BOXP_F32;
    static constexpr bool PAIRS = false;
    static constexpr bool MIX = false;
    static __device__ __forceinline__ float get(const char *p) { return *(const float *)p; }
    static __device__ __forceinline__ float half(unsigned, int) { return 0.f; }
};
template <>
struct Store<st_f16> {
    using R = float;
    static constexpr int BYTES = 2;
    static constexpr bool STAGED = true;
    static constexpr int ZR = TKV_BP_ZR_F16;
    static constexpr int P = TKV_BP_BOXP_F32;
    static constexpr bool PAIRS = false;
    static constexpr bool MIX = false;
    static __device__ __forceinline__ float get(const char *p)
    {
        return __half2float(__ushort_as_half(*(const unsigned short *)p));
    }
    static __device__ __forceinline__ float half(unsigned w, int hi)
    {
        return __half2float(__ushort_as_half((unsigned short)(hi ? w >> 16 : w & 0xffffu)));
    }
};
template <>
struct Store<st_bf16> {
    using R = float;
    static constexpr int BYTES = 2;
    static constexpr bool STAGED = true;
    static constexpr int ZR = TKV_BP_ZR_BF16;
    static constexpr int P = TKV_BP_BOXP_F32;
    static constexpr bool PAIRS = false;
    static constexpr bool MIX = false;
    static __device__ __forceinline__ float get(const char *p)
    {
        return __uint_as_float((unsigned)(*(const unsigned short *)p) << 16);
    }
    static __device__ __forceinline__ float half(unsigned w, int hi)
    {
        return __uint_as_float(hi ? (w & 0xffff0000u) : (w << 16));
    }
};
template <>
struct Store<st_f16m> : Store<st_f16> {
    static constexpr int P = TKV_BP_BOXP_F16P;
    static constexpr bool PAIRS = true;
    static constexpr bool MIX = true;
};
template <>
struct Store<st_f16p> : Store<st_f16> {
    static constexpr int ZR = TKV_BP_ZR_F16P;
    static constexpr int P = TKV_BP_BOXP_F16P;
    static constexpr bool PAIRS = true;
};
template <>
struct Store<st_f64> {
    using R = double;
    static constexpr int BYTES = 8;
    static constexpr bool STAGED = false;
    static constexpr int ZR = 8;
    static constexpr int P = 64;   // unused: FP64 is gathered from HBM
    static constexpr bool PAIRS = false;
    static constexpr bool MIX = false;
    static __device__ __forceinline__ double get(const char *p) { return *(const double *)p; }
    static __device__ __forceinline__ float half(unsigned, int) { return 0.f; }
};

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

template <typename R>
__device__ __forceinline__ R rfma(R a, R b, R c);
template <>
__device__ __forceinline__ float rfma(float a, float b, float c) { return fmaf(a, b, c); }
template <>
__device__ __forceinline__ double rfma(double a, double b, double c) { return fma(a, b, c); }
// x - floor(x) in one instruction (v_fract); exact for the finite x used here
template <typename R>
__device__ __forceinline__ R rfract(R x);
template <>
__device__ __forceinline__ float rfract(float x) { return __builtin_amdgcn_fractf(x); }
template <>
__device__ __forceinline__ double rfract(double x) { return __builtin_amdgcn_fract(x); }

// ---- LDS gather of one angle for one slice of a thread's z-run ------------------------
// acc[k] += W * bilinear(box; u, v_k) with v_k = az[k]*Uv + cz; col is where the
// thread's column would lie in detector row 0 (a pointer, so that a sample's
// address is one multiply-add from the row).
// FAST: every v_k of every lane of the wave lies inside [0.01, Nv-1.01].
// MIX: word (r, c) of the box holds the FP16 samples c and c+1 of row r.  Each
// column's difference along v and its lerp are mixed-precision FMAs that read the
// FP16 halves directly (v_fma_mix_f32; the product with `one`, 1 at run time, is
// exact and the result rounds once to FP32), so they equal the FP32 operations on
// the widened samples.
template <bool FAST, bool MIX, int P>
struct LdsGather {
    using Q = typename std::conditional<MIX, half2_t, float2>::type;
    float fv;
    Q q0, q1;   // rows iv and iv + 1
    bool ok;
    __device__ __forceinline__ void issue(float az, const float *box, float Uv, float cz,
                                          const char *col, float vmax)
    {
        const float v = fmaf(az, Uv, cz);
        fv = __builtin_amdgcn_fractf(v);
        // v >= 0 where used
        const float *p0 = (const float *)(col + (int)__umul24((unsigned)(int)v, 4u * P));
        ok = true;
        if (!FAST) {
            ok = v >= 0.f && v <= vmax;
            p0 = ok ? p0 : box;
        }
        if constexpr (MIX) {
            q0 = *(const half2_t *)p0;
            q1 = *(const half2_t *)(p0 + P);
        } else {
            q0 = make_float2(p0[0], p0[1]);
            q1 = make_float2(p0[P], p0[P + 1]);
        }
    }
    // taps outside the detector get zero weight (the staged values are finite)
    __device__ __forceinline__ float add(float acc, float wu0, float wu1, float one) const
    {
        float d0, d1;
        if constexpr (MIX) {
            d0 = fmaf((float)q1.x, one, -(float)q0.x);
            d1 = fmaf((float)q1.y, one, -(float)q0.y);
        } else {
            d0 = q1.x - q0.x;
            d1 = q1.y - q0.y;
        }
        const float c0 = fmaf(fv, d0, (float)q0.x), c1 = fmaf(fv, d1, (float)q0.y);
        return fmaf(ok ? wu1 : 0.f, c1, fmaf(ok ? wu0 : 0.f, c0, acc));
    }
};

// FP16 pairs in LDS, packed-FP16 interpolation (FDK_F16_PACKED): the lerp
// along v runs in packed FP16; the two column weights (FP16, normalised to at
// most U^2) and the two lerped columns meet in one v_dot2_f32_f16, summed in
// FP32.
template <bool FAST, int P>
struct PairGather {
    half2_t f, w0[2], w1[2];   // the two slices' fractions, their rows iv and iv + 1
    bool ok[2];
    __device__ __forceinline__ void issue(const float *az, const float *box, float Uv, float cz,
                                          const char *col, float vmax)
    {
        const float v[2] = {fmaf(az[0], Uv, cz), fmaf(az[1], Uv, cz)};
        // one conversion serves two slices; each lerp broadcasts its half
        f = __builtin_bit_cast(half2_t,
                               __builtin_amdgcn_cvt_pkrtz(__builtin_amdgcn_fractf(v[0]),
                                                          __builtin_amdgcn_fractf(v[1])));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            // v >= 0 where used
            const float *p0 = (const float *)(col + (int)__umul24((unsigned)(int)v[j], 4u * P));
            ok[j] = true;
            if (!FAST) {
                ok[j] = v[j] >= 0.f && v[j] <= vmax;
                p0 = ok[j] ? p0 : box;
            }
            w0[j] = *(const half2_t *)p0;
            w1[j] = *(const half2_t *)(p0 + P);
        }
    }
    // the three-address VOP3P form (the builtin selects the two-address
    // v_dot2c form, whose tied accumulator costs register copies here)
    __device__ __forceinline__ void add(float *acc, half2_t wuh) const
    {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const half2_t fj = j ? half2_t{f.y, f.y} : half2_t{f.x, f.x};
            const half2_t c = fj * (w1[j] - w0[j]) + w0[j];
            const half2_t w = ok[j] ? wuh : half2_t{0, 0};
            float r;
            asm("v_dot2_f32_f16 %0, %1, %2, %3" : "=v"(r) : "v"(c), "v"(w), "v"(acc[j]));
            acc[j] = r;
        }
    }
};

// all ZR slices of a thread for one staged angle
template <bool FAST, typename ST, int ZR, int P>
__device__ __forceinline__ void gather_run(float (&acc)[ZR], const float (&az)[ZR],
                                           const float *box, float Uv, float cz,
                                           const char *col, float wu0, float wu1, half2_t wuh,
                                           float vmax, float one)
{
    if constexpr (ST::PAIRS && !ST::MIX) {
        PairGather<FAST, P> g[2];
        g[0].issue(az, box, Uv, cz, col, vmax);
#pragma unroll
        for (int k = 0; k < ZR; k += 2) {
            __builtin_amdgcn_sched_barrier(0);
            if (k + 2 < ZR) g[(k / 2 + 1) & 1].issue(az + k + 2, box, Uv, cz, col, vmax);
            __builtin_amdgcn_sched_barrier(0);
            g[k / 2 & 1].add(acc + k, wuh);
        }
        __builtin_amdgcn_sched_barrier(0);
    } else {
        // one slice's samples are on their way while the slice before is added: left
        // to itself the compiler waits for each slice's or holds those of several,
        // which takes registers (256^3 from 360, FP32: 1.83 ms, 1.97 with a wait per
        // slice, 1.87 with two slices together, 1.89 with two on their way)
        LdsGather<FAST, ST::MIX, P> g[2];
        g[0].issue(az[0], box, Uv, cz, col, vmax);
#pragma unroll
        for (int k = 0; k < ZR; ++k) {
            __builtin_amdgcn_sched_barrier(0);
            if (k + 1 < ZR) g[(k + 1) & 1].issue(az[k + 1], box, Uv, cz, col, vmax);
            __builtin_amdgcn_sched_barrier(0);
            acc[k] = g[k & 1].add(acc[k], wu0, wu1, one);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Box staging in two steps, so the loads of the next angle's box fly while
// the current angle is gathered: issue() loads rows [bv0, bv0+bh] of a
// projection (the last is the +1 neighbour row; rows past the detector are
// zero) x columns [bu0, bu0+64) or the box's into registers, 4 samples per lane and row,
// 16 lanes per row (columns past the row end read the stack's zero padding);
// commit() writes them into the LDS box, widened to FP32; FP16 pair boxes hold
// words (q[c], q[c+1]), the 4th word of a lane taking the next lane's first
// sample (word 63 is never read).
template <typename S, int ROWS, bool TRIM>
struct BoxStage {
    using ST = Store<S>;
    static constexpr int PER = (ROWS + 15) / 16;   // rows per thread
    using Raw = typename std::conditional<ST::BYTES == 4, float4, uint2>::type;
    Raw raw[PER];

    __device__ __forceinline__ void issue(const char *proj, int bu0, int bv0, int bh, int w4,
                                          uint32_t row_bytes, int Nv, int tid)
    {
        // buffer loads: a scalar descriptor at the box origin whose range ends
        // with the last row inside the detector, so rows past it read as zero
        // (raw buffer range check), and one 32-bit offset per row
        // (a projection is below 2 GiB, checked at launch: 32-bit offsets)
        const char *base = proj + ((uint32_t)bv0 * row_bytes + (uint32_t)bu0 * ST::BYTES);
        const int rows = min(bh, Nv - 1 - bv0);   // last row inside the detector
        const int nrec = (rows + 1) * (int)row_bytes - bu0 * ST::BYTES;
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, nrec, 0x00020000);
        int off = (int)((uint32_t)(tid >> 4) * row_bytes + (tid & 15) * 4 * ST::BYTES);
        // lanes past the box's last column (w4: its columns over 4) read zeros outside
        // the descriptor's range, a quarter of the bytes: 640^2 x 321 FP32 from 120
        // x 1280 x 900 5.13 -> 5.00 ms, 1024^3 FP16 315 -> 312.  Volumes in shorter
        // runs sit in the caches, and the test costs them 0.5 to 1 %.
        if constexpr (TRIM) off = (tid & 15) < w4 ? off : 0x40000000;
        // the packed-FP16 kernel forms the PER offsets anew for every box: held,
        // they would take it past the 96 registers of five waves per SIMD
        if constexpr (ST::PAIRS) asm volatile("" : "+v"(off));
#pragma unroll
        for (int i = 0; i < PER; ++i, off += (int)(16 * row_bytes)) {
            if constexpr (ST::BYTES == 4) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
                raw[i] = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]),
                                     __uint_as_float(v[2]), __uint_as_float(v[3]));
            } else {
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0);
                raw[i] = make_uint2(v[0], v[1]);
            }
        }
    }

    // rows are written in blocks of 16 (one per load) while the block starts
    // inside the box (bh uniform: a scalar branch); rows past the box in the
    // last block were loaded as zeros (outside the descriptor range), so the
    // tile stays finite
    __device__ __forceinline__ void commit(float *box, int bh, int tid) const
    {
        const int r0 = tid >> 4, col = (tid & 15) * 4;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (16 * i > bh) break;
            const int r = r0 + 16 * i;
            float *dst = box + r * ST::P + col;
            if constexpr (ST::PAIRS) {
                const uint2 w = raw[i];
                // the next lane's first two samples (DPP row shift by one
                // within the 16 lanes of a row; the last lane's 4th word, column
                // 63, is never read)
                const unsigned nx = (unsigned)__builtin_amdgcn_mov_dpp((int)w.x, 0x101, 0xf, 0xf,
                                                                       true);
                *(uint4 *)dst = make_uint4(w.x, __builtin_amdgcn_alignbyte(w.y, w.x, 2), w.y,
                                           __builtin_amdgcn_alignbyte(nx, w.y, 2));
            } else if constexpr (ST::BYTES == 4) {
                *(float4 *)dst = raw[i];
            } else {
                const uint2 w = raw[i];
                *(float4 *)dst = make_float4(ST::half(w.x, 0), ST::half(w.x, 1),
                                             ST::half(w.y, 0), ST::half(w.y, 1));
            }
        }
    }
};

// a workgroup-uniform value, kept in a scalar register
template <typename R>
__device__ __forceinline__ R uniform_load(const R *p) { return *p; }
template <>
__device__ __forceinline__ float uniform_load(const float *p)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(*p)));
}

// n / d correctly rounded (Markstein 1990: a Newton step on the reciprocal, two
// residual corrections of the quotient) for normal n, d and quotient: without
// the exponent scaling and special cases of the general division, 9
// instructions instead of 13.  The staged angles have d = D - S > D/100, and D is
// at least 1/2 and at most 2^100 here.
__device__ __forceinline__ float div_normal(float n, float d)
{
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.f), r, r);
    float q = n * r;
    q = fmaf(fmaf(-d, q, n), r, q);
    return fmaf(fmaf(-d, q, n), r, q);
}

// ---- the backprojector --------------------------------------------------------------
// G: 256-thread groups of a workgroup, each with its own box, that take the
// staged angles in turn; their sums meet in LDS at the end (see bp_shape)
template <typename S, int ZR, int G>
__global__ void __launch_bounds__(256 * G) bp_kernel(BPArgs<typename Store<S>::R> a)
{
    using R = typename Store<S>::R;
    using ST = Store<S>;
    constexpr bool STAGED = ST::STAGED;
    constexpr int BOX_H = box_rows<ZR>();
    constexpr int P = ST::P;
    constexpr int INNER_U = 1 << 30;   // flag beside an angle's index
    static_assert(P >= BOX_W && P % 4 == 0, "box pitch");
    extern __shared__ __align__(16) float bp_mem[];   // per group a.box_h rows of P words
    // per batch of 64 angles, in two slots (batches g and g+1): each group's
    // staged angles, inner ones first (first column and last row of the footprint,
    // its first row, the angle's index, cos), with their sin and scale; the
    // numbers of inner and of all staged angles of each group; and whether any
    // angle is left to pass 2.  (Kept within 3 KiB, so that five FP16 workgroups
    // fit a CU.)
    __shared__ int4 ebox[STAGED ? 128 : 1];
    __shared__ float2 ess[STAGED ? 128 : 1];
    __shared__ int2 counts[2 * G];
    __shared__ int hbm_flag;

    // XCD-aware block order: hardware dispatches workgroup i to XCD i % 8; the
    // remap gives each XCD a contiguous range of logical blocks.
    const int nb = a.nblocks;
    const int bid = blockIdx.x;
    const int per = (nb + 7) / 8;
    const int xcd = bid & 7;
    const int full = nb - (per - 1) * 8;   // XCDs that receive `per` blocks
    const int lb = (xcd < full) ? xcd * per + (bid >> 3)
                                : full * per + (xcd - full) * (per - 1) + (bid >> 3);
    const int zr = lb / a.tiles_xy;        // z-run major: neighbours share rows
    const int tile = lb - zr * a.tiles_xy;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;

    const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int tid = G == 1 ? threadIdx.x : threadIdx.x & 255;   // within the group
    float *boxmem = bp_mem + grp * (P * a.box_h);
    const int lane = threadIdx.x & 63, wave = tid >> 6;
    const int x = tx * 16 + (wave & 1) * 8 + (lane & 7);
    const int y = ty * 16 + (wave >> 1) * 8 + (lane >> 3);
    const int z0 = zr * ZR;
    const bool valid_xy = x < a.Nx && y < a.Ny;

    const R aX = valid_xy ? a.ax[x] : (R)0;
    const R aY = valid_xy ? a.ay[y] : (R)0;
    const bool inside =
        valid_xy && ((double)aX * (double)aX + (double)aY * (double)aY < a.maskR2);

    R acc[ZR];
#pragma unroll
    for (int k = 0; k < ZR; ++k) acc[k] = 0;

    // packed FP16 carries the column weights in FP16: they are normalised by
    // the largest projection scale (rounded up to a power of two, g), so they
    // stay within [0, U^2], and the sums are multiplied by g at the end
    constexpr bool PACKED = ST::PAIRS && !ST::MIX;
    R wnorm = 1, wback = 1;
    if constexpr (PACKED) {
        float m = 0.f;
        for (int i = lane; i < a.nang; i += 64) m = fmaxf(m, (float)a.scales[i]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        const float g = m > 0.f ? exp2f(ceilf(log2f(m))) : 1.f;
        wnorm = 1.f / g;
        wback = g;
    }

    // every wave of the workgroup joins the staging barriers, so the decision to
    // skip the angle loop is workgroup-wide
    if (__syncthreads_or(inside)) {
        R az[ZR];
#pragma unroll
        for (int k = 0; k < ZR; ++k) az[k] = uniform_load(a.az + z0 + k);
        const R azlo = az[0] < az[ZR - 1] ? az[0] : az[ZR - 1];
        const R azhi = az[0] < az[ZR - 1] ? az[ZR - 1] : az[0];
        // block corner coordinates
        const int xa = tx * 16, xb = min(xa + 15, a.Nx - 1);
        const int ya = ty * 16, yb = min(ya + 15, a.Ny - 1);
        const float cx0 = (float)a.ax[xa], cx1 = (float)a.ax[xb];
        const float cy0 = (float)a.ay[ya], cy1 = (float)a.ay[yb];

        // pass 1: angles whose footprint fits the LDS tile.  Wave 0 evaluates
        // a batch's 64 footprints (one per lane) and sorts the staged angles
        // into inner ones (every tap row inside the detector: gathers without
        // range tests) and edge ones; each kind runs in a loop of its own, so
        // the accumulators never pass a branch merge (which costs a copy of
        // all of them per angle).  Angles missing the detector are dropped;
        // those whose box exceeds the tile are left to pass 2.  A staged angle's
        // cos, sin and scale come from LDS, so that nothing of its set-up waits
        // for memory.
        bool need_hbm = !STAGED;
        if constexpr (STAGED) {
            const bool any_in = __any(inside), all_in = __all(inside);
            auto angles_of_group = [&](int g) {
                if (threadIdx.x >= 64) return;
                const int bb = g * 64 + lane, slot = g & 1;
                int4 q = make_int4(0, 0, 0, 0);
                float c = 0.f, s = 0.f;
                if (bb < a.nang) {
                    c = a.ang[2 * bb];
                    s = a.ang[2 * bb + 1];
                    q = footprint(c, s, cx0, cx1, cy0, cy1, azlo, azhi, a.cX, a.cZ, a.D, a.Nu,
                                  a.Nv, a.box_h);
                }
                // this lane's angle belongs to group lane % G; its rank among the
                // lanes below of the group and kind, inner ones first
                const bool staged = q.z > 0, inner = staged && (q.z & BOX_INNER_V);
                const uint64_t own = (G == 4 ? 0x1111111111111111ull
                                      : G == 2 ? 0x5555555555555555ull : ~0ull) << (lane % G);
                const uint64_t mi = __ballot(inner) & own, me = __ballot(staged && !inner) & own;
                const uint64_t mh = __ballot(q.z < 0);
                const uint64_t mk = inner ? mi : me;
                const int rank =
                    __builtin_amdgcn_mbcnt_hi((unsigned)(mk >> 32),
                                              __builtin_amdgcn_mbcnt_lo((unsigned)mk, 0)) +
                    (inner ? 0 : __popcll(mi));
                if (staged) {
                    // the index with a flag: every tap column lies on the detector
                    // (columns are below 8192, a box has at most 127 rows and 63
                    // columns)
                    const int at = slot * 64 + (lane % G) * (64 / G) + rank;
                    ebox[at] = make_int4(q.x | q.w << 16 | ((q.z & 0xff) + 3) / 4 << 24, q.y,
                                         bb | (q.z & BOX_INNER_U ? INNER_U : 0), __float_as_int(c));
                    ess[at] = make_float2(s, a.scales[bb] * wnorm);
                }
                if (lane < G)
                    counts[slot * G + lane] = make_int2(__popcll(mi), __popcll(mi) + __popcll(me));
                if (lane == 0 && mh) hbm_flag = 1;
            };
            auto uniform_int = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
            // the tile starts finite: rows of a box past its last 16-row block
            // are never written
            for (int i = tid; i < P * a.box_h; i += 256) boxmem[i] = 0.f;
            if (threadIdx.x == 0) hbm_flag = 0;
            __syncthreads();
            angles_of_group(0);
            angles_of_group(1);
            __syncthreads();
            BoxStage<S, BOX_H, (ZR > 16)> stage;
            // the box being loaded: first column, first row, last row, index (its
            // columns over 4 in the top byte of the entry)
            int bu0 = 0, bv0 = 0, bh = -1, bi = 0;
            auto issue = [&](const int4 &e) {
                const int uh = uniform_int(e.x);
                bu0 = uh & 0xffff;
                bh = uh >> 16 & 0xff;
                bv0 = uniform_int(e.y);
                bi = uniform_int(e.z);
                stage.issue(a.stack + (size_t)(bi & ~INNER_U) * a.angle_bytes, bu0, bv0, bh,
                            uh >> 24, a.row_bytes, a.Nv, tid);
            };
            // column weights and LDS offsets of the staged angle, then its gathers
            auto gather_angle = [&](auto fast_tag, int qu, int qv, bool inner_u, float wc, float ws,
                                    float wscale) {
                constexpr bool FAST = decltype(fast_tag)::value;
                // the reference's S, T, U and u with nvcc's contractions; the
                // packed-FP16 path, whose error is set by its FP16 weights,
                // takes U from the hardware reciprocal instead of the IEEE
                // quotient
                const R Sx = rfma(aX, wc, aY * ws);
                const R T = rfma(aY, wc, -(aX * ws));
                R U;
                if constexpr (PACKED)
                    U = a.D * __builtin_amdgcn_rcpf(a.D - Sx);
                else
                    U = div_normal(a.D, a.D - Sx);
                const R u = rfma(T, U, a.cX);
                const R fu = rfract(u);
                int iu = (int)u;                            // u >= 0: trunc = floor
                R W = U * U * wscale;
                R Uv = U, cz = a.cZ;
                // inactive lanes get weight 0 and sit at v = bv0, column 0; no
                // lane is inactive when every column of the wave lies in the
                // cylinder and every tap column on the detector
                if (!(all_in && inner_u)) {
                    const bool act = inside && u >= (R)0 && u <= a.umax;
                    iu = act ? iu : qu;
                    W = act ? W : (R)0;
                    Uv = act ? Uv : (R)0;
                    cz = act ? cz : (R)qv;
                }
                const R wu1 = W * fu, wu0 = W - wu1;
                half2_t wuh = {0, 0};
                if constexpr (PACKED) wuh = half2_t{(_Float16)wu0, (_Float16)wu1};
                // sample (row iv, column iu) lies at col + iv*4*P
                const char *col = (const char *)boxmem + (iu * 4 - (qu * 4 + qv * (4 * P)));
                gather_run<FAST, ST, ZR, P>(acc, az, boxmem, Uv, cz, col, wu0, wu1, wuh,
                                                a.vmax, a.one);
            };
            using fast_t = std::integral_constant<bool, true>;
            using edge_t = std::integral_constant<bool, false>;
            const int ngroups = (a.nang + 63) >> 6;
            bool loading = false;   // this group's first box is already on its way
            for (int g = 0; g < ngroups; ++g) {
                const int slot = g & 1;
                if (g > 0) {
                    // the slot of batch g-1 is free once every wave is here
                    __syncthreads();
                    angles_of_group(g + 1);
                    __syncthreads();
                }
                // this group's inner and staged angles, the most of any group, and
                // whether this group has any in the next batch
                const int ni = uniform_int(counts[slot * G + grp].x);
                const int n = uniform_int(counts[slot * G + grp].y);
                int mi = ni, me = n - ni;
                if constexpr (G > 1)
                    for (int h = 0; h < G; ++h) {
                        const int hi = uniform_int(counts[slot * G + h].x);
                        mi = max(mi, hi);
                        me = max(me, uniform_int(counts[slot * G + h].y) - hi);
                    }
                const int n1 = uniform_int(counts[(slot ^ 1) * G + grp].y);
                const int base = slot * 64 + grp * (64 / G), base1 = base ^ 64;
                if (!loading && n > 0) issue(ebox[base]);
                loading = n > 0 && g + 1 < ngroups && n1 > 0;
                // this group's entries [e0, e1), in `most` steps; while one is
                // gathered the next one's box is loaded (the next batch's first
                // after the last)
                auto run = [&](auto fast_tag, int e0, int e1, int most) {
                    for (int j = e0; G == 1 ? j < e1 : j < e0 + most; ++j) {
                        const bool mine = G == 1 || j < e1;
                        const int qu = bu0, qv = bv0, qh = bh;
                        const bool inner_u = bi & INNER_U;
                        const int at = j + 1 < n ? base + j + 1 : base1;
                        const bool more = mine && (j + 1 < n || loading);
                        const int4 e = ebox[at];            // (read, not used, if no more)
                        const int own = base + (mine ? j : 0);
                        const float wc = __int_as_float(ebox[own].w);
                        const float2 ss = ess[own];
                        __syncthreads();   // every wave is done with the previous box
                        if (mine) stage.commit(boxmem, qh, tid);
                        __syncthreads();
                        if (more) issue(e);
                        if (mine && any_in)
                            gather_angle(fast_tag, qu, qv, inner_u, wc, ss.x, ss.y);
                    }
                };
                run(fast_t{}, 0, ni, mi);
                run(edge_t{}, ni, n, me);
            }
            need_hbm = uniform_int(hbm_flag) != 0;
        }

        // pass 2: angles gathered straight from HBM -- all of them for FP64,
        // and those whose box exceeds the LDS tile for the staged types
        if (need_hbm && grp == 0 && __any(inside)) {
            const char *proj = a.stack;
            for (int b = 0; b < a.nang; ++b, proj += a.angle_bytes) {
                if constexpr (STAGED) {
                    const int4 bx = footprint(a.ang[2 * b], a.ang[2 * b + 1], cx0, cx1, cy0, cy1,
                                              azlo, azhi, a.cX, a.cZ, a.D, a.Nu, a.Nv, a.box_h);
                    if (bx.z >= 0) continue;
                }
                const R c = a.ang[2 * b], s = a.ang[2 * b + 1];
                const R Sx = rfma(aX, c, aY * s);
                const R T = rfma(aY, c, -(aX * s));
                const R U = a.D / (a.D - Sx);
                const R u = rfma(T, U, a.cX);
                const bool act = inside && u >= (R)0 && u <= a.umax;
                const R fu = rfract(u);
                const int iu = act ? (int)u : 0;
                const R W = act ? U * U * (a.scales[b] * wnorm) : (R)0;
                const R wu1 = W * fu, wu0 = W - wu1;
                const R Uv = act ? U : (R)0;
                const R cz = act ? a.cZ : (R)0;
                const char *colp = proj + (size_t)iu * ST::BYTES;
#pragma unroll
                for (int k = 0; k < ZR; ++k) {
                    const R v = rfma(az[k], Uv, cz);
                    const bool ok = act && v >= (R)0 && v <= a.vmax;
                    const int iv = ok ? (int)v : 0;
                    const R fv = rfract(v);
                    const char *p0 = colp + (size_t)iv * a.row_bytes;
                    // rows are zero-padded past Nu; row Nv-1 is only sampled
                    // with fv = 0, and its missing neighbour is replaced by itself
                    const int dn = iv + 1 < a.Nv ? (int)a.row_bytes : 0;
                    const R q00 = ST::get(p0), q01 = ST::get(p0 + ST::BYTES);
                    const R q10 = ST::get(p0 + dn), q11 = ST::get(p0 + dn + ST::BYTES);
                    const R c0 = rfma(fv, q10 - q00, q00);
                    const R c1 = rfma(fv, q11 - q01, q01);
                    acc[k] = rfma(ok ? wu1 : (R)0, c1, rfma(ok ? wu0 : (R)0, c0, acc[k]));
                }
            }
        }
    }

    if constexpr (G > 1) {
        // the groups' sums, through LDS in pieces that fit one box (at least 16
        // rows), added in the order of the groups
        constexpr int BP_PIECE = 4;
        static_assert(BP_PIECE * 256 <= 16 * P, "piece of the group sums beyond a box");
#pragma unroll
        for (int h = 1; h < G; ++h)
#pragma unroll
            for (int k0 = 0; k0 < ZR; k0 += BP_PIECE) {
                __syncthreads();
                if (grp == h) {
#pragma unroll
                    for (int k = 0; k < BP_PIECE; ++k)
                        if (k0 + k < ZR) bp_mem[k * 256 + tid] = acc[k0 + k];
                }
                __syncthreads();
                if (grp == 0) {
#pragma unroll
                    for (int k = 0; k < BP_PIECE; ++k)
                        if (k0 + k < ZR) acc[k0 + k] += bp_mem[k * 256 + tid];
                }
            }
        if (grp > 0) return;
    }
    if (!valid_xy) return;
    const size_t plane = (size_t)a.Nx * a.Ny;
    R *out = a.vol + (size_t)y * a.Nx + x;
#pragma unroll
    for (int k = 0; k < ZR; ++k) {
        const int z = z0 + k;
        if (z < a.Nz) {
            const R r = inside ? acc[k] * (a.out_scale * wback) : (R)0;
            if (a.accumulate)
                out[(size_t)z * plane] += r;
            else
                out[(size_t)z * plane] = r;
        }
    }
}

static int native_zrun(int dtype)
{
    switch (dtype) {
    case FDK_F32: return Store<st_f32>::ZR;
    case FDK_F16: return Store<st_f16>::ZR;
    case FDK_F16_PACKED: return Store<st_f16p>::ZR;
    case FDK_BF16: return Store<st_bf16>::ZR;
    case FDK_F64: return Store<st_f64>::ZR;
    default: return 0;
    }
}

// The long z-runs (slices per thread, TKV_BP_ZR_*) spread a column's set-up over the
// most updates and read each box row for the most slices, but a volume of few blocks
// leaves CUs idle, or ends on a mostly idle last wave.  So a smaller volume takes runs of 16 slices, and one
// whose blocks still don't fill the 256 CUs has 2 or 4 groups of 256 threads per
// block, each gathering every 2nd or 4th angle from a box of its own; their sums
// meet in LDS.  By blocks of 16^3 voxels; us for the long runs, runs of 16 with 1, 2, 4
// groups, runs of 8 with 4 groups, FP32 / FP16 (BF16 like FP16; packed FP16 within 10 %
// at the shapes taken):
//       8  32^3, 36                      57 / 57        34 / 35        26 / 26        24 / 24        17 / 18
//      64  64^3, 90                    133 / 133        83 / 85        60 / 61        51 / 52        37 / 37
//     108  96^2 x 40, 120              180 / 220      133 / 136        90 / 90        70 / 70        42 / 43
//     180  96^2 x 80, 150              223 / 278      139 / 142        97 / 98        78 / 79      101 / 103
//     512  128^3, 180                  302 / 269      198 / 201      160 / 161      184 / 186      239 / 246
//    1000  160^2 x 150, 240            498 / 528      406 / 407      438 / 402      508 / 516      636 / 655
//    1560  203 x 190 x 157, 251        713 / 676      562 / 556      643 / 574      769 / 782    1056 / 1090
//    4096  256^3, 360                1907 / 1828    1817 / 1769    2125 / 1881    2638 / 2690    3606 / 3708
//    7600  320^2 x 300, 360          3267 / 3355    3212 / 3104    3886 / 3390    4878 / 4967    6652 / 6844
//   15625  400^3, 400                6924 / 7004    7112 / 6780    8740 / 7567  11195 / 11413  15583 / 16031
// One rule serves all types, where a single one could do better: FP32 by 8 % with one
// group at 1000 blocks, 16-bit samples by 3 % with runs of 16 at 15625.
// Taken from the whole volume and from neither the angles nor the slices of one
// launch, so that a volume in z-chunks gets the sums of one launch.  (FP64 gathers
// from HBM without boxes and keeps its runs of 8.)
BPShape bp_shape(int dtype, int Nx, int Ny, int Nz)
{
    const int native = native_zrun(dtype);
    const long long n = (long long)((Nx + 15) / 16) * ((Ny + 15) / 16) * ((Nz + 15) / 16);
    if (dtype == FDK_F64 || n > 8192) return {native, 1, native};
    if (n <= 128) return {8, 4, 32};
    if (n <= 256) return {16, 4, 32};
    if (n <= 1024) return {16, 2, 32};
    return {16, 1, 32};
}

int sample_bytes_of(int dtype)
{
    switch (dtype) {
    case FDK_F32: return 4;
    case FDK_F16: return 2;
    case FDK_F16_PACKED: return 2;
    case FDK_BF16: return 2;
    case FDK_F64: return 8;
    default: return 0;
    }
}

// Rows of the LDS box that every block of this geometry fits (footprint() counts
// a box's rows plus the +1 neighbour and two of margin either side), a multiple
// of the 16 rows a load covers, at most box_rows: a workgroup takes no more LDS
// than its geometry needs, which at two samples per voxel leaves room for five
// workgroups on a CU instead of four (BF16 512^3 from 900 x 1024^2: 37.5 ms
// with 96 rows, 36.1 with 80).
template <int ZR>
static int box_height(const BPLaunch &L)
{
    const double reach = std::sqrt(L.maskR2) + 22. * L.scale;   // a tile's far corner
    const double U = L.D > reach ? L.D / (L.D - reach) : 100.;
    // U varies over a tile (15 sqrt 2 voxels across) by at most U^2/D per unit of S
    const double rows = (ZR - 1) * L.scale * U + L.az_max * 21.3 * L.scale * U * U / L.D + 8.;
    const int most = box_rows<ZR>();
    return rows >= most ? most : ((int)rows + 16) / 16 * 16;
}

template <typename S, int ZR, int G>
static int launch_bp_z(const BPLaunch &L, hipStream_t st)
{
    using R = typename Store<S>::R;
    if (L.pitch < stack_pitch(L.Nu))
        return fail(FDK_ERR_INVALID_ARGUMENT, "backproject: stack pitch below the padded width");
    BPArgs<R> a;
    a.stack = (const char *)L.stack;
    a.row_bytes = (uint32_t)((size_t)L.pitch * Store<S>::BYTES);
    a.angle_bytes = (size_t)a.row_bytes * L.Nv;
    if (a.angle_bytes > 0x7fffffffULL)
        return fail(FDK_ERR_UNSUPPORTED, "backproject: projection of 2 GiB or more");
    a.ang = (const R *)L.ang;
    a.scales = (const R *)L.scales;
    a.ax = (const R *)L.ax;
    a.ay = (const R *)L.ay;
    a.az = (const R *)L.az;
    a.vol = (R *)L.vol;
    a.Nx = L.Nx;
    a.Ny = L.Ny;
    a.Nz = L.Nz;
    a.Nu = L.Nu;
    a.Nv = L.Nv;
    a.nang = L.nang;
    a.cX = (R)L.cX;
    a.cZ = (R)L.cZ;
    // FP32: from 2^100 on D - S rounds to D and U is 1 (|S| < 4096 in the cylinder),
    // and the reciprocal in div_normal stays a normal number
    const bool far = sizeof(R) == 4 && L.D > 0x1p100 && std::isfinite((R)L.D);
    a.D = far ? (R)0x1p100 : (R)L.D;
    a.umax = (R)(L.Nu - 1);
    a.vmax = (R)(L.Nv - 1);
    a.out_scale = (R)L.out_scale;
    a.one = (R)1;
    a.maskR2 = L.maskR2;
    a.accumulate = L.accumulate;
    a.tiles_x = (L.Nx + 15) / 16;
    a.tiles_xy = a.tiles_x * ((L.Ny + 15) / 16);
    const long long nzrun = (L.Nz + ZR - 1) / ZR;
    const long long nb = (long long)a.tiles_xy * nzrun;
    if (nb == 0) return FDK_OK;
    if (!grid_fits(nb, 256)) return fail(FDK_ERR_UNSUPPORTED, "backproject: volume too large");
    a.nblocks = (int)nb;
    a.box_h = Store<S>::STAGED ? box_height<ZR>(L) : 0;
    const size_t lds = sizeof(float) * Store<S>::P * a.box_h * G;
    // beyond 64 KiB a workgroup takes up to the 160 KiB of LDS of a gfx950 CU
    if (lds > 61440)
        TKV_HIP(hipFuncSetAttribute((const void *)bp_kernel<S, ZR, G>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((bp_kernel<S, ZR, G>), dim3((unsigned)nb), dim3(256 * G), lds, st, a);
    TKV_HIP(hipGetLastError());
    return FDK_OK;
}

template <typename S>
static int launch_bp_t(const BPLaunch &L, hipStream_t st)
{
    constexpr int ZR = Store<S>::ZR;
    const int z = L.shape.zrun, g = L.shape.groups;
    if (z == ZR && g == 1) {
        // FP32 samples of a box of more than 80 rows leave room for four workgroups
        // on a CU, FP16 pairs for five, and boxes that high are those of wide
        // samplings and steep rays, whose gathers meet in the LDS banks: 512^3 at two
        // samples per voxel from 150 angles, D 4096 (96 rows), 5.88 ms with pairs and
        // 6.98 with FP32 samples.  With 80 rows the FP32 samples win: 512^3 from 900,
        // D 10000, 38.8 and 36.8 ms; 512^2 x 300 at 1.8 samples from 150, 4.14 and 3.52.
        if constexpr (std::is_same<S, st_f16>::value)
            if (box_height<ZR>(L) > 80) return launch_bp_z<st_f16m, ZR, 1>(L, st);
        return launch_bp_z<S, ZR, 1>(L, st);
    }
    if constexpr (Store<S>::STAGED) {
        if (z == 8 && g == 4) return launch_bp_z<S, 8, 4>(L, st);
        if (z == 16 && g == 4) return launch_bp_z<S, 16, 4>(L, st);
        if (z == 16 && g == 2) return launch_bp_z<S, 16, 2>(L, st);
        if (z == 16 && g == 1) return launch_bp_z<S, 16, 1>(L, st);
    }
    return fail(FDK_ERR_INVALID_ARGUMENT, "backproject: no kernel of this shape");
}

int launch_backproject(int dtype, const BPLaunch &a, hipStream_t st)
{
    switch (dtype) {
    case FDK_F32: return launch_bp_t<st_f32>(a, st);
    case FDK_F16: return launch_bp_t<st_f16>(a, st);
    case FDK_F16_PACKED: return launch_bp_t<st_f16p>(a, st);
    case FDK_BF16: return launch_bp_t<st_bf16>(a, st);
    case FDK_F64: return launch_bp_t<st_f64>(a, st);
    default: return fail(FDK_ERR_INVALID_ARGUMENT, "backproject: unknown storage type");
    }
}

}  // namespace tkv
