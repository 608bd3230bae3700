// Scanco RSQ raw projections: header on the host, preprocessing on the GPU.
//
// The raw sinograms stay 16-bit until they are on the device (a quarter of the
// bytes of the reference's FP64 sinograms cross the host link).  Every output
// sample comes from at most two raw samples: flat/dark correction and the
// beam-hardening line on each, and for the full-fan rebinning the linear
// interpolation between the two angle rows of the redundant ray.
//
// All arithmetic is FP64 in the reference's order of operations (no contraction
// into FMAs, except inside the quotient and the logarithm, which are functions of
// their own: the quotient is the correctly rounded one, the logarithm is within
// 0.52 ulp), so a result does not depend on how the work is cut.
#include "tomokvas/fdk.h"
#include "tomokvas/fdk_rsq.h"
#include "fdk_internal.hpp"

#include <hip/hip_runtime.h>
#include <sys/types.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#pragma clang fp contract(off)

using tkv::fail;

namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr int kHeaderBytes = 512;     // sizeof(ima_data_type)
constexpr int kBhOffset = 3432, kBhBytes = 152;

struct RsqArgs {
    const uint16_t *raw;   // [n][sin_y + 2][sin_x]
    void *out;             // [n][sy][sx]
    int sin_x, sin_y, sx, sy, axis_move, start, flip, invert;
    int nsin, rows;        // sinograms; angle rows per wave
    int waves_x, tiles_x, tiles_y;   // log2 of a workgroup's waves side by side; tiles
    double A, B, distance, delta_fi, inv_delta;
};

// ---- logarithm --------------------------------------------------------------------
// Table-driven FP64 log of a positive normal number (the scheme of P. T. P. Tang,
// "Table-driven implementation of the logarithm function in IEEE floating-point
// arithmetic", ACM TOMS 16(4), 1990): x = 2^e m with m in [0.703125, 1.40625), the
// interval of m (128 of them) gives inv close to 1/m in 8 bits and -log(inv) as
// hi + lo, r = m inv - 1 is exact, and log x = (e ln2 + hi) + r + (lo + log1p(r) - r)
// with the first sum exact (hi and ln2_hi are multiples of 2^-42) and the second
// one's rounding carried along.  The two intervals that meet at 1 have inv = 1 and
// hi = lo = 0, so log x is accurate to the last bit around 1 too.  Within 0.52 ulp
// over the quotients of 16-bit counts (the device library's log is within 1).
struct LogTable {
    double inv[128], hi[128], lo[128], ln2_hi, ln2_lo;
};

constexpr LogTable make_log_table()
{
    LogTable t{};
    for (int i = 0; i <= 128; ++i) {   // the last entry is ln 2 = -log(256/512)
        // 512 over the centre of the interval, rounded to a multiple of 2
        const int num = i < 76 ? 512 * 512 : 512 * 256;
        const int den = i < 76 ? 360 + 2 * i + 1 : 256 + 2 * (i - 76) + 1;
        const int j = i == 128 ? 256 : i == 75 || i == 76 ? 512 : (num + den) / (2 * den) * 2;
        // -log(j/512) = 2 atanh((512 - j)/(512 + j)) in units of 2^-100
        const int a = 512 - j, b = 512 + j;
        __int128 term = ((__int128)1 << 101) / b * a, sum = 0;
        for (int k = 1; k < 60; k += 2) {
            sum += term / k;
            term = term / (b * b) * (a * a);
        }
        const __int128 one = (__int128)1 << 58;
        const __int128 h = (sum + (sum < 0 ? -one : one) / 2) / one;
        const double hi = (double)(long long)h * 0x1p-42;
        const double lo = (double)(long long)(sum - h * one) * 0x1p-100;
        if (i < 128) {
            t.inv[i] = j / 512.;
            t.hi[i] = hi;
            t.lo[i] = lo;
        } else {
            t.ln2_hi = hi;
            t.ln2_lo = lo;
        }
    }
    return t;
}

constexpr LogTable kLog = make_log_table();
__device__ const LogTable d_log = make_log_table();

struct LogLds {
    double2 inv_hi[128];
    double lo[128];
};

__device__ __forceinline__ double log_table(double x, const LogLds &t)
{
    const int hi = __double2hiint(x);
    const int o = hi - 0x3fe68000;   // 0.703125
    const int e = o >> 20, i = (o >> 13) & 127;
    const double m = __hiloint2double(hi - (o & 0xfff00000), __double2loint(x));
    const double2 ih = t.inv_hi[i];
    const double r = fma(m, ih.x, -1.);
    const double c = fma((double)e, kLog.ln2_hi, ih.y);
    const double s = c + r;
    double p = fma(r, -1. / 8, 1. / 7);
    p = fma(r, p, -1. / 6);
    p = fma(r, p, 1. / 5);
    p = fma(r, p, -1. / 4);
    p = fma(r, p, 1. / 3);
    p = fma(r, p, -1. / 2);
    const double low = ((c - s) + r) + fma((double)e, kLog.ln2_lo, t.lo[i]);
    return s + fma(r * r, p, low);
}

// a / b, correctly rounded, from b's correctly rounded reciprocal (P. W. Markstein,
// "Computation of elementary functions on the IBM RISC System/6000 processor", IBM
// J. Res. Dev. 34(1), 1990); NaN for b = 0
__device__ __forceinline__ double quotient(double a, double b, double rcp_b)
{
    const double q = a * rcp_b;
    return fma(fma(-q, b, a), rcp_b, q);
}

// line integral of a raw count i on a column of dark count d and flat - dark = b
// (FlatFieldCorrection, rsq_load.cpp:299-325)
__device__ __forceinline__ double line_integral(const RsqArgs &a, const LogLds &t, int i, int d,
                                                double b, double rcp_b)
{
    const double q = quotient((double)(i - d), b, rcp_b);
    double v = log_table(q, t);
    if (!(q > 0)) {   // no flat field, or a count at or below dark
        const double z = (double)(i - d) / b;
        v = z > 0 ? INFINITY : z == 0 ? -INFINITY : NAN;
    }
    v = a.A * v + a.B;
    return a.invert ? -v : v;
}

// The line integrals of columns axis_move .. sin_x-1, once each, and from them the
// measured half of the output (CutHalfSin, rsq_load.cpp:393-410: all of it) and for
// FULL the redundant rays (Half2FullFan, :327-391).
//
// A lane owns column x and walks `rows` angle rows of K sinograms.  The redundant
// ray of output angle f at x columns left of the central ray lies between two
// consecutive rows ib, ia of column x, nearly a constant number of rows from f: a
// lane that has just computed row y owns the output angle f = y - shift(x), whose
// pair is then (y - 1, y).  That assignment only says which lane writes f: the pair
// and its weight are computed as the reference does, from f, and where they come
// out otherwise (rounding, or delta_fi other than 2 pi / sin_y) the two line
// integrals are computed for this output alone.  So each raw sample is read and
// each logarithm taken once, and no line integral goes through memory.
//
// K sinograms share the pair and the weight of an output angle.  Bound by the FP64
// issue and by the stores: 248 sinograms of 2000 x 1024, full fan in FP32, take 1.88
// ms (2.7 TB/s of raw and output bytes; 1.33 without the redundant half's stores),
// where the device library's log and division and the line integrals through an
// FP64 scratch took 4.56.  A wave's redundant outputs of one step spread over about
// 8 rows, whose cache lines fill over the next steps: the measured half's stores
// bypass the caches there, so that those lines stay in L2 until they are whole (2.0
// ms otherwise; without the redundant half the caches are the better way, 0.66
// against 0.74 ms for 200 sinograms).
template <typename T, bool FULL, int K>
__global__ void __launch_bounds__(256) rsq_kernel(RsqArgs a)
{
    __shared__ LogLds tab;
    for (int i = threadIdx.x; i < 128; i += 256) {
        tab.inv_hi[i] = make_double2(d_log.inv[i], d_log.hi[i]);
        tab.lo[i] = d_log.lo[i];
    }
    __syncthreads();
    const int w = a.sin_x - a.axis_move, N = a.sin_y;
    // workgroup i runs on XCD i % 8: each XCD takes a contiguous range of logical
    // blocks, column tiles fastest, so that the cache lines that two tiles share
    // meet in one L2
    const int nb = gridDim.x, xcd = blockIdx.x & 7, more = nb & 7;
    const int lb = xcd * (nb >> 3) + min(xcd, more) + (blockIdx.x >> 3);
    const int by = lb / a.tiles_x, bx = lb - by * a.tiles_x;
    const int bz = by / a.tiles_y, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = ((bx << a.waves_x) + (wave & ((1 << a.waves_x) - 1))) * 64 + (threadIdx.x & 63);
    const long long y00 =
        (long long)(((by - bz * a.tiles_y) << (2 - a.waves_x)) + (wave >> a.waves_x)) * a.rows;
    if (x >= w || y00 >= N) return;
    const int y0 = (int)y00, y1 = min(y0 + a.rows, N);
    const int k0 = bz * K, nk = min(K, a.nsin - k0);
    const size_t per = (size_t)(N + 2) * a.sin_x, ostride = (size_t)a.sy * a.sx;
    const uint16_t *raw = a.raw + k0 * per + a.axis_move;
    T *out = static_cast<T *>(a.out) + k0 * ostride;
    // sinograms past the last one repeat it, without stores
    int d[K];
    double b[K], rcp[K];
    const uint16_t *col[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        col[k] = raw + min(k, nk - 1) * per;
        d[k] = col[k][x];
        b[k] = (double)(col[k][a.sin_x + x] - d[k]);
        rcp[k] = 1. / b[k];
    }
    auto count = [&](int k, int y) -> int { return col[k][(size_t)(y + 2) * a.sin_x + x]; };
    auto line = [&](int k, int i) { return line_integral(a, tab, i, d[k], b[k], rcp[k]); };
    // output row of angle row f
    auto row_of = [&](int f) { return a.flip ? a.sy - 1 - f + a.start : f; };

    const int c0 = FULL ? w - 1 : 0;   // output column of the central ray
    const double at2 = 2 * atan(-x / a.distance);
    int ia, ib;
    double wgt;
    bool two;
    auto pair_of = [&](int f) {
        const double fi = f * a.delta_fi, base = fi - at2;
        double nf = quotient(base - kPi, a.delta_fi, a.inv_delta);
        if (nf > N - 1 || nf < 0) nf = quotient(base + kPi, a.delta_fi, a.inv_delta);
        const double ca = ceil(nf), fb = floor(nf);
        ia = (int)ca;
        ib = (int)fb;
        // inside the scan for delta_fi = 2 pi / sin_y (ia <= sin_y wraps to row 0
        // as in the reference); any other angle wraps too
        if ((unsigned)ia >= (unsigned)N) ia = ((ia % N) + N) % N;
        if ((unsigned)ib >= (unsigned)N) ib = ((ib % N) + N) % N;
        wgt = -nf + ca;
        two = ca != fb;
    };
    int shift = 0;
    double prev[K];
    if constexpr (FULL) {
        pair_of(0);
        shift = ia;
#pragma unroll
        for (int k = 0; k < K; ++k) prev[k] = line(k, count(k, y0 > 0 ? y0 - 1 : N - 1));
    }
    int next[K];
#pragma unroll
    for (int k = 0; k < K; ++k) next[k] = count(k, y0);
    for (int y = y0; y < y1; ++y) {
        double v[K];
        int i[K];
#pragma unroll
        for (int k = 0; k < K; ++k) i[k] = next[k];
#pragma unroll
        for (int k = 0; k < K; ++k) next[k] = count(k, min(y + 1, N - 1));
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = line(k, i[k]);
        const int r = row_of(y);
        if (r >= 0 && r < a.sy) {
            T *o = out + (size_t)r * a.sx + c0;
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (k < nk) {
                    if constexpr (FULL) __builtin_nontemporal_store((T)v[k], &o[k * ostride + x]);
                    else o[k * ostride + x] = (T)v[k];
                }
        }
        if constexpr (FULL) {
            const int f = y >= shift ? y - shift : y - shift + N;
            const int q = row_of(f);
            if (x > 0 && q >= 0 && q < a.sy) {
                pair_of(f);
                T *o = out + (size_t)q * a.sx + (c0 - x);
                if (ia == y && (!two || ib == (y > 0 ? y - 1 : N - 1))) {
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (k < nk) o[k * ostride] = (T)(two ? v[k] + (prev[k] - v[k]) * wgt : v[k]);
                } else {
                    for (int k = 0; k < nk; ++k) {
                        const uint16_t *s = raw + k * per;
                        const int dk = s[x];
                        const double bk = (double)(s[a.sin_x + x] - dk), rk = 1. / bk;
                        double u = line_integral(a, tab, s[(size_t)(ia + 2) * a.sin_x + x], dk, bk, rk);
                        if (two) {
                            const double l =
                                line_integral(a, tab, s[(size_t)(ib + 2) * a.sin_x + x], dk, bk, rk);
                            u = u + (l - u) * wgt;
                        }
                        o[k * ostride] = (T)u;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) prev[k] = v[k];
        }
    }
}

template <typename T, bool FULL, int K>
hipError_t launch_rsq_k(RsqArgs a, hipStream_t st)
{
    // a launch takes at most 2^32 - 1 threads
    const long long tiles = (long long)a.tiles_x * a.tiles_y;
    const int n = a.nsin, most = (int)std::max(1LL, std::min((1LL << 23) / tiles, 1LL << 23)) * K;
    for (int k0 = 0; k0 < n; k0 += most) {
        a.nsin = std::min(n - k0, most);
        const long long blocks = tiles * ((a.nsin + K - 1) / K);
        hipLaunchKernelGGL((rsq_kernel<T, FULL, K>), dim3((unsigned)blocks), dim3(256), 0, st, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        a.raw += (size_t)a.nsin * (a.sin_y + 2) * a.sin_x;
        a.out = static_cast<T *>(a.out) + (size_t)a.nsin * a.sy * a.sx;
    }
    return hipSuccess;
}

template <typename T, bool FULL>
hipError_t launch_rsq(RsqArgs a, hipStream_t st)
{
    // Four waves side by side where the columns allow (whole cache lines between
    // them: 0.66 against 0.75 ms for the 200 sinograms above).  16 rows per wave,
    // whose set-up (table, reciprocals, first row) they pay for; 8, and 4, where
    // that leaves the chip with too few waves: 20 sinograms of 700 x 300 take 42 us
    // with 16, 41 with 8 and 44 with 4 rows, 4 of 360 x 96 take 30, 24 and 21.
    const int w = a.sin_x - a.axis_move;
    const long long cols = (w + 63) / 64, groups = (a.nsin + 1) / 2;
    auto waves = [&](int rows) { return cols * ((a.sin_y + rows - 1) / rows) * groups; };
    a.rows = waves(16) >= 4096 ? 16 : waves(8) >= 1024 ? 8 : 4;
    a.waves_x = w > 128 ? 2 : w > 64 ? 1 : 0;
    a.tiles_x = (int)((cols + (1 << a.waves_x) - 1) >> a.waves_x);
    a.tiles_y = (a.sin_y + (a.rows << (2 - a.waves_x)) - 1) / (a.rows << (2 - a.waves_x));
    return a.nsin > 1 ? launch_rsq_k<T, FULL, 2>(a, st) : launch_rsq_k<T, FULL, 1>(a, st);
}

int read_i32(const unsigned char *b, int off)
{
    int v;
    std::memcpy(&v, b + off, 4);   // little-endian file, little-endian host
    return v;
}

// the file layout: sinogram size and data offset
int check_layout(const fdk_rsq_params *p)
{
    if (!p) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null parameters");
    if (p->sin_x < 1 || p->sin_y < 1 || p->header_offset < 0)
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: sizes must be positive");
    return FDK_OK;
}

// the layout and the processing options
int check_params(const fdk_rsq_params *p)
{
    if (int rc = check_layout(p)) return rc;
    if (p->axis_move < 0 || p->axis_move >= p->sin_x)
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: axis_move outside the detector");
    if (p->complete && (!(p->distance > 0) || !(p->delta_fi > 0)))
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: distance and delta_fi must be positive");
    return FDK_OK;
}

// CalculateSizeOfSinogram (rsq_load.cpp:82-105), parallel branch not provided
void out_size(const fdk_rsq_params *p, int *sx, int *sy)
{
    if (p->complete) {
        *sx = 2 * p->sin_x - 1 - 2 * p->axis_move;
        *sy = p->minimal ? (int)std::ceil((kPi + 2 * std::atan(*sx / 2. / p->distance)) / p->delta_fi)
                         : p->sin_y;
        if (p->minimal && *sy > p->sin_y) *sy = p->sin_y;
    } else {
        *sx = p->sin_x - p->axis_move;
        *sy = p->sin_y;
    }
}

}  // namespace

struct fdk_rsq {
    std::string path;
    fdk_rsq_header h{};
};

extern "C" int fdk_rsq_default_params(fdk_rsq_params *p)
{
    if (!p) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null parameters");
    p->sin_x = 1024;
    p->sin_y = 2000;
    p->header_offset = 3584;
    p->axis_move = 21;
    p->distance = 125810. / 24.;
    p->delta_fi = 2 * kPi / p->sin_y;
    p->flip = p->invert = p->complete = p->minimal = 0;
    return FDK_OK;
}

extern "C" int fdk_rsq_open(const char *path, fdk_rsq **out)
{
    if (!path || !out) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null argument");
    *out = nullptr;
    FILE *f = std::fopen(path, "rb");
    if (!f) return fail(FDK_ERR_INVALID_ARGUMENT, std::string("rsq: cannot open ") + path);
    unsigned char b[kBhOffset + kBhBytes] = {};
    const size_t got = std::fread(b, 1, sizeof b, f);
    fseeko(f, 0, SEEK_END);
    const long long size = (long long)ftello(f);
    std::fclose(f);
    if (got < sizeof b) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: file shorter than its header");
    auto *r = new fdk_rsq;
    r->path = path;
    fdk_rsq_header &h = r->h;
    // ima_data_type (rsq_load.h:13-49): check[16], then 4-byte ints; name[40]
    // at 128, data_offset the last int of the 512 bytes
    std::memcpy(h.check, b, 16);
    h.check[16] = 0;
    h.data_type = read_i32(b, 16);
    h.nr_of_bytes = read_i32(b, 20);
    h.nr_of_blocks = read_i32(b, 24);
    h.patient_index = read_i32(b, 28);
    h.scanner_id = read_i32(b, 32);
    h.dimx_p = read_i32(b, 44);
    h.dimy_p = read_i32(b, 48);
    h.dimz_p = read_i32(b, 52);
    h.dimx_um = read_i32(b, 56);
    h.dimy_um = read_i32(b, 60);
    h.dimz_um = read_i32(b, 64);
    h.mu_scaling = read_i32(b, 88);
    h.nr_of_samples = read_i32(b, 92);
    h.nr_of_projections = read_i32(b, 96);
    h.scandist_um = read_i32(b, 100);
    h.scanner_type = read_i32(b, 104);
    h.reference_line_um = read_i32(b, 120);
    h.energy = read_i32(b, 168);
    h.intensity = read_i32(b, 172);
    h.data_offset = read_i32(b, kHeaderBytes - 4);
    h.file_size = size;
    char bh[kBhBytes + 1];
    std::memcpy(bh, b + kBhOffset, kBhBytes);
    bh[kBhBytes] = 0;
    if (std::sscanf(bh, "Corr at %d %d %d: %lf %lf %lf", &h.bh_x[0], &h.bh_x[1], &h.bh_x[2],
                    &h.bh_y[0], &h.bh_y[1], &h.bh_y[2]) != 6 ||
        h.bh_x[2] == h.bh_x[0]) {
        delete r;
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: no beam-hardening line at byte 3432");
    }
    h.bh_a = (h.bh_y[2] - h.bh_y[0]) / (h.bh_x[2] - h.bh_x[0]);
    h.bh_b = h.bh_y[0] - h.bh_a * h.bh_x[0];
    *out = r;
    return FDK_OK;
}

extern "C" void fdk_rsq_close(fdk_rsq *r) { delete r; }

extern "C" int fdk_rsq_get_header(const fdk_rsq *r, fdk_rsq_header *h)
{
    if (!r || !h) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null argument");
    *h = r->h;
    return FDK_OK;
}

namespace {
int count_sinograms(const fdk_rsq *r, const fdk_rsq_params *p)
{
    const long long per = 2LL * p->sin_x * (p->sin_y + 2);
    const long long data = r->h.file_size - p->header_offset;
    return data > 0 ? (int)(data / per) : 0;
}
}  // namespace

extern "C" int fdk_rsq_sizes(const fdk_rsq *r, const fdk_rsq_params *p, int *num, int *sx,
                             int *sy)
{
    if (!r || !num || !sx || !sy) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null argument");
    int rc = check_params(p);
    if (rc) return rc;
    *num = count_sinograms(r, p);
    out_size(p, sx, sy);
    return FDK_OK;
}

extern "C" int fdk_rsq_load(const fdk_rsq *r, const fdk_rsq_params *p, int first, int last,
                            uint16_t *dst)
{
    if (!r || !dst) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null argument");
    int rc = check_layout(p);
    if (rc) return rc;
    const int num = count_sinograms(r, p);
    if (first < 0 || last < first || last >= num)
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: sinograms " + std::to_string(first) + ".." +
                                                  std::to_string(last) + " outside 0.." +
                                                  std::to_string(num - 1));
    FILE *f = std::fopen(r->path.c_str(), "rb");
    if (!f) return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: cannot open " + r->path);
    const size_t per = (size_t)p->sin_x * (p->sin_y + 2);
    const size_t count = per * (size_t)(last + 1 - first);
    const off_t off = (off_t)(p->header_offset + (long long)per * 2 * first);
    const bool ok = fseeko(f, off, SEEK_SET) == 0 && std::fread(dst, 2, count, f) == count;
    std::fclose(f);
    return ok ? FDK_OK : fail(FDK_ERR_INVALID_ARGUMENT, "rsq: short read from " + r->path);
}

extern "C" int fdk_rsq_process(const fdk_rsq_params *p, double bh_a, double bh_b,
                               const uint16_t *d_raw, int nsin, int out_dtype, void *d_out,
                               void *stream)
{
    int rc = check_params(p);
    if (rc) return rc;
    if (!d_raw || !d_out || nsin < 0)
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: null buffer or negative count");
    if (out_dtype != FDK_F32 && out_dtype != FDK_F64)
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: output must be FDK_F32 or FDK_F64");
    RsqArgs a;
    a.raw = d_raw;
    a.out = d_out;
    a.sin_x = p->sin_x;
    a.sin_y = p->sin_y;
    out_size(p, &a.sx, &a.sy);
    a.axis_move = p->axis_move;
    a.start = p->flip && p->complete ? p->sin_y - a.sy : 0;
    a.flip = p->flip;
    a.invert = p->invert;
    a.A = bh_a;
    a.B = bh_b;
    a.distance = p->distance;
    a.delta_fi = p->delta_fi;
    a.inv_delta = 1. / p->delta_fi;
    if ((size_t)a.sx * a.sy * nsin == 0) return FDK_OK;
    if (a.sin_y > 65535)
        return fail(FDK_ERR_INVALID_ARGUMENT, "rsq: more than 65535 projections per sinogram");
    hipStream_t st = (hipStream_t)stream;
    const bool f64 = out_dtype == FDK_F64, full = p->complete;
    a.nsin = nsin;
    const hipError_t e = full ? (f64 ? launch_rsq<double, true>(a, st) : launch_rsq<float, true>(a, st))
                              : (f64 ? launch_rsq<double, false>(a, st) : launch_rsq<float, false>(a, st));
    if (e != hipSuccess) return tkv::hip_fail(e, "rsq");
    // the full fan is complete when the call returns
    if (full) TKV_HIP(hipStreamSynchronize(st));
    return FDK_OK;
}
