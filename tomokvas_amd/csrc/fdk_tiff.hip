// TIFF export of reconstructed slices, device part: range and 16-bit scaling
// on the GPU, files written by the host writer of fdk_tiff_host.cpp.
//
// The scaling u = (unsigned short)(65535 * (x - min) / (max - min)) is
// evaluated in FP64 in that order (no FMA contraction), on the device and on
// the host alike, so both paths write the same bytes.  Values outside
// [min, max] clamp to 0 / 65535 and NaN gives 0 (the reference's conversion
// of such values to unsigned short is undefined).
#include "tomokvas/fdk.h"
#include "tomokvas/fdk_tiff.h"
#include "fdk_internal.hpp"
#include "fdk_tiff_internal.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#pragma clang fp contract(off)

using tkv::fail;
using tkv::scale_u16;
using tkv::write_slices;
using tkv::write_slices_parallel;
using tkv::writer_threads;

namespace {

// Range of a volume: every workgroup leaves its smallest and largest value (NaN
// skipped; +inf, -inf where it saw none) in part, the host reduces them.
// HBM-bound: 2048 workgroups (8 per CU), each thread with four 16-byte loads in
// flight.  Ordered integer keys raised with two atomics per workgroup of 8192
// had taken 222 us for 512^3 floats: 16384 atomics on one cache line.
// VEC: v is 16-byte aligned; the body reads float4 and the last n % 4
// values one by one
constexpr int kRangeBlocks = 2048;

template <bool VEC>
__global__ void __launch_bounds__(256) minmax_kernel(const float *__restrict__ v, size_t n,
                                                     float2 *__restrict__ part)
{
    float lo = __builtin_inff(), hi = -__builtin_inff();
    auto take = [&](float x) {   // fmin and fmax return the other operand for a NaN
        lo = fminf(lo, x);
        hi = fmaxf(hi, x);
    };
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nth = (size_t)gridDim.x * blockDim.x;
    size_t done = 0;
    if (VEC) {
        const float4 *v4 = reinterpret_cast<const float4 *>(v);
        const size_t n4 = n / 4;
        size_t i = tid;
        for (; i + 3 * nth < n4; i += 4 * nth) {
            const float4 q[4] = {v4[i], v4[i + nth], v4[i + 2 * nth], v4[i + 3 * nth]};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                take(q[j].x);
                take(q[j].y);
                take(q[j].z);
                take(q[j].w);
            }
        }
        for (; i < n4; i += nth) {
            const float4 q = v4[i];
            take(q.x);
            take(q.y);
            take(q.z);
            take(q.w);
        }
        done = 4 * n4;
    }
    for (size_t i = done + tid; i < n; i += nth) take(v[i]);
    for (int o = 32; o > 0; o >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, o));
        hi = fmaxf(hi, __shfl_xor(hi, o));
    }
    __shared__ float2 wave[4];
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = make_float2(lo, hi);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; ++k) {
            lo = fminf(lo, wave[k].x);
            hi = fmaxf(hi, wave[k].y);
        }
        part[blockIdx.x] = make_float2(lo, hi);
    }
}

// Device scratch of the range: a few file-scope slots per GPU, so that a call
// allocates nothing (hipMalloc and hipFree were most of a small volume's call).
// A call owns its slot from acquire() to release(), after its stream is
// synchronised; when every slot is taken, or the GPU's index is beyond the
// table, it allocates its own.
constexpr int kRangeSlots = 8, kRangeDevices = 64;
__device__ float2 range_scratch[kRangeSlots][kRangeBlocks];

class RangeScratch {
  public:
    ~RangeScratch() { release(); }
    int acquire()
    {
        TKV_HIP(hipGetDevice(&dev_));
        if (dev_ >= 0 && dev_ < kRangeDevices) {
            std::lock_guard<std::mutex> lock(mu_);
            if (!base_[dev_]) {
                void *p = nullptr;
                TKV_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(range_scratch)));
                base_[dev_] = (float2 *)p;
            }
            for (int s = 0; s < kRangeSlots && base_[dev_]; ++s)
                if (!(taken_[dev_] & (1u << s))) {
                    taken_[dev_] |= 1u << s;
                    slot_ = s;
                    ptr = base_[dev_] + (size_t)s * kRangeBlocks;
                    return FDK_OK;
                }
        }
        TKV_HIP(hipMalloc((void **)&ptr, kRangeBlocks * sizeof(float2)));
        return FDK_OK;
    }
    float2 *ptr = nullptr;

  private:
    void release()
    {
        if (slot_ >= 0) {
            std::lock_guard<std::mutex> lock(mu_);
            taken_[dev_] &= ~(1u << slot_);
        } else if (ptr) {
            (void)hipFree(ptr);
        }
    }
    int dev_ = -1, slot_ = -1;
    static std::mutex mu_;
    static float2 *base_[kRangeDevices];
    static unsigned taken_[kRangeDevices];
};
std::mutex RangeScratch::mu_;
float2 *RangeScratch::base_[kRangeDevices] = {};
unsigned RangeScratch::taken_[kRangeDevices] = {};

// VEC: v is 16-byte and out 8-byte aligned; the body converts four values per
// step, the last n % 4 one by one
template <bool VEC>
__global__ void __launch_bounds__(256) to_u16_kernel(const float *v, size_t n, double vmin,
                                                     double vmax, uint16_t *out)
{
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nth = (size_t)gridDim.x * blockDim.x;
    size_t done = 0;
    if (VEC) {
        const float4 *v4 = reinterpret_cast<const float4 *>(v);
        uint2 *o4 = reinterpret_cast<uint2 *>(out);
        const size_t n4 = n / 4;
        for (size_t i = tid; i < n4; i += nth) {
            const float4 q = v4[i];
            const unsigned a = scale_u16(q.x, vmin, vmax), b = scale_u16(q.y, vmin, vmax);
            const unsigned c = scale_u16(q.z, vmin, vmax), d = scale_u16(q.w, vmin, vmax);
            o4[i] = make_uint2(a | (b << 16), c | (d << 16));
        }
        done = 4 * n4;
    }
    for (size_t i = done + tid; i < n; i += nth) out[i] = scale_u16(v[i], vmin, vmax);
}

unsigned grid_for(size_t n) { return (unsigned)std::min<size_t>((n + 255) / 256, 8192); }

}  // namespace

extern "C" int fdk_volume_minmax(const float *d_vol, size_t n, double *minmax, void *stream)
{
    if (!d_vol || !minmax || n == 0) return fail(FDK_ERR_INVALID_ARGUMENT, "minmax: empty input");
    hipStream_t st = (hipStream_t)stream;
    RangeScratch scratch;
    if (int rc = scratch.acquire()) return rc;
    // 16 values per thread at least
    const unsigned blocks = (unsigned)std::min<size_t>((n + 4095) / 4096, kRangeBlocks);
    if (((uintptr_t)d_vol & 15) == 0)
        hipLaunchKernelGGL(minmax_kernel<true>, dim3(blocks), dim3(256), 0, st, d_vol, n,
                           scratch.ptr);
    else
        hipLaunchKernelGGL(minmax_kernel<false>, dim3(blocks), dim3(256), 0, st, d_vol, n,
                           scratch.ptr);
    float2 part[kRangeBlocks];
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(part, scratch.ptr, blocks * sizeof(float2), hipMemcpyDeviceToHost, st);
    const hipError_t es = hipStreamSynchronize(st);   // also before the slot goes back
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) return tkv::hip_fail(e, "minmax");
    float lo = part[0].x, hi = part[0].y;
    for (unsigned k = 1; k < blocks; ++k) {   // -0 below +0, as in the kernel
        if (part[k].x < lo || (part[k].x == lo && std::signbit(part[k].x))) lo = part[k].x;
        if (part[k].y > hi || (part[k].y == hi && !std::signbit(part[k].y))) hi = part[k].y;
    }
    if (lo > hi) return fail(FDK_ERR_INVALID_ARGUMENT, "minmax: no value that is not NaN");
    minmax[0] = lo;
    minmax[1] = hi;
    return FDK_OK;
}

extern "C" int fdk_volume_to_u16(const float *d_vol, size_t n, double vmin, double vmax,
                                 uint16_t *d_out, void *stream)
{
    if (!d_vol || !d_out) return fail(FDK_ERR_INVALID_ARGUMENT, "to_u16: null buffer");
    if (n == 0) return FDK_OK;
    if (((uintptr_t)d_vol & 15) == 0 && ((uintptr_t)d_out & 7) == 0)
        hipLaunchKernelGGL(to_u16_kernel<true>, dim3(grid_for(n)), dim3(256), 0,
                           (hipStream_t)stream, d_vol, n, vmin, vmax, d_out);
    else
        hipLaunchKernelGGL(to_u16_kernel<false>, dim3(grid_for(n)), dim3(256), 0,
                           (hipStream_t)stream, d_vol, n, vmin, vmax, d_out);
    TKV_HIP(hipGetLastError());
    return FDK_OK;
}

extern "C" int fdk_tiff_export_device(const float *d_vol, int x, int y, int z, const char *dir,
                                      int first_index, double *minmax_out)
{
    if (!d_vol || x < 1 || y < 1 || z < 1)
        return fail(FDK_ERR_INVALID_ARGUMENT, "tiff export: empty volume");
    const size_t plane = (size_t)x * y;
    double mm[2];
    int rc = fdk_volume_minmax(d_vol, plane * z, mm, nullptr);
    if (rc) return rc;
    if (minmax_out) {
        minmax_out[0] = mm[0];
        minmax_out[1] = mm[1];
    }
    // slabs of about 64 MiB of 16-bit slices: slab k is written on a thread
    // while slab k+1 is converted and copied
    const int slab = (int)std::max<size_t>(1, std::min<size_t>(z, (64u << 20) / (2 * plane)));
    uint16_t *d_u16 = nullptr, *h_u16[2] = {nullptr, nullptr};
    hipError_t e = hipMalloc((void **)&d_u16, (size_t)slab * plane * 2);
    for (int i = 0; i < 2 && e == hipSuccess; ++i)
        e = hipHostMalloc((void **)&h_u16[i], (size_t)slab * plane * 2, hipHostMallocDefault);
    std::thread writer;
    int wrc = FDK_OK;
    std::string werr;
    auto join = [&]() {
        if (writer.joinable()) writer.join();
    };
    for (int z0 = 0; z0 < z && e == hipSuccess && !rc; z0 += slab) {
        const int nz = std::min(slab, z - z0);
        uint16_t *h = h_u16[(z0 / slab) & 1];
        rc = fdk_volume_to_u16(d_vol + (size_t)z0 * plane, (size_t)nz * plane, mm[0], mm[1], d_u16,
                               nullptr);
        if (rc) break;
        join();   // the buffer written two slabs ago is free again
        if (wrc) break;
        e = hipMemcpy(h, d_u16, (size_t)nz * plane * 2, hipMemcpyDeviceToHost);
        if (e != hipSuccess) break;
        auto write = [&, h, nz, z0]() {
            wrc = write_slices_parallel(nz, writer_threads(nz), werr, [&](int, int k) {
                return write_slices(h + (size_t)k * plane, x, y, 1, dir, first_index + z0 + k);
            });
        };
        try {
            writer = std::thread(write);
        } catch (const std::system_error &) {
            write();   // no thread available: write now
        }
    }
    join();
    (void)hipFree(d_u16);
    for (auto p : h_u16)
        if (p) (void)hipHostFree(p);
    if (rc) return rc;
    if (e != hipSuccess) return tkv::hip_fail(e, "tiff export");
    if (wrc) return fail(wrc, werr);
    return FDK_OK;
}
