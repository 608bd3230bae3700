// The engine's host code on the CPU: this program defines the HIP calls the library
// makes (memory from malloc, kernels only counted), so that an allocation can be
// refused when the test says so, and a call be seen to launch nothing.  `alloc_host
// MODE` prints one line per checked fact and returns 0 if all hold.
#include "tomokvas/fdk.h"

#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

namespace tkv {
double engine_bytes_per_sample(int storage, int Nu);   // fdk_host.cpp
}

namespace {
int launches = 0, allowed = -1, device = 0;   // allocations left (-1: any number)
std::map<void *, std::pair<size_t, int>> live;   // bytes and device of each allocation
}

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) { device = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    if (allowed == 0) return hipErrorOutOfMemory;
    if (allowed > 0) --allowed;
    *p = std::calloc(1, n);
    live[*p] = {n, device};
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)&launches; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)&launches; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
    ++launches;
    return hipSuccess;
}
}

namespace {
bool good = true;
void check(const char *what, bool ok)
{
    std::printf("%s: %s\n", ok ? "ok" : "FAILED", what);
    if (!ok) good = false;
}

size_t bytes()
{
    size_t n = 0;
    for (const auto &a : live) n += a.second.first;
    return n;
}

fdk_ctx *context(int gpu, int storage)
{
    fdk_ctx *c = nullptr;
    std::vector<float> sino(40 * 12 * 30, 1.f);
    if (fdk_create(gpu, &c) || fdk_set_sinogram_properties(c, sino.data(), 40, 19.5f, 12, 30, 14.5f, 0.5f, 200.f, 0.1f) ||
        fdk_set_reconstruction_properties(c, 24, 11.5f, 24, 11.5f, 16, 7.5f, 0.f) ||
        fdk_set_storage(c, storage) || fdk_initialize(c)) {
        std::printf("FAILED: %s\n", fdk_last_error_string());
        std::exit(1);
    }
    return c;
}
}

int main(int argc, char **argv)
{
    const std::string mode = argc > 1 ? argv[1] : "";
    if (mode == "stack") {
        // a larger stored stack can't be had: no reconstruction runs without one
        fdk_ctx *c = context(0, FDK_BF16);
        allowed = 0;
        check("storage refused", fdk_set_storage(c, FDK_F32) == FDK_ERR_OUT_OF_MEMORY);
        launches = 0;
        check("not initialized", fdk_calculate_reconstruction(c, nullptr, nullptr) == FDK_ERR_NOT_INITIALIZED);
        check("no launch", launches == 0);
        check("no projections", fdk_device_sinogram(c) == nullptr);
        allowed = -1;
        check("initialized again", fdk_initialize(c) == FDK_OK);
        check("reconstruction", fdk_calculate_reconstruction(c, nullptr, nullptr) == FDK_OK && launches > 0);
        fdk_destroy(c);
    } else if (mode == "filtered") {
        // the stack fits, the filtered projections don't: the old storage goes on
        fdk_ctx *c = context(0, FDK_F32);
        allowed = 0;
        check("storage refused", fdk_set_storage(c, FDK_F16) == FDK_ERR_OUT_OF_MEMORY);
        check("reconstruction in F32", fdk_calculate_reconstruction(c, nullptr, nullptr) == FDK_OK);
        allowed = -1;
        check("storage accepted", fdk_set_storage(c, FDK_F16) == FDK_OK);
        check("reconstruction in F16", fdk_calculate_reconstruction(c, nullptr, nullptr) == FDK_OK);
        fdk_destroy(c);
    } else if (mode == "device") {
        // another device is current when the storage grows
        fdk_ctx *c = context(1, FDK_BF16);
        (void)hipSetDevice(0);
        check("storage accepted", fdk_set_storage(c, FDK_F32) == FDK_OK);
        bool own = true;
        for (const auto &a : live) own = own && a.second.second == 1;
        check("every allocation on the context's device", own);
        fdk_destroy(c);
    } else if (mode == "overlap") {
        // fdk_filter_into: rows [Nv][nang][Nu] = [30][12][40] and stored stacks
        fdk_ctx *c = context(0, FDK_F32);
        const size_t n = 40 * 12 * 30;
        std::vector<float> buf(4 * n + fdk_stack_bytes(c, FDK_F32, 12) / 4 + 8);
        float *p = buf.data();
        while ((uintptr_t)p & 15) ++p;
        float scales[12];
        auto into = [&](const float *in, int in_nang, int nang, int store, void *out) {
            launches = 0;
            const int rc = fdk_filter_into(c, FDK_F32, in, in_nang, nang, store < 0 ? 0 : 1, 0, store, out,
                                           store < 0 ? nullptr : scales, nullptr, nullptr);
            return rc == FDK_OK && launches > 0 ? 1 : rc == FDK_ERR_INVALID_ARGUMENT && launches == 0 ? 0 : -1;
        };
        check("in place", into(p, 12, 12, -1, p) == 1);
        check("out of place, side by side", into(p, 12, 12, -1, p + n) == 1 && into(p + n, 12, 12, -1, p) == 1);
        check("one row further", into(p, 12, 12, -1, p + 40) == 0);
        check("one row before", into(p + 40, 12, 12, -1, p) == 0);
        check("the last sample", into(p, 12, 12, -1, p + n - 1) == 0 && into(p + n - 1, 12, 12, -1, p) == 0);
        // angles [4, 9) of 12: from row 4 of the first detector row to row 8 of the last
        const float *s = p + 4 * 40;
        check("a slice", into(s, 12, 5, -1, p + n) == 1);
        check("a slice onto its first sample", into(s, 12, 5, -1, (void *)s) == 0);
        check("a slice onto the gap before it", into(p + n, 12, 5, -1, p + n - 5 * 40 * 30) == 1);
        check("a slice onto its last sample", into(s, 12, 5, -1, p + n - 3 * 40 - 1) == 0);
        check("after a slice's last sample", into(s, 12, 5, -1, p + n - 3 * 40) == 1);
        // one angle of 45 in a stack of 30 x 45 rows; its 30 rows fit between two of its rows
        check("between a slice's rows", into(p, 45, 1, -1, p + 40) == 1 && into(p, 45, 1, -1, p + 15 * 40) == 1 &&
                                            into(p, 45, 1, -1, p + 15 * 40 + 1) == 0 &&
                                            into(p, 45, 1, -1, p + 39) == 0 &&
                                            into(p, 45, 1, -1, p + 3 * 45 * 40 + 40) == 1 &&
                                            into(p, 45, 1, -1, p + 29 * 45 * 40 + 39) == 0 &&
                                            into(p, 45, 1, -1, p + 29 * 45 * 40 + 40) == 1);
        check("into a stack", into(p, 12, 12, FDK_F32, p + n) == 1 && into(p, 12, 12, FDK_BF16, p + n) == 1);
        check("into a stack over the rows", into(p, 12, 12, FDK_F32, p) == 0 && into(p + 8, 12, 12, FDK_BF16, p) == 0);
        const size_t rows = fdk_stack_bytes(c, FDK_BF16, 12) - fdk_stack_bytes(c, FDK_BF16, 0);
        check("rows right after a stack", into(p + rows / 4, 12, 12, FDK_BF16, p) == 1 &&
                                              into(p + rows / 4 - 1, 12, 12, FDK_BF16, p) == 0);
        check("no angles", fdk_filter_into(c, FDK_F32, p, 12, 0, 0, 0, -1, p + 1, nullptr, nullptr, nullptr) == FDK_OK);
        fdk_destroy(c);
    } else if (mode == "budget") {
        // what the reconstruction program charges for a projection is what the engine
        // allocates for it (and for its angle's table entries)
        for (int storage : {FDK_F32, FDK_F16, FDK_BF16, FDK_F16_PACKED})
            for (int Nu : {40, 300, 1000}) {
                size_t held[2] = {0, 0};
                for (int i = 0; i < 2; ++i) {
                    fdk_ctx *c = context(0, storage);
                    const size_t before = bytes();
                    if (fdk_set_sinogram_properties(c, nullptr, Nu, 0.f, 40 << i, 64, 0.f, 0.1f, 2000.f, 0.1f) ||
                        fdk_initialize(c))
                        check("initialized", false);
                    held[i] = bytes();
                    check("grown", held[i] > before);
                    fdk_destroy(c);
                }
                const double per = (double)(held[1] - held[0]) / (40. * 64 * Nu);
                const double charged = tkv::engine_bytes_per_sample(storage, Nu);
                std::printf("storage %d Nu %d: %.4f bytes a sample, charged %.4f\n", storage, Nu, per, charged);
                check("charged", std::fabs(per - charged) <= 0.02 + 100. / (64 * Nu));
            }
    } else {
        std::printf("FAILED: unknown mode\n");
        return 2;
    }
    check("nothing left allocated", live.empty());
    return good ? 0 : 1;
}
