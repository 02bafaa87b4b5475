// Field transfers between the device layout and the dense Fortran arrays of
// the host (runtime.h Stage).
//
// A field's rows are padded on the device and dense on the host, so a plain
// copy goes row by row: 6.8 us per row whatever its length (a 64^3 field 33 ms,
// a 512^3 field 2 s: 0.5 GB/s).  Here a kernel gathers (or scatters) a piece of
// the dense array straight between the device and pinned host memory, and the
// CPU copies the pieces to or from the caller's pageable array while the next
// piece is under way.  The kernel's time is the link's; the CPU copy bounds
// the whole.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "runtime.h"

namespace clover {

constexpr int kPackThreads = 256;

// element q of the dense array (extents ex, ey, ...) in the device layout
__device__ inline int lay_of_dense(const Lay &g, int ex, int ey, int q)
{
    const int row = q / ex, x = q - row * ex;
    const int z = row / ey, y = row - z * ey;
    return g.base + x + g.ld * y + g.plane * z;
}

// dense elements first..first+n-1 of `dev`, as doubles (the FP32-store form's
// values widen exactly)
template <typename S>
__global__ void __launch_bounds__(kPackThreads)
k_pack(Lay g, int ex, int ey, int first, int n, const S *__restrict__ dev, double *__restrict__ out)
{
    for (int q = (int)(blockIdx.x * kPackThreads + threadIdx.x); q < n; q += (int)gridDim.x * kPackThreads)
        out[q] = (double)dev[lay_of_dense(g, ex, ey, first + q)];
}

__global__ void __launch_bounds__(kPackThreads)
k_unpack(Lay g, int ex, int ey, int first, int n, const double *__restrict__ in, double *__restrict__ dev)
{
    for (int q = (int)(blockIdx.x * kPackThreads + threadIdx.x); q < n; q += (int)gridDim.x * kPackThreads)
        dev[lay_of_dense(g, ex, ey, first + q)] = in[q];
}

void Stage::release()
{
    for (Buf &b : buf_) {
        if (b.busy) (void)hipEventSynchronize(b.done);
        if (b.done) (void)hipEventDestroy(b.done);
        if (b.host) (void)hipHostFree(b.host);
        b = Buf{};
    }
    elems_ = 0;
}

// The stream's device as the calling thread's current one, as long as this lives
struct DeviceScope {
    int before = 0;
    explicit DeviceScope(hipStream_t st)
    {
        int device = 0;
        hip_check(hipGetDevice(&before), "hipGetDevice");
        hip_check(hipStreamGetDevice(st, &device), "hipStreamGetDevice");
        hip_check(hipSetDevice(device), "hipSetDevice");
    }
    ~DeviceScope() { (void)hipSetDevice(before); }
};

// Room for pieces of a field of `total` elements.  The buffers and events are
// the stream's device's, whichever is current: an event of another one cannot be
// recorded on it, and a caller may fetch from chunks on several devices.
void Stage::reserve(int64_t total, hipStream_t st)
{
    const int64_t want = std::min(total, kPieceElems);
    if (want <= elems_) return;
    release();
    const DeviceScope device(st);
    for (Buf &b : buf_) {
        hip_check(hipHostMalloc((void **)&b.host, sizeof(double) * (size_t)want, hipHostMallocDefault), "hipHostMalloc");
        hip_check(hipHostGetDevicePointer((void **)&b.dev, b.host, 0), "hipHostGetDevicePointer");
        hip_check(hipEventCreateWithFlags(&b.done, hipEventDisableTiming), "hipEventCreate");
    }
    elems_ = want;
}

void Stage::wait(Buf &b)
{
    if (!b.busy) return;
    hip_check(hipEventSynchronize(b.done), "hipEventSynchronize");
    b.busy = false;
}

static dim3 pack_grid(int n) { return dim3((unsigned)std::min((n + kPackThreads - 1) / kPackThreads, 4096)); }

void Stage::download(const Lay &g, int cls, const void *dev, size_t es, double *host, hipStream_t st)
{
    std::lock_guard<std::mutex> lock(mu_);
    int ex, ey, ez;
    class_extents(cls, g.x_max - g.x_min + 1, g.y_max - g.y_min + 1, g.z_max - g.z_min + 1, ex, ey, ez);
    const int64_t total = (int64_t)ex * ey * ez;
    reserve(total, st);
    const int64_t pieces = (total + elems_ - 1) / elems_;
    auto len = [&](int64_t p) { return (int)std::min(elems_, total - p * elems_); };
    auto start = [&](int64_t p) {
        Buf &b = buf_[p & 1];
        wait(b);
        const int n = len(p), first = (int)(p * elems_);
        if (es == sizeof(float))
            hipLaunchKernelGGL(k_pack<float>, pack_grid(n), dim3(kPackThreads), 0, st, g, ex, ey, first, n,
                               static_cast<const float *>(dev), b.dev);
        else
            hipLaunchKernelGGL(k_pack<double>, pack_grid(n), dim3(kPackThreads), 0, st, g, ex, ey, first, n,
                               static_cast<const double *>(dev), b.dev);
        hip_check(hipGetLastError(), "pack");
        hip_check(hipEventRecord(b.done, st), "hipEventRecord");
        b.busy = true;
    };
    for (int64_t p = 0; p < std::min<int64_t>(pieces, 2); p++) start(p);
    for (int64_t p = 0; p < pieces; p++) {
        Buf &b = buf_[p & 1];
        wait(b);
        memcpy(host + p * elems_, b.host, sizeof(double) * (size_t)len(p));
        if (p + 2 < pieces) start(p + 2);
    }
}

void Stage::upload(const Lay &g, int cls, const double *host, double *dev, hipStream_t st)
{
    std::lock_guard<std::mutex> lock(mu_);
    int ex, ey, ez;
    class_extents(cls, g.x_max - g.x_min + 1, g.y_max - g.y_min + 1, g.z_max - g.z_min + 1, ex, ey, ez);
    const int64_t total = (int64_t)ex * ey * ez;
    reserve(total, st);
    const int64_t pieces = (total + elems_ - 1) / elems_;
    for (int64_t p = 0; p < pieces; p++) {
        Buf &b = buf_[next_];
        next_ ^= 1;
        wait(b);  // the kernel that reads its last piece
        const int n = (int)std::min(elems_, total - p * elems_);
        memcpy(b.host, host + p * elems_, sizeof(double) * (size_t)n);
        hipLaunchKernelGGL(k_unpack, pack_grid(n), dim3(kPackThreads), 0, st, g, ex, ey, (int)(p * elems_), n, b.dev,
                           dev);
        hip_check(hipGetLastError(), "unpack");
        hip_check(hipEventRecord(b.done, st), "hipEventRecord");
        b.busy = true;
    }
}

}  // namespace clover
