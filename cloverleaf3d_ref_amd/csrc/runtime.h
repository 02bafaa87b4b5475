// Internal runtime helpers shared by the drop-in ABI and the resident driver:
// error propagation across the C boundary and host<->device copies between
// dense Fortran arrays and the device layout.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>

#include "kernels.h"
#include "layout.h"

namespace clover {

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

enum : int {
    E_HIP = -1,     // a HIP runtime call failed
    E_ARG = -2,     // invalid argument (shape, class, pointer)
    E_STATE = -3,   // library not initialised / wrong state
    E_NOMEM = -4,   // device allocation failed
};

void set_last_error(const std::string &msg);

inline void hip_check(hipError_t e, const char *what)
{
    if (e != hipSuccess)
        throw Error(e == hipErrorOutOfMemory ? E_NOMEM : E_HIP,
                    std::string(what) + ": " + hipGetErrorString(e));
}

// CUs of a device: 256 on a whole MI355X, fewer of a partition
inline int cu_count(int device)
{
    int cus = 0;
    hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device), "CU count");
    return cus;
}

// Waits for the dt tagged seq, which a launch_dt_final on the stream is bound to
// deliver: if the stream ends or fails without it, so does the wait.  Polling
// pinned memory saves the copy back and the wake-up of a stream synchronisation.
// Past the first polls, some 20 us, the core is offered to other threads between
// them: those of other chunks or processes may need it to get their own work to
// the GPU.
inline double wait_dt(const DtSlot *slot, unsigned long long seq, hipStream_t st)
{
    for (long spins = 0;; spins++) {
        if (__atomic_load_n(&slot->seq, __ATOMIC_ACQUIRE) == seq) return slot->dtlp;
        if (spins < 1000) __builtin_ia32_pause();
        else std::this_thread::yield();
        if (spins % 100000 == 99999) {
            const hipError_t e = hipStreamQuery(st);
            if (e == hipErrorNotReady) continue;
            hip_check(e, "calc_dt");
            if (__atomic_load_n(&slot->seq, __ATOMIC_ACQUIRE) == seq) return slot->dtlp;
            throw Error(E_HIP, "calc_dt: the stream ended without a dt");
        }
    }
}

#define CLOVER_API_BEGIN try {
#define CLOVER_API_END                                    \
    return 0;                                             \
    }                                                     \
    catch (const clover::Error &e) {                      \
        clover::set_last_error(e.what());                 \
        return e.code;                                    \
    }                                                     \
    catch (const std::exception &e) {                     \
        clover::set_last_error(e.what());                 \
        return clover::E_ARG;                             \
    }

// Moves 3-D fields between the device layout g and dense Fortran arrays of
// class `cls` on the host, through two pinned buffers that its owner keeps
// (at most kPieceElems doubles each; allocated on first use, freed by the
// owner's release()).  Every piece is enqueued on the stream, after what is
// there.  Threads may fetch fields of one owner at the same time: one transfer
// has the buffers at a time.
class Stage {
  public:
    Stage() = default;
    Stage(const Stage &) = delete;
    Stage &operator=(const Stage &) = delete;
    // dev holds es-byte elements (8 or 4); returns when host is filled
    void download(const Lay &g, int cls, const void *dev, size_t es, double *host, hipStream_t st);
    // returns when host has been read; the device copy follows on the stream
    void upload(const Lay &g, int cls, const double *host, double *dev, hipStream_t st);
    // waits for the kernels that use the buffers and frees them; not a
    // destructor's work, since an owner of static lifetime may outlive the
    // device runtime
    void release();

  private:
    struct Buf {
        double *host = nullptr, *dev = nullptr;  // one pinned allocation, seen from both sides
        hipEvent_t done = nullptr;               // the kernel that uses it last
        bool busy = false;
    };
    static constexpr int64_t kPieceElems = 512 * 1024;  // 4 MiB
    void reserve(int64_t total, hipStream_t st);
    void wait(Buf &b);
    std::mutex mu_;
    Buf buf_[2];
    int64_t elems_ = 0;  // doubles per buffer
    int next_ = 0;       // upload's next buffer
};

// element count of the dense host array of class cls
int64_t dense_elems(const Lay &g, int cls);

// the current device's address of the allocation-free entry point's fixed
// scratch array (looked up on first use per device)
double *noalloc_scratch();

}  // namespace clover
