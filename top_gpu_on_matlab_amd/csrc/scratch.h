// Working memory lent for one call.
#pragma once

#include <memory>
#include <mutex>
#include <vector>

#include "tg_internal.h"

namespace tg {

// Working memory of the calls that have no object of their own (reductions, the OC update, the scatter entries' checks): device scratch and a
// few pinned values that the last kernel writes and then publishes, so a call neither allocates (hipMalloc,
// hipHostMalloc and their frees took 0.2 to 0.4 ms a call) nor copies.  Blocks are lent for one call, each to one
// caller at a time, and come back once the host has seen the result, when nothing of theirs runs any more; at
// most SCRATCH_KEPT idle ones per device are kept, the rest are freed.
constexpr size_t SCRATCH_DOUBLES = 17 * 1024;
constexpr size_t SCRATCH_KEPT = 4;
struct ScratchBlock {
    DevBuf<double> dev{SCRATCH_DOUBLES};
    double *host = nullptr, *mapped = nullptr;  // 16 doubles, then the published number; their device address
    unsigned long long seq = 0;
    ScratchBlock() {
        TG_HIP(hipHostMalloc((void **)&host, 17 * sizeof(double), hipHostMallocMapped | hipHostMallocCoherent), "topgpu:alloc");
        *(unsigned long long *)(host + 16) = 0ull;
        if (hipHostGetDevicePointer((void **)&mapped, host, 0) != hipSuccess) {
            (void)hipHostFree(host);
            fail(TG_ERR_HIP, "topgpu:alloc", "pinned memory is not mapped");
        }
    }
    ~ScratchBlock() { (void)hipHostFree(host); }
};
struct ScratchPool {
    std::mutex mu;
    std::vector<std::unique_ptr<ScratchBlock>> idle[64];
};
inline ScratchPool &scratch_pool() {
    static ScratchPool *p = new ScratchPool;  // not destroyed: the runtime may be gone before it at exit
    return *p;
}
class Scratch {
    hipStream_t st;
    int dev = 0;
    std::unique_ptr<ScratchBlock> b;
    bool busy = false;  // work may be in flight that the host has not seen the end of

  public:
    explicit Scratch(hipStream_t s) : st(s) {
        TG_HIP(hipGetDevice(&dev), "topgpu:alloc");
        if (dev < 0 || dev >= 64) fail(TG_ERR_HIP, "topgpu:alloc", "device ordinal %d out of range", dev);
        {
            ScratchPool &p = scratch_pool();
            std::lock_guard<std::mutex> lock(p.mu);
            p.idle[dev].reserve(SCRATCH_KEPT);  // so that giving a block back, in a destructor, allocates nothing
            if (!p.idle[dev].empty()) {
                b = std::move(p.idle[dev].back());
                p.idle[dev].pop_back();
            }
        }
        if (!b) b.reset(new ScratchBlock);
        busy = true;
    }
    ~Scratch() {
        if (busy) (void)hipStreamSynchronize(st);
        ScratchPool &p = scratch_pool();
        std::lock_guard<std::mutex> lock(p.mu);
        if (p.idle[dev].size() < SCRATCH_KEPT) p.idle[dev].push_back(std::move(b));
    }
    double *dbl() const { return b->dev.p; }
    double *host() const { return b->mapped; }                                              // device address
    unsigned long long *seq_ptr() const { return (unsigned long long *)(b->mapped + 16); }  // device address
    unsigned long long next() {
        busy = true;
        return ++b->seq;
    }
    // The values once the last kernel has published them.  The stream is queried now and then, so a device
    // error, or a stream that finished without publishing, ends the wait.
    const double *wait(const char *id) {
        unsigned long long *hs = (unsigned long long *)(b->host + 16);
        for (unsigned spins = 1; __atomic_load_n(hs, __ATOMIC_ACQUIRE) != b->seq; ++spins)
            if ((spins & 4095) == 0) {
                const hipError_t e = hipStreamQuery(st);
                if (e != hipErrorNotReady) {
                    TG_HIP(e, id);
                    if (__atomic_load_n(hs, __ATOMIC_ACQUIRE) != b->seq) fail(TG_ERR_HIP, id, "result not published by a finished stream");
                }
            }
        busy = false;
        return b->host;
    }
};

}  // namespace tg
