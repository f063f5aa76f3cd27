// The rows an operator's plan counts per expert, brought to the host without a copy and without waiting for anything
// behind the plan: the kernel stores the counts into host memory and the host watches them arrive.  (Two blocking
// copies after the permute took about 20 us of a call, and held the host until the rows had moved.)
//
// One buffer per thread, given back with it, whichever devices the thread works on: it is allocated with the first
// call's device current and is portable, i.e. mapped for every device.  A call is over when its counts are complete, so a
// thread needs no second one, unless a call ends by an error after its kernels were queued: these may yet store, so
// that buffer is left to them (4 KB a failed call) and the next call takes a new one.
#ifndef CAM_HOST_COUNTS_H_
#define CAM_HOST_COUNTS_H_

#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <stdexcept>
#include <string>

namespace cam_torch {

class HostCounts {
public:
    static constexpr int64_t kMost = 512;  // experts an operator admits

    // Memory for the n counts of one call on `device`, none of which has arrived.
    HostCounts(int64_t n, int device) : n_(n)
    {
        if (n < 0 || n > kMost) {
            throw std::runtime_error("too many experts");
        }
        Buffer &b = of_thread();
        if (b.p == nullptr) {
            int current = device;
            bool ok = hipGetDevice(&current) == hipSuccess && (current == device || hipSetDevice(device) == hipSuccess);
            void *p = nullptr;
            ok = ok && hipHostMalloc(&p, kMost * sizeof(int64_t), hipHostMallocCoherent | hipHostMallocPortable) == hipSuccess;
            if (current != device) {
                (void)hipSetDevice(current);
            }
            if (!ok) {
                throw std::runtime_error("out of pinned host memory");
            }
            b.p = (int64_t *)p;
        }
        for (int64_t i = 0; i < n; ++i) {
            b.p[i] = -1;
        }
    }
    HostCounts(const HostCounts &) = delete;
    HostCounts &operator=(const HostCounts &) = delete;
    ~HostCounts()
    {
        if (queued_) {
            of_thread().p = nullptr;
        }
    }

    int64_t *data() { return of_thread().p; }

    // From here on a kernel may store to the buffer.
    void queued() { queued_ = true; }

    // Waits for all counts and copies them to out.  The stream is asked now and then: once it has nothing left to run, or
    // an error, the wait ends either way.
    void wait(hipStream_t stream, int64_t *out)
    {
        volatile int64_t *p = of_thread().p;
        int64_t i = 0;
        for (unsigned spin = 1; i < n_; ++spin) {
            while (i < n_ && p[i] >= 0) {
                ++i;
            }
            if (i < n_ && (spin & 0xffff) == 0) {
                const hipError_t e = hipStreamQuery(stream);
                if (e != hipSuccess && e != hipErrorNotReady) {
                    throw std::runtime_error(std::string("moe_dispatch_prefill: ") + hipGetErrorString(e));
                }
                if (e == hipSuccess) {  // the kernels are done, so whatever they stored is there
                    for (; i < n_; ++i) {
                        if (p[i] < 0) {
                            throw std::runtime_error("moe_dispatch_prefill: the counts did not arrive");
                        }
                    }
                }
            }
        }
        queued_ = false;
        for (i = 0; i < n_; ++i) {
            out[i] = p[i];
        }
    }

private:
    struct Buffer {
        int64_t *p = nullptr;
        ~Buffer()
        {
            if (p != nullptr) {
                (void)hipHostFree(p);
            }
        }
    };
    static Buffer &of_thread()
    {
        static thread_local Buffer b;
        return b;
    }
    int64_t n_;
    bool queued_ = false;
};

}  // namespace cam_torch

#endif  // CAM_HOST_COUNTS_H_
