// What the two torch-facing libraries share: torch.ops registration (torch_binding.cpp) and the Python module behind
// ops.py (py_native.cpp).  Tensors become camTensor structs, phase 1 says how large the workspace is, the workspace comes
// from torch's caching allocator and phase 2 enqueues on the current stream of the tensors' device.
#ifndef CAM_TORCH_UTIL_H_
#define CAM_TORCH_UTIL_H_

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <vector>

#include "../../include/cam_mi355x.h"

namespace cam_torch {

// The CAM code of a torch dtype, or -1.
inline int32_t cam_dtype(at::ScalarType t)
{
    switch (t) {
        case at::kFloat: return CAM_DT_FLOAT;
        case at::kHalf: return CAM_DT_FLOAT16;
        case at::kChar: return CAM_DT_INT8;
        case at::kInt: return CAM_DT_INT32;
        case at::kByte: return CAM_DT_UINT8;
        case at::kLong: return CAM_DT_INT64;
        case at::kBool: return CAM_DT_BOOL;
        case at::kBFloat16: return CAM_DT_BF16;
        case at::kFloat8_e4m3fn: return CAM_DT_FLOAT8_E4M3FN;
        default: return -1;
    }
}

inline camTensor view_of(const at::Tensor &t, int32_t dtype, int32_t format)
{
    camTensor c{};
    c.data = t.data_ptr();
    c.dtype = dtype;
    c.ndim = (int32_t)t.dim();
    for (int64_t d = 0; d < t.dim(); ++d) {
        c.sizes[d] = t.size(d);
        c.strides[d] = t.stride(d);
    }
    c.format = format;
    return c;
}

// A contiguous uninitialised tensor on `like`'s device, without the round through the dispatcher.
inline at::Tensor new_empty(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor &like)
{
    return at::Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}

typedef camStatus (*Phase2)(void *, uint64_t, camOpExecutor *, camStream_t);

// Phase 2 of an operator whose phase 1 has produced (bytes, executor): the workspace, the stream and the launches
// belong to the device `like` lives on.
inline camStatus launch(Phase2 fn, uint64_t bytes, camOpExecutor *executor, const at::Tensor &like)
{
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(like.device());
    at::Tensor ws;
    if (bytes > 0) {
        ws = new_empty({(int64_t)bytes}, at::kByte, like);
    }
    return fn(bytes > 0 ? ws.data_ptr() : nullptr, bytes, executor,
              (camStream_t)c10::hip::getCurrentHIPStream(like.device().index()).stream());
}

// The rows an operator's plan counts per expert, brought to the host without a copy and without waiting for anything
// behind the plan: the kernel stores the counts into host memory and the host watches them arrive.  (Two blocking
// copies after the permute took about 20 us of a call, and held the host until the rows had moved.)  One buffer per
// thread, given back with it; a call is over when its counts are complete, so a thread needs no second one.
class HostCounts {
public:
    static constexpr int64_t kMost = 512;  // experts an operator admits

    // Memory for n counts, none of which has arrived.
    static int64_t *begin(int64_t n)
    {
        HostCounts &b = of_thread();
        if (b.p_ == nullptr) {
            TORCH_CHECK(hipHostMalloc((void **)&b.p_, kMost * sizeof(int64_t), hipHostMallocCoherent) == hipSuccess,
                        "out of pinned host memory");
        }
        TORCH_CHECK(n <= kMost, "too many experts");
        for (int64_t i = 0; i < n; ++i) {
            b.p_[i] = -1;
        }
        return b.p_;
    }

    // Waits for all of them.  The stream is asked now and then: once it has nothing left to run, or an error, the wait
    // ends either way.
    static at::Tensor wait(int64_t n, const at::Tensor &like)
    {
        volatile int64_t *p = of_thread().p_;
        const hipStream_t stream = c10::hip::getCurrentHIPStream(like.device().index()).stream();
        int64_t i = 0;
        for (unsigned spin = 1; i < n; ++spin) {
            while (i < n && p[i] >= 0) {
                ++i;
            }
            if (i < n && (spin & 0xffff) == 0) {
                const hipError_t e = hipStreamQuery(stream);
                TORCH_CHECK(e == hipSuccess || e == hipErrorNotReady, "moe_dispatch_prefill: ", hipGetErrorString(e));
                if (e == hipSuccess) {  // the kernels are done, so whatever they stored is there
                    for (; i < n; ++i) {
                        TORCH_CHECK(p[i] >= 0, "moe_dispatch_prefill: the counts did not arrive");
                    }
                }
            }
        }
        at::Tensor out = at::empty({n}, at::TensorOptions().dtype(at::kLong));
        int64_t *dst = out.data_ptr<int64_t>();
        for (i = 0; i < n; ++i) {
            dst[i] = p[i];
        }
        return out;
    }

private:
    static HostCounts &of_thread()
    {
        static thread_local HostCounts b;
        return b;
    }
    ~HostCounts()
    {
        if (p_ != nullptr) {
            (void)hipHostFree(p_);
        }
    }
    int64_t *p_ = nullptr;
};

}  // namespace cam_torch

#endif  // CAM_TORCH_UTIL_H_
