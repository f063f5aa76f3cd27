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
#include "host_counts.h"

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

// The current stream of the device `like` lives on.
inline hipStream_t stream_of(const at::Tensor &like)
{
    return c10::hip::getCurrentHIPStream(like.device().index()).stream();
}

typedef camStatus (*Phase2)(void *, uint64_t, camOpExecutor *, camStream_t);

// Phase 2 of an operator whose phase 1 has produced (bytes, executor): the workspace, the stream and the launches
// belong to the device `like` lives on.
inline camStatus launch(Phase2 fn, uint64_t bytes, camOpExecutor *executor, const at::Tensor &like)
{
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(like.device());
    at::Tensor ws;
    if (bytes > 0) {
        try {
            ws = new_empty({(int64_t)bytes}, at::kByte, like);
        } catch (...) {  // out of memory: phase 2, which frees the executor, will not run
            camDestroyExecutor(executor);
            throw;
        }
    }
    return fn(bytes > 0 ? ws.data_ptr() : nullptr, bytes, executor, (camStream_t)stream_of(like));
}

}  // namespace cam_torch

#endif  // CAM_TORCH_UTIL_H_
