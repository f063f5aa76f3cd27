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

#include <algorithm>
#include <optional>
#include <string>
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

// ---- what both libraries call an operator with.  `Host` is the library's side of it: how a tensor is checked and viewed
// (view), how an output is allocated (empty), and how a status becomes an error (check, of an operator; fail).

template <class Host>
struct ListView {  // a list argument; keeps the structs alive
    std::vector<camTensor> items;
    std::vector<const camTensor *> ptrs;
    camTensorList list{};
    ListView(at::TensorList ts, int32_t format)
    {
        items.reserve(ts.size());
        ptrs.reserve(ts.size());
        for (const at::Tensor &t : ts) {
            items.push_back(Host::view(t, format));
            ptrs.push_back(&items.back());
        }
        list.tensors = ptrs.data();
        list.count = ptrs.size();
    }
};

template <class Host>
struct OptionalView {  // an optional argument: NULL when it is None
    camTensor c{};
    const camTensor *p = nullptr;
    explicit OptionalView(const std::optional<at::Tensor> &t)
    {
        if (t.has_value() && t->defined()) {
            c = Host::view(*t, CAM_FORMAT_ND);
            p = &c;
        }
    }
};

// -> {output, expertTokenNums}
template <class Host>
std::vector<at::Tensor> fused_deep_moe(const at::Tensor &x, const at::Tensor &ids, at::TensorList w1, at::TensorList w1s,
                                       at::TensorList w2, at::TensorList w2s, const at::Tensor &gates,
                                       const std::optional<at::Tensor> &smooth, const std::optional<at::Tensor> &mask,
                                       std::string group, int64_t rank_size, int64_t rank_id, int64_t experts,
                                       int64_t shared_num, int64_t shared_rank_num, int64_t quant_mode, int64_t global_bs)
{
    const int64_t local = rank_id < shared_rank_num ? 1 : experts / std::max<int64_t>(rank_size - shared_rank_num, 1);
    at::Tensor out = Host::empty({x.size(0), x.size(1)}, x.scalar_type(), x), etn = Host::empty({local}, at::kLong, x);
    camTensor cx = Host::view(x, CAM_FORMAT_ND), ci = Host::view(ids, CAM_FORMAT_ND), cg = Host::view(gates, CAM_FORMAT_ND),
              co = Host::view(out, CAM_FORMAT_ND), ce = Host::view(etn, CAM_FORMAT_ND);
    ListView<Host> l1(w1, CAM_FORMAT_MFMA_B), l1s(w1s, CAM_FORMAT_ND), l2(w2, CAM_FORMAT_MFMA_B), l2s(w2s, CAM_FORMAT_ND);
    OptionalView<Host> os(smooth), om(mask);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    Host::check(camFusedDeepMoeGetWorkspaceSize(&cx, &ci, &l1.list, &l1s.list, &l2.list, &l2s.list, &cg, os.p, om.p,
                                                group.data(), rank_size, rank_id, experts, shared_num, shared_rank_num,
                                                quant_mode, global_bs, &co, &ce, &bytes, &ex), "camFusedDeepMoe");
    Host::check(launch(camFusedDeepMoe, bytes, ex, x), "camFusedDeepMoe");
    return {out, etn};
}

struct PrefillRows {
    at::Tensor rows, scales, info, recv_count;  // for at most `rows` rows; scales only where they are asked for
    at::Tensor counts;                          // per expert, on the CPU
};

// MoeDispatchPrefill with the counts per expert on the host.  wait is called with what waits for them.
template <class Host, class Wait>
PrefillRows dispatch_prefill(const at::Tensor &x, const at::Tensor &ids, int64_t experts, int64_t quant_mode, int64_t rows,
                             int64_t rank, int64_t ranks, bool with_scales, const Wait &wait)
{
    const int64_t T = x.size(0), H = x.size(1), K = ids.size(1), A = std::max<int64_t>(rows, 1);
    camTensor cx = Host::view(x, CAM_FORMAT_ND), ci = Host::view(ids, CAM_FORMAT_ND);
    const bool fp8 = quant_mode == 4;  // E4M3 rows, one E8M0 scale per row and 128 columns
    PrefillRows r;
    r.rows = Host::empty({A, H}, fp8 ? at::kFloat8_e4m3fn : quant_mode != 0 ? at::kChar : x.scalar_type(), x);
    r.info = Host::empty({3 * A}, at::kInt, x);
    r.recv_count = Host::empty({experts}, at::kInt, x);
    at::Tensor pos = Host::empty({T, K}, at::kInt, x);
    camTensor crx = Host::view(r.rows, CAM_FORMAT_ND), cidx = Host::view(r.info, CAM_FORMAT_ND), crs{},
              crc = Host::view(r.recv_count, CAM_FORMAT_ND), cpos = Host::view(pos, CAM_FORMAT_ND);
    if (with_scales) {
        r.scales = fp8 ? Host::empty({A, H / 128}, at::kByte, x) : Host::empty({A}, at::kFloat, x);
        crs = Host::view(r.scales, CAM_FORMAT_ND);
    }
    const int64_t per_rank = experts / std::max<int64_t>(ranks, 1);
    if (per_rank < 1 || per_rank > HostCounts::kMost) {
        Host::fail(CAM_ERR_RANGE, "numExperts " + std::to_string(experts) + " outside (0, 512]");
    }
    r.counts = at::empty({per_rank}, at::TensorOptions().dtype(at::kLong));
    HostCounts host(per_rank, x.get_device());
    camTensor cpe{};  // the counts per expert, in host memory the plan kernel stores to
    cpe.data = host.data();
    cpe.dtype = CAM_DT_INT64;
    cpe.ndim = 1;
    cpe.sizes[0] = per_rank;
    cpe.strides[0] = 1;
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    Host::check(camMoeDispatchPrefillGetWorkspaceSize(&cx, &ci, experts, ranks, rank, quant_mode, &crx,
                                                      with_scales ? &crs : nullptr, &cidx, &cpos, nullptr, nullptr, nullptr,
                                                      &crc, &cpe, nullptr, &bytes, &ex), "camMoeDispatchPrefill");
    host.queued();
    Host::check(launch(camMoeDispatchPrefill, bytes, ex, x), "camMoeDispatchPrefill");
    wait([&] { host.wait(stream_of(x), r.counts.template data_ptr<int64_t>()); });
    return r;
}

}  // namespace cam_torch

#endif  // CAM_TORCH_UTIL_H_
