// The Python module behind ops.py: the operators of this package that are not torch.ops of the reference, from
// arguments to launches in C++.  Through ctypes (_lib.call) an operator with eleven output tensors took 44 us of host
// time, five times what its kernels take on a small batch; here it takes about a third.  Errors are the CamError of
// _lib.py, as there.
#include <torch/csrc/utils/pybind.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include "torch_util.h"

namespace py = pybind11;

namespace {

[[noreturn]] void fail(int status, const char *message)
{
    const py::object cls = py::module_::import("umdk_original_amd._lib").attr("CamError");
    const py::object err = cls(status, message);
    PyErr_SetObject(cls.ptr(), err.ptr());
    throw py::error_already_set();
}

void check(camStatus st)
{
    if (st != CAM_OK) {
        fail((int)st, camGetRecentErrMsg());
    }
}

// An output beside `like`.  Where that is in host memory nothing is launched, but phase 1 has its say first.
at::Tensor new_empty(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor &like)
{
    return like.is_cuda() ? cam_torch::new_empty(sizes, dtype, like) : at::empty(sizes, at::TensorOptions().dtype(dtype));
}

// Phase 2 of an operator whose first input is `like`.
void run(cam_torch::Phase2 fn, uint64_t bytes, camOpExecutor *executor, const at::Tensor &like)
{
    if (!like.is_cuda()) {
        camDestroyExecutor(executor);
        fail(CAM_ERR_WORKSPACE, "no device to allocate the workspace on");
    }
    check(cam_torch::launch(fn, bytes, executor, like));
}

camTensor to_cam(const at::Tensor &t, int32_t format = CAM_FORMAT_ND)
{
    const int32_t dtype = cam_torch::cam_dtype(t.scalar_type());
    if (dtype < 0) {
        fail(CAM_ERR_DTYPE, (std::string("torch dtype ") + c10::toString(t.scalar_type()) + " has no CAM code").c_str());
    }
    if (t.dim() > CAM_MAX_DIMS) {
        fail(CAM_ERR_SHAPE, "too many dimensions");
    }
    return cam_torch::view_of(t, dtype, format);
}

// This library's side of what torch_util.h shares (an operator's name is not part of a CamError).
struct Host {
    static camTensor view(const at::Tensor &t, int32_t format) { return to_cam(t, format); }
    static at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor &like)
    {
        return new_empty(sizes, dtype, like);
    }
    static void check(camStatus st, const char *) { ::check(st); }
    static void fail(int status, const std::string &message) { ::fail(status, message.c_str()); }
};
typedef cam_torch::ListView<Host> List;
typedef cam_torch::OptionalView<Host> Optional;

// Fresh outputs, by name, as the operators of ops.py return them.
py::dict moe_dispatch_fused(const at::Tensor &x, const at::Tensor &ids, int64_t experts, int64_t quant_mode, int64_t rows,
                            int64_t rank, int64_t ranks)
{
    const int64_t T = x.size(0), H = x.size(1), K = ids.size(1), A = std::max<int64_t>(rows < 0 ? T * K : rows, 1);
    camTensor cx = to_cam(x), ci = to_cam(ids);
    const bool fp8 = quant_mode == 4;  // E4M3 rows, one E8M0 scale per row and 128 columns
    at::Tensor rx = new_empty({A, H}, fp8 ? at::kFloat8_e4m3fn : quant_mode != 0 ? at::kChar : x.scalar_type(), x);
    at::Tensor rs = fp8 ? new_empty({A, H / 128}, at::kByte, x) : new_empty({A}, at::kFloat, x);
    at::Tensor idx = new_empty({3 * A}, at::kInt, x), pos = new_empty({T, K}, at::kInt, x);
    at::Tensor slot = new_empty({T, K}, at::kInt, x), cnt = new_empty({experts}, at::kInt, x);
    at::Tensor off = new_empty({experts}, at::kInt, x), rc = new_empty({experts}, at::kInt, x);
    at::Tensor tpe = new_empty({experts / std::max<int64_t>(ranks, 1)}, at::kLong, x), total = new_empty({1}, at::kLong, x);
    camTensor crx = to_cam(rx), crs = to_cam(rs), cidx = to_cam(idx), cpos = to_cam(pos), cslot = to_cam(slot), ccnt = to_cam(cnt),
              coff = to_cam(off), crc = to_cam(rc), ctpe = to_cam(tpe), ctotal = to_cam(total);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    check(camMoeDispatchPrefillGetWorkspaceSize(&cx, &ci, experts, ranks, rank, quant_mode, &crx, &crs, &cidx, &cpos, &cslot,
                                                &ccnt, &coff, &crc, &ctpe, &ctotal, &bytes, &ex));
    run(camMoeDispatchPrefill, bytes, ex, x);
    py::dict d;
    d["recv_x"] = rx;
    d["recv_x_scales"] = rs;
    d["expand_idx"] = idx;
    d["send_token_idx"] = pos;
    d["slot_row"] = slot;
    d["num_tokens_per_expert"] = cnt;
    d["send_offset"] = off;
    d["recv_count"] = rc;
    d["num_recv_tokens_per_expert"] = tpe;
    d["total"] = total;
    return d;
}

// -> (recv_x, recv_x_scales, expand_idx, recv_count, counts per expert on the CPU)
py::tuple moe_dispatch_prefill(const at::Tensor &x, const at::Tensor &ids, int64_t experts, int64_t quant_mode, int64_t rows,
                               int64_t rank, int64_t ranks)
{
    const cam_torch::PrefillRows r = cam_torch::dispatch_prefill<Host>(
        x, ids, experts, quant_mode, rows < 0 ? x.size(0) * ids.size(1) : rows, rank, ranks, true, [](const auto &wait) {
            py::gil_scoped_release nogil;
            wait();
        });
    return py::make_tuple(r.rows, r.scales, r.info, r.recv_count, r.counts);
}

void moe_combine_gather(const at::Tensor &rows, const std::optional<at::Tensor> &info, const at::Tensor &slot_row,
                        const std::optional<at::Tensor> &counts, const at::Tensor &weights,
                        const std::optional<at::Tensor> &shared, const at::Tensor &out)
{
    camTensor cr = to_cam(rows), cs = to_cam(slot_row), cw = to_cam(weights), co = to_cam(out);
    Optional oi(info), oc(counts), os(shared);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    check(camMoeCombineGatherGetWorkspaceSize(&cr, oi.p, &cs, oc.p, &cw, os.p, &co, &bytes, &ex));
    run(camMoeCombineGather, bytes, ex, rows);
}

py::tuple grouped_matmul_swiglu_quant(const at::Tensor &x, const at::Tensor &x_scale, const std::vector<at::Tensor> &w,
                                      const std::vector<at::Tensor> &ws, const at::Tensor &group_list, int64_t type)
{
    const int64_t A = x.size(0), I = w.at(0).size(-1) / 2;
    at::Tensor y = new_empty({A, I}, at::kChar, x), ys = new_empty({A}, at::kFloat, x);
    camTensor cx = to_cam(x), cs = to_cam(x_scale), cg = to_cam(group_list), cy = to_cam(y), cys = to_cam(ys);
    List lw(w, CAM_FORMAT_MFMA_B), ls(ws, CAM_FORMAT_ND);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    check(camGroupedMatmulSwigluQuantGetWorkspaceSize(&cx, &cs, &lw.list, &ls.list, &cg, type, &cy, &cys, &bytes, &ex));
    run(camGroupedMatmulSwigluQuant, bytes, ex, x);
    return py::make_tuple(y, ys);
}

void grouped_matmul_dequant(const at::Tensor &x, const at::Tensor &x_scale, const std::vector<at::Tensor> &w,
                            const std::vector<at::Tensor> &ws, const at::Tensor &group_list, int64_t type, const at::Tensor &out)
{
    camTensor cx = to_cam(x), cs = to_cam(x_scale), cg = to_cam(group_list), co = to_cam(out);
    List lw(w, CAM_FORMAT_MFMA_B), ls(ws, CAM_FORMAT_ND);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    check(camGroupedMatmulDequantGetWorkspaceSize(&cx, &cs, &lw.list, &ls.list, &cg, type, &co, &bytes, &ex));
    run(camGroupedMatmulDequant, bytes, ex, x);
}

void grouped_matmul_fp8(const at::Tensor &x, const at::Tensor &x_scale, const at::Tensor &w, const at::Tensor &ws, bool gate_up,
                        const at::Tensor &group_list, int64_t type, const at::Tensor &out,
                        const std::optional<at::Tensor> &out_scale)
{
    camTensor cx = to_cam(x), cs = to_cam(x_scale), cw = to_cam(w, CAM_FORMAT_MFMA_B), cws = to_cam(ws), cg = to_cam(group_list),
              co = to_cam(out);
    Optional oo(out_scale);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    check(camGroupedMatmulFp8GetWorkspaceSize(&cx, &cs, &cw, &cws, gate_up ? 1 : 0, &cg, type, &co, oo.p, &bytes, &ex));
    run(camGroupedMatmulFp8, bytes, ex, x);
}

py::list fused_deep_moe_fp8(const at::Tensor &x, const at::Tensor &ids, const at::Tensor &w1, const at::Tensor &w1s,
                            const at::Tensor &w2, const at::Tensor &w2s, const at::Tensor &gates,
                            const std::optional<at::Tensor> &mask, int64_t experts)
{
    at::Tensor out = new_empty({x.size(0), x.size(1)}, at::kBFloat16, x), etn = new_empty({experts}, at::kLong, x);
    camTensor cx = to_cam(x), ci = to_cam(ids), c1 = to_cam(w1, CAM_FORMAT_MFMA_B), c1s = to_cam(w1s),
              c2 = to_cam(w2, CAM_FORMAT_MFMA_B), c2s = to_cam(w2s), cg = to_cam(gates), co = to_cam(out), ce = to_cam(etn);
    Optional om(mask);
    uint64_t bytes = 0;
    camOpExecutor *ex = nullptr;
    check(camFusedDeepMoeFp8GetWorkspaceSize(&cx, &ci, &c1, &c1s, &c2, &c2s, &cg, om.p, experts, &co, &ce, &bytes, &ex));
    run(camFusedDeepMoeFp8, bytes, ex, x);
    py::list l;
    l.append(out);
    l.append(etn);
    return l;
}

py::list fused_deep_moe(const at::Tensor &x, const at::Tensor &ids, const std::vector<at::Tensor> &w1,
                        const std::vector<at::Tensor> &w1s, const std::vector<at::Tensor> &w2,
                        const std::vector<at::Tensor> &w2s, const at::Tensor &gates, const std::optional<at::Tensor> &smooth,
                        const std::optional<at::Tensor> &mask, std::string group, int64_t rank_size, int64_t rank_id,
                        int64_t experts, int64_t shared_num, int64_t shared_rank_num, int64_t quant_mode, int64_t global_bs)
{
    py::list l;
    for (const at::Tensor &t : cam_torch::fused_deep_moe<Host>(x, ids, w1, w1s, w2, w2s, gates, smooth, mask, std::move(group),
                                                               rank_size, rank_id, experts, shared_num, shared_rank_num,
                                                               quant_mode, global_bs)) {
        l.append(t);
    }
    return l;
}

}  // namespace

PYBIND11_MODULE(_cam_native, m)
{
    // which build of the library this module calls: the address of one of its functions
    m.def("library", [] { return (uintptr_t)&camGetVersion; });
    m.def("moe_dispatch_fused", &moe_dispatch_fused);
    m.def("moe_dispatch_prefill", &moe_dispatch_prefill);
    m.def("moe_combine_gather", &moe_combine_gather);
    m.def("grouped_matmul_swiglu_quant", &grouped_matmul_swiglu_quant);
    m.def("grouped_matmul_dequant", &grouped_matmul_dequant);
    m.def("grouped_matmul_fp8", &grouped_matmul_fp8);
    m.def("fused_deep_moe_fp8", &fused_deep_moe_fp8);
    m.def("fused_deep_moe", &fused_deep_moe);
}
