"""Calls that ask for derivatives the operators do not have are refused, whichever way they ask: tangents (forward mode)
on any input, and calls inside a functorch transform, also where none of the call's own inputs is wrapped."""
import pytest
import torch
from torch.autograd import forward_ad

from umdk_original_amd import synth
from gpu_util import announce

pytestmark = pytest.mark.gpu

OPS = torch.ops.umdk_cam_op_lib
T, K, E, H, I = 16, 2, 8, 1024, 512


@pytest.fixture(scope="module")
def calls(gpu):
    """name -> (operator, floating-point inputs by position (a list: the tensors of a list argument), all arguments)."""
    ids, gates = synth.softmax_topk_routing(T, E, K, seed=1)
    ids, gates = ids.to(torch.int32).to(gpu), gates.to(gpu)
    x = synth.normal_bf16(T, H, seed=2).to(gpu)
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=3)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=4)
    w1, w2 = OPS.prepack_weight(w1.to(gpu), True), OPS.prepack_weight(w2.to(gpu), False)
    per_rank, per_expert, in_rank = OPS.get_dispatch_layout(ids, E, 1)
    prefill = [x, ids, gates, per_rank, in_rank, per_expert, 0, "", 0, 1]
    rows, info, counts, _ = OPS.moe_dispatch_prefill(*prefill)
    smooth = torch.rand(E, H, device=gpu) + 0.5
    shmem = [x, ids, smooth, None, 1, 0, E, 1, 0, 0, 1, 0, 2, 0, 1, 0]
    d = OPS.moe_dispatch_shmem(*shmem)
    y = synth.normal_bf16(T * K, H, seed=5).to(gpu)
    return dict(
        fused=(OPS.fused_deep_moe, [0, 3, 6], [x, ids, [w1], [w1s.to(gpu)], [w2], [w2s.to(gpu)], gates, None, None, "", 1, 0,
                                               E, 1, 0, 0, 0]),
        layout=(OPS.get_dispatch_layout, [], [ids, E, 1]),
        prefill=(OPS.moe_dispatch_prefill, [0, 2], prefill),
        combine=(OPS.moe_combine_prefill, [0, 2], [rows, ids, gates, info, counts, "", 0, 1]),
        dispatch_shmem=(OPS.moe_dispatch_shmem, [0, 2], shmem),
        combine_shmem=(OPS.moe_combine_shmem, [0, 4], [y, ids, d[2], d[4], gates, None, None, None, None, None, None, 1, 0, E,
                                                       1, 0, 0, 1, 0, 0, 0, 0, 0, 0]),
    )


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("name", ["fused", "prefill", "combine", "dispatch_shmem", "combine_shmem"])
def test_tangents_are_refused(calls, name, grad):
    op, floats, args = calls[name]
    announce("tangents into %s, gradients %s" % (name, grad))
    with torch.set_grad_enabled(grad):
        for i in floats:
            with forward_ad.dual_level():
                dual = list(args)
                if isinstance(args[i], list):
                    dual[i] = [forward_ad.make_dual(t, torch.ones_like(t)) for t in args[i]]
                else:
                    dual[i] = forward_ad.make_dual(args[i], torch.ones_like(args[i]))
                with pytest.raises(RuntimeError, match="jvp is not implemented"):
                    op(*dual)
        op(*args)   # without a tangent the same call is accepted


@pytest.mark.parametrize("name", ["fused", "layout", "prefill", "combine", "dispatch_shmem", "combine_shmem"])
def test_calls_inside_a_functorch_transform_are_refused(gpu, calls, name):
    op, _, args = calls[name]
    announce("%s inside torch.func.grad" % name)

    def f(z):
        op(*args)
        return z.sum()

    with pytest.raises(RuntimeError, match="functorch transform"):
        torch.func.grad(f)(torch.ones(3, device=gpu))
    op(*args)   # and accepted again behind it
