"""Layers whose plan, schedules and quantised tokens come from one launch, against the oracle: the edges of the ids a thread keeps (12 and
32, 6144 and 16384 ids), one id more (two launches), the most experts and few, top-1 ids that are all the same, dropped ids, masks
that end inside a workgroup's tokens, both row lengths that have a kernel of their own, a wave of tokens that is not full."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, recorded_kernels
from test_gpu_fp8 import _check_layer, _layer_inputs, _u8
from test_gpu_fused import _check, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,K,I,active", [(1024, 1024, 8, 6, 512, None),     # 6144 ids
                                              (6145, 640, 3, 1, 512, None),
                                              (2048, 1024, 512, 8, 512, None),   # 16384
                                              (4096, 512, 16, 4, 512, 4090),
                                              (5462, 512, 8, 3, 512, None),      # 16386, two launches
                                              (701, 4224, 5, 2, 768, 333)])      # rows beyond 4096 columns
def test_layer_bit_exact(gpu, oracle, T, H, E, K, I, active):
    announce("whole plan T=%d H=%d E=%d K=%d I=%d active=%s" % (T, H, E, K, I, active))
    g = torch.Generator().manual_seed(T)
    ids = torch.rand(T, E, generator=g).topk(K, dim=1).indices
    if K == 1:
        ids[: T // 2] = 1   # the same for many
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=1)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=2)
    d = dict(x=synth.normal_bf16(T, H, seed=3), ids=ids, gates=torch.rand(T, K, generator=g), w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)
    mask = None if active is None else torch.arange(T) < active
    assert _check(oracle, d, *_run(gpu, d, mask=mask), n_active=active) == 0


def test_dropped_ids(gpu):
    """What a layer with dropped ids gives for a token is what it gives for it when the dropped ones name an expert at weight 0."""
    T, H, E, K, I = 1500, 1024, 12, 4, 1024
    announce("whole plan with dropped ids")
    g = torch.Generator().manual_seed(4)
    ids = torch.rand(T, E - 1, generator=g).topk(K, dim=1).indices
    gates = torch.rand(T, K, generator=g)
    drop = torch.rand(T, K, generator=g) < 0.3
    drop[7] = True
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=1)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=2)
    d = dict(x=synth.normal_bf16(T, H, seed=3), w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)
    out, etn = _run(gpu, dict(d, ids=torch.where(drop, -1, ids), gates=gates))
    want, want_etn = _run(gpu, dict(d, ids=torch.where(drop, E - 1, ids), gates=torch.where(drop, 0.0, gates)))
    assert torch.equal(out + 0.0, want + 0.0)   # (a zero's sign may differ)
    assert torch.equal(etn[: E - 1], want_etn[: E - 1]) and int(etn[E - 1]) == 0


@pytest.mark.parametrize("T,H,E,K,I", [(3000, 1024, 8, 2, 512), (1370, 4224, 6, 3, 512)])
def test_fp8_layer(gpu, oracle, T, H, E, K, I):
    announce("whole plan FP8 T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    ids, w, x, w1, s1, w2, s2 = _layer_inputs(T, H, E, K, I, seed=T)
    out, etn = cam.fused_deep_moe_fp8(x.to(gpu), ids.to(torch.int32).to(gpu), cam.prepack_weight(w1.to(gpu), True), s1.to(gpu),
                                      cam.prepack_weight(w2.to(gpu), False), s2.to(gpu), w.to(gpu))
    want, dbg = oracle.fp8_fused_layer(synth.bf16_bits(x), ids.numpy(), w.numpy(), _u8(w1), s1.numpy(), _u8(w2), s2.numpy(), debug=True)
    assert np.array_equal(etn.cpu().numpy(), dbg["cnt"])
    _check_layer(out.float().cpu().numpy(), want)


@pytest.mark.parametrize("T,launches", [(16384, 5), (16385, 6)])
def test_launches(gpu, T, launches):
    announce("whole plan launches T=%d" % T)
    E, H, I = 5, 512, 512
    dev = [[cam.prepack_weight(torch.empty(E, H, 2 * I, dtype=torch.int8, device=gpu), True)], [torch.empty(E, 2 * I, device=gpu)],
           [cam.prepack_weight(torch.empty(E, I, H, dtype=torch.int8, device=gpu), False)], [torch.empty(E, H, device=gpu)]]
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, 1, dtype=torch.int32, device=gpu)
    gates = torch.empty(T, 1, device=gpu)
    assert recorded_kernels(lambda: cam.fused_deep_moe(x, ids, *dev, gates, None, None, "", 1, 0, E, 1, 0, 0, 0)) == launches
