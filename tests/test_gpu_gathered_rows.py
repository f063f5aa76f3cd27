"""Fused layers whose gate/up GEMM gathers its rows from the quantised tokens, against the oracle: one and several ranking
workgroups in front of it, tiles of every kind (tall, flat, narrow, partly filled, experts without rows), dropped ids, tokens
under a mask, scale rows that are whole words and that are not.  Tolerances are those of the ordinary layer tests: int8 bit
for bit, FP8 as test_gpu_fp8.py derives them."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, recorded_names
from test_gpu_fp8 import _check_layer, _layer_inputs, _u8
from test_gpu_fused import _check, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,K,I,active,drop", [
    (512, 1024, 2, 2, 2176, None, False),    # 1024 ids: one ranking workgroup
    (513, 1024, 3, 2, 2176, None, True),     # 1026: five
    (4099, 1024, 5, 1, 640, None, False),    # tall tiles, the last ones short
    (1500, 1152, 64, 4, 512, 1111, False),   # a mask, narrow tiles
    (2100, 1024, 300, 2, 512, None, True),   # flat tiles of a few rows
    (400, 7168, 2, 2, 3072, 1, False),       # one token of many
    (2049, 1024, 16, 2, 1152, None, False),  # over 256 rows per expert, and not
    (2048, 1024, 16, 2, 1152, None, False),
])
def test_int8_layer_bit_exact(gpu, oracle, T, H, E, K, I, active, drop):
    announce("gathered rows T=%d H=%d E=%d K=%d I=%d active=%s drop=%s" % (T, H, E, K, I, active, drop))
    ids, gates = synth.softmax_topk_routing(T, E, K, seed=T + I)
    if drop:
        ids[::5, 0] = -1
        ids[ids == 1] = 0 if K == 1 else -1   # an expert without rows
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=17)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=18)
    x = synth.normal_bf16(T, H, seed=19)
    x[T // 2] = 0
    d = dict(x=x, ids=ids, gates=gates, w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)
    mask = None if active is None else torch.arange(T) < active
    out, etn = _run(gpu, d, mask=mask)
    assert _check(oracle, d, out, etn, n_active=active) == 0


@pytest.mark.parametrize("T,H,E,K,I", [(1400, 1152, 8, 3, 1024),    # 9 scale bytes a row
                                       (1400, 2048, 8, 3, 1024),    # 16
                                       (2100, 1024, 40, 2, 1536)])
def test_fp8_layer(gpu, oracle, T, H, E, K, I):
    announce("gathered rows FP8 T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    ids, w, x, w1, s1, w2, s2 = _layer_inputs(T, H, E, K, I, seed=T + H)
    out, etn = cam.fused_deep_moe_fp8(x.to(gpu), ids.to(torch.int32).to(gpu), cam.prepack_weight(w1.to(gpu), True),
                                      s1.to(gpu), cam.prepack_weight(w2.to(gpu), False), s2.to(gpu), w.to(gpu))
    want, dbg = oracle.fp8_fused_layer(synth.bf16_bits(x), ids.numpy(), w.numpy(), _u8(w1), s1.numpy(), _u8(w2),
                                       s2.numpy(), debug=True)
    assert np.array_equal(etn.cpu().numpy(), dbg["cnt"])
    _check_layer(out.float().cpu().numpy(), want)


@pytest.mark.parametrize("T,E,K,plainly", [(8192, 32, 1, False), (8193, 32, 1, True), (4096, 64, 4, False), (4097, 64, 4, True)])
def test_how_quantised_tokens_are_stored(gpu, T, E, K, plainly):
    announce("quantised tokens T=%d E=%d K=%d" % (T, E, K))
    H, I = 1024, 1024
    w1, w2 = torch.empty(E, H, 2 * I, dtype=torch.int8, device=gpu), torch.empty(E, I, H, dtype=torch.int8, device=gpu)
    dev = [[cam.prepack_weight(w1, True)], [torch.empty(E, 2 * I, device=gpu)], [cam.prepack_weight(w2, False)],
           [torch.empty(E, H, device=gpu)]]
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, dtype=torch.int32, device=gpu)
    names = recorded_names(lambda: cam.fused_deep_moe(x, ids, *dev, torch.empty(T, K, device=gpu), None, None, "", 1, 0, E, 1, 0, 0, 0))
    assert "plan_quant_kernelILi8ELi2ELi0ELb%dEE" % plainly in names[0]
