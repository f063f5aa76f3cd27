"""Layers whose second GEMM quantises the SwiGLU products in tiles cut out of its 128-row form, against the oracle: the most rows such a
tile takes (16 at I 2048, 32 at 1024, 64 at 512) and one more token (a launch of its own), tokens that name an expert more than
once (several tiles to an expert), masked tokens."""
import pytest
import torch

from umdk_original_amd import synth
import umdk_original_amd as cam
from gpu_util import announce, recorded_kernels
from test_gpu_fused import _check, _run

pytestmark = pytest.mark.gpu


def _layer(T, H, E, K, I, ids):
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=1)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=2)
    x = synth.normal_bf16(T, H, seed=3)
    x[T // 2] = 0
    return dict(x=x, ids=ids, gates=torch.rand(T, K, generator=torch.Generator().manual_seed(T)), w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)


@pytest.mark.parametrize("T,H,E,K,I,active,repeated", [
    (16, 6144, 16, 8, 2048, None, False),
    (16, 6144, 16, 8, 2048, None, True),    # 128 rows to an expert, eight tiles
    (9, 7040, 14, 4, 1920, 5, False),
    (32, 7168, 14, 4, 1024, None, False),
    (31, 6272, 16, 6, 1024, 17, True),
    (64, 6144, 16, 2, 512, None, False)])
def test_layer_bit_exact(gpu, oracle, T, H, E, K, I, active, repeated):
    announce("tall products T=%d H=%d E=%d K=%d I=%d active=%s repeated=%d" % (T, H, E, K, I, active, repeated))
    g = torch.Generator().manual_seed(T)
    ids = torch.rand(T, E, generator=g).topk(K, dim=1).indices
    if repeated:
        ids[:, :] = ids[:, :1] % 3
    d = _layer(T, H, E, K, I, ids)
    mask = None if active is None else torch.arange(T) < active
    assert _check(oracle, d, *_run(gpu, d, mask=mask), n_active=active) == 0


@pytest.mark.parametrize("T,H,E,I,launches", [(16, 6144, 16, 2048, 4), (17, 6144, 16, 2048, 5), (16, 6144, 15, 2048, 5), (32, 7168, 14, 1024, 4),
                                              (33, 7168, 14, 1024, 5), (16, 7168, 18, 2048, 4), (16, 7168, 19, 2048, 5)])
def test_launches(gpu, T, H, E, I, launches):
    announce("tall products, launches T=%d H=%d E=%d I=%d" % (T, H, E, I))
    K = 4
    dev = [[cam.prepack_weight(torch.empty(E, H, 2 * I, dtype=torch.int8, device=gpu), True)], [torch.empty(E, 2 * I, device=gpu)],
           [cam.prepack_weight(torch.empty(E, I, H, dtype=torch.int8, device=gpu), False)], [torch.empty(E, H, device=gpu)]]
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, dtype=torch.int32, device=gpu)
    gates = torch.empty(T, K, device=gpu)
    assert recorded_kernels(lambda: cam.fused_deep_moe(x, ids, *dev, gates, None, None, "", 1, 0, E, 1, 0, 0, 0)) == launches
