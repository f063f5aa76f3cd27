"""The fused layer where its second GEMM quantises the SwiGLU products itself, against the oracle: around the limits of
that form (32768 products a tile, rows rounded up to a power of two), one and several threads, waves and row tiles per
row, an intermediate size that is no multiple of a turn of the waves, masked tokens."""
import pytest
import torch

from umdk_original_amd import synth
from gpu_util import announce
from test_gpu_fused import _check, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,K,I,active", [
    (1, 1024, 16, 1, 3072, None),    # one row, all 512 threads on it
    (1, 4096, 32, 8, 1536, None),    # a tile could have 8 rows
    (3, 1024, 8, 1, 640, None),      # rows no power of two; K no multiple of a turn
    (5, 1024, 4, 2, 2048, None),     # 16 rows x 2048: the most products a tile may have
    (5, 1024, 4, 2, 2176, None),     # 16 x 2176: too many
    (64, 1024, 2, 1, 1024, None),    # 32 rows x 1024 and more than one tile per expert
    (33, 1024, 2, 2, 896, None),     # 33 rows: a tile of one row behind a full one
    (32, 1024, 2, 1, 1152, None),    # 32 x 1152: too many
    (60, 1024, 4, 2, 512, 41),       # masked tokens
])
def test_layer_of_few_rows_bit_exact(gpu, oracle, T, H, E, K, I, active):
    announce("few rows T=%d H=%d E=%d K=%d I=%d active=%s" % (T, H, E, K, I, active))
    ids, gates = synth.softmax_topk_routing(T, E, K, seed=T + I)
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=7)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=8)
    x = synth.normal_bf16(T, H, seed=9)
    x[T // 2] = 0  # a row of zero products
    d = dict(x=x, ids=ids, gates=gates, w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)
    mask = None if active is None else torch.arange(T) < active
    out, etn = _run(gpu, d, mask=mask)
    assert _check(oracle, d, out, etn, n_active=active) == 0
