"""The permute on both sides of the output sizes from which its rows are stored plainly (16-bit rows 72 MiB, rows that are no whole lines
48, 8-bit rows of whole lines never): 16-bit, int8 and FP8 rows, rows under smooth scales, ids that name no expert.  Bit for bit, as
everywhere in the dispatch."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, recorded_names
from test_gpu_dispatch import _check_fused
import test_gpu_shmem

pytestmark = pytest.mark.gpu
K, E, H = 16, 300, 7168      # 659 tokens of 8-bit rows are 72 MiB, 330 of 16-bit rows


@pytest.mark.parametrize("T,quant_mode,H", [(658, 2, H), (659, 2, H), (659, 3, H), (1390, 2, H), (329, 0, H), (330, 0, H),
                                            (439, 2, 7160), (440, 2, 7160), (220, 0, 7160)])
def test_rows_around_the_lines(gpu, oracle, T, quant_mode, H):
    announce("permute stores T=%d H=%d quant=%d" % (T, H, quant_mode))
    rng = np.random.default_rng(T)
    ids = np.where(rng.random((T, K)) < 0.1, -1, rng.integers(0, E, size=(T, K))).astype(np.int64)
    x = synth.normal_bf16(T, H, seed=T)
    x[3] = 0
    d = cam.moe_dispatch_fused(x.to(gpu), torch.from_numpy(ids).to(gpu), E, quant_mode=quant_mode)
    _check_fused(oracle, d, x, ids, E, quant_mode)


def test_fp8_rows_between_the_lines(gpu, oracle):
    T = 659
    announce("permute stores T=%d fp8" % T)
    ids, _ = synth.sigmoid_zipf_routing(T, E, K, seed=3)
    x = synth.normal_bf16(T, H, seed=4)
    d = cam.moe_dispatch_fused(x.to(gpu), ids.to(torch.int32).to(gpu), E, quant_mode=4)
    q, sc = oracle.fp8_quant_rows(synth.bf16_bits(x))
    row = d["slot_row"].cpu().numpy()
    assert np.array_equal(d["recv_x"].view(torch.uint8).cpu().numpy()[row], np.broadcast_to(q[:, None], (T, K, H)))
    assert np.array_equal(d["recv_x_scales"].cpu().numpy()[row], np.broadcast_to(sc[:, None], (T, K, H // 128)))


def test_smooth_rows_between_the_lines(gpu, oracle):
    test_gpu_shmem.test_dispatch_shmem_bit_exact(gpu, oracle, 660, K, E, H, 2, True, False, 1)


@pytest.mark.parametrize("T,quant_mode,H,plainly", [(329, 0, H, False), (330, 0, H, True), (219, 0, 7160, False), (220, 0, 7160, True),
                                                    (439, 2, 7160, False), (440, 2, 7160, True), (659, 2, H, False), (1389, 2, H, False),
                                                    (3000, 2, H, False), (659, 4, H, False)])
def test_how_rows_are_stored(gpu, T, quant_mode, H, plainly):
    announce("permute how stored T=%d H=%d quant=%d" % (T, H, quant_mode))
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, dtype=torch.int32, device=gpu)
    permute = recorded_names(lambda: cam.moe_dispatch_fused(x, ids, E, quant_mode=quant_mode))[-1]
    form = {0: 0, 2: 1, 4: 3}[quant_mode]    # (rows copied, quantised to int8, to FP8)
    assert "dispatch_kernelILi%dELi0ELb%dEE" % (form, plainly) in permute
