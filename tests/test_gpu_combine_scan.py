"""The combine on both sides of the row count up to which it finds its rows among the triples without a map (1024 rows and
slots) and of what its workgroups look through between them (5 x 2^20 triples): rows that name no slot, several that name the
same one (the last counts), rows past the receive total, more rows than slots, both activation types.  Bit for bit, as everywhere in the combine."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, recorded_kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,A,valid,H", [(1, 1, 1, 1, 1024), (1, 16, 1024, 1000, 7168), (64, 16, 1024, 1024, 1032),
                                           (1024, 1, 1023, 900, 1024), (128, 8, 1025, 1025, 2048), (129, 8, 1024, 1024, 2048),
                                           (7, 3, 21, 0, 1024), (1024, 1, 1024, 1000, 7168)])
@pytest.mark.parametrize("fp16", [False, True])
def test_rows_found_by_their_triples(gpu, oracle, T, K, A, valid, H, fp16):
    announce("combine scan T=%d K=%d A=%d valid=%d H=%d fp16=%d" % (T, K, A, valid, H, fp16))
    rng = np.random.default_rng(T + A)
    slots = np.concatenate([rng.permutation(T * K), np.zeros(max(A - T * K, 0), np.int64)])[:A]
    src = np.stack([np.zeros(A, np.int64), slots // K, slots % K], axis=1).astype(np.int32)
    src[rng.random(A) < 0.1, 1] = T          # no such token
    src[rng.random(A) < 0.1, 2] = -1         # no such slot
    if A <= 1024 and T * K <= 1024 and T * -(-H // 1024) * A <= 5 << 20 and A > 8:
        src[A // 2] = src[A // 4]            # (with a map it is either of them)
    elif A > T * K:
        src[T * K:, 1] = -1
    if valid > 8:
        src[valid - 1] = (0, T - 1, K - 1)   # the last row that counts ...
        src[:valid - 1][(src[:valid - 1, 1] == T - 1) & (src[:valid - 1, 2] == K - 1), 1] = -1
    y = synth.normal_bf16(A, H, seed=T)
    y = y.half() if fp16 else y
    w = torch.rand(T, K, generator=torch.Generator().manual_seed(A))
    row_of = oracle.rows_from_src_info(np.ascontiguousarray(src[:valid].reshape(-1)), valid, T, K)
    want = oracle.combine_act(y.view(torch.int16).numpy().view(np.uint16), row_of, w.numpy(), fp16)
    counts = torch.tensor([0, valid], dtype=torch.int32, device=gpu)
    got = cam.moe_combine_normal(y.to(gpu), torch.from_numpy(src.reshape(-1)).to(gpu), counts, w.to(gpu))
    assert_bits_equal(got.view(torch.int16).cpu().numpy().view(np.uint16), want, "combined x")


@pytest.mark.parametrize("T,K,A,H,launches", [(1024, 1, 1024, 5120, 1), (1024, 1, 1024, 5128, 2), (865, 1, 865, 7168, 1),
                                              (866, 1, 866, 7168, 2), (128, 8, 1025, 1024, 2), (129, 8, 1024, 1024, 2)])
def test_launches(gpu, T, K, A, H, launches):
    announce("combine launches T=%d K=%d A=%d H=%d" % (T, K, A, H))
    y, w = torch.empty(A, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, device=gpu)
    src, counts = torch.empty(3 * A, dtype=torch.int32, device=gpu), torch.empty(2, dtype=torch.int32, device=gpu)
    assert recorded_kernels(lambda: cam.moe_combine_normal(y, src, counts, w)) == launches
