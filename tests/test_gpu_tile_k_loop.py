"""The K loop of the tile GEMM at its edges: every number of row fragments of both tile shapes (the last with one row, or one
short of full), K of fewer 128-byte stages than the ring, odd and even numbers of them, column blocks of which the last is
ragged."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, to_np

pytestmark = pytest.mark.gpu

FLAT = [1, 31, 32, 33, 64, 65, 96, 97, 127, 128]
TALL = [129, 160, 161, 191, 193, 224, 225, 256, 257, 300]


@pytest.mark.parametrize("Kd", [128, 256, 384, 512, 640, 1152])
@pytest.mark.parametrize("name,sizes,N,gate_up", [("flat", FLAT, 9 * 64, False), ("tall", TALL, 9 * 64, False),
                                                  ("flat", FLAT, 11 * 128, True), ("tall", TALL, 5 * 128, True)])
def test_int32_sums_bit_exact(gpu, oracle, name, sizes, N, gate_up, Kd):
    announce("tile form, K loop: %s tiles, K=%d N=%d gate_up=%s" % (name, Kd, N, gate_up))
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    x = synth.uniform_int8((sum(sizes), Kd), Kd)   # no row behind the last tile's
    w = synth.uniform_int8((len(sizes), Kd, N), Kd + N)
    got = cam.grouped_matmul_int32(x.to(gpu), cam.prepack_weight(w.to(gpu), gate_up), gl.to(gpu))
    assert_bits_equal(to_np(got), oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy()), "int32 sums")


@pytest.mark.parametrize("Kd", [128, 256, 384, 1024])
@pytest.mark.parametrize("sizes", [FLAT, TALL])
def test_fp8_sums(gpu, oracle, sizes, Kd):
    """Tolerance as in test_gpu_fp8.py: the matrix core aligns the 64 products of an instruction before it adds them."""
    N = 640
    announce("tile form, fp8 K loop: sizes=%s K=%d" % (sizes[:3], Kd))
    gen = torch.Generator().manual_seed(Kd)
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    x = torch.randn(sum(sizes), Kd, generator=gen).mul_(2).to(torch.float8_e4m3fn)
    w = torch.randn(len(sizes), Kd, N, generator=gen).to(torch.float8_e4m3fn)
    xs = torch.randint(121, 130, (sum(sizes), Kd // 128), generator=gen, dtype=torch.uint8)
    ws = torch.randint(121, 130, (len(sizes), Kd // 128, N // 128), generator=gen, dtype=torch.uint8)
    got = cam.grouped_matmul_fp8(x.to(gpu), xs.to(gpu), cam.prepack_weight(w.to(gpu), False), ws.to(gpu), gl.to(gpu),
                                 out_dtype=torch.float32).cpu().numpy()
    want = oracle.fp8_gemm(x.view(torch.uint8).numpy(), xs.numpy(), w.view(torch.uint8).numpy(), ws.numpy(), gl.numpy())
    assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 2e-4 * np.abs(want).max()).all(), float(np.abs(got - want).max())
