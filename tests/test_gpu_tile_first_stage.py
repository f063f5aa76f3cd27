"""The tile form of the grouped GEMM where a K loop is hardly longer than its ring of stages, so that the first refill of a
stage follows its first use at once: many launches over operands that lie in the caches, each against the first, and
that against the oracle.  (The first refill once did not wait for the other team's first fragments; a wave that was late
with them multiplied the weights of a later step, which showed in one of many runs of the long-schedule test.)"""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Kd", [128, 256, 320 + 64])
@pytest.mark.parametrize("name,sizes", [
    ("tall", [256, 200, 129, 512, 700, 1100, 161, 300, 257, 900, 256, 256]),
    ("flat", [128, 97, 33, 1, 64, 128] * 16),
    ("both", [1000, 128, 300, 40, 600, 100, 150, 7] * 3),
])
def test_repeated_launches_bit_exact(gpu, oracle, name, sizes, Kd):
    N, launches = 1024, 40
    announce("tile form, %d launches of %s tiles, K=%d" % (launches, name, Kd))
    A = sum(sizes)
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    x, w = synth.uniform_int8((A, Kd), Kd), synth.uniform_int8((len(sizes), Kd, N), Kd + 1)
    xd, wp, gld = x.to(gpu), cam.prepack_weight(w.to(gpu), False), gl.to(gpu)
    first = cam.grouped_matmul_int32(xd, wp, gld)
    differ = [i for i in range(launches) if not torch.equal(cam.grouped_matmul_int32(xd, wp, gld), first)]
    assert_bits_equal(to_np(first), oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy()), "int32 accumulators")
    assert not differ, "launches %s differ from the first" % differ
