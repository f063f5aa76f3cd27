"""The dispatch layout on both sides of the lines between one workgroup alone and several (256 and 1024 tokens, 8192 flags, what the tokens
beyond 256 may all name); dropped, repeated and out-of-range ids, both id types."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from gpu_util import announce, assert_bits_equal, recorded_kernels, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E,R", [(256, 16, 512, 32), (256, 2, 33, 33), (257, 16, 512, 1), (1023, 8, 64, 1), (1024, 8, 512, 8),
                                     (1024, 3, 9, 9), (1025, 8, 64, 1), (300, 1, 1, 1), (1024, 1, 64, 1), (512, 4, 64, 1), (320, 16, 512, 1),
                                     (307, 10, 64, 16)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_layout_of_one_workgroup(gpu, oracle, T, K, E, R, dtype):
    announce("layout alone T=%d K=%d E=%d R=%d %s" % (T, K, E, R, dtype))
    ids = np.random.default_rng(T + E).integers(-1, E + 1, size=(T, K)).astype(np.int64)
    got = cam.get_dispatch_layout(torch.from_numpy(ids).to(dtype).to(gpu), E, R)
    want = oracle.layout(ids, E, R, skip_out_of_range=True)
    for name, g, w in zip(("per rank", "per expert", "in rank"), got, want):
        assert_bits_equal(to_np(g).astype(np.int32), w.astype(np.int32), name)


@pytest.mark.parametrize("T,K,E,R,launches", [(256, 16, 64, 32, 1), (320, 16, 512, 1, 1), (321, 16, 512, 1, 2), (512, 4, 64, 1, 1),
                                              (513, 4, 64, 1, 2), (1024, 1, 64, 1, 1), (1024, 1, 64, 8, 2), (1024, 8, 256, 1, 2),
                                              (307, 10, 64, 16, 1), (308, 10, 64, 16, 2), (257, 11, 64, 16, 2), (512, 2, 34, 17, 2)])
def test_launches(gpu, T, K, E, R, launches):
    announce("layout launches T=%d K=%d E=%d R=%d" % (T, K, E, R))
    ids = torch.empty(T, K, dtype=torch.int32, device=gpu)
    assert recorded_kernels(lambda: cam.get_dispatch_layout(ids, E, R)) == launches
