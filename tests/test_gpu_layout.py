"""The dispatch layout at the edges of its workgroups (256 tokens, then 64 workgroups of them) and of its limits, with
dropped, repeated and out-of-range ids, for both id types."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from gpu_util import announce, assert_bits_equal, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E,R", [(1, 16, 512, 1), (255, 3, 384, 384), (256, 8, 64, 8), (257, 8, 64, 1),
                                     (513, 1, 7, 7), (8449, 2, 510, 255), (16384, 1, 9, 3), (16385, 2, 12, 2)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_layout_counts(gpu, oracle, T, K, E, R, dtype):
    announce("layout edges T=%d K=%d E=%d R=%d %s" % (T, K, E, R, dtype))
    rng = np.random.default_rng(T + E)
    ids = rng.integers(-1, E + 1, size=(T, K)).astype(np.int64)
    got = cam.get_dispatch_layout(torch.from_numpy(ids).to(dtype).to(gpu), E, R)
    want = oracle.layout(ids, E, R, skip_out_of_range=True)
    for name, g, w in zip(("per rank", "per expert", "in rank"), got, want):
        assert_bits_equal(to_np(g).astype(np.int32), w.astype(np.int32), name)
