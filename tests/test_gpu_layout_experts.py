"""The dispatch layout in one launch, a workgroup per expert and per rank: the edges of the ids a thread keeps (4, 8, 12, 16) and of its
range (16384 ids, 131072 flags, one more), ranks of one expert, ids that name none (64-bit ones whose lower half does among them), tokens
that all name the same experts or none.  All results are whole numbers."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from gpu_util import announce, assert_bits_equal, recorded_kernels, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E,R", [(1, 1, 1, 1), (63, 5, 512, 1), (256, 16, 384, 384), (1025, 3, 64, 1), (4096, 1, 7, 7),
                                     (4097, 1, 8, 2), (1170, 7, 512, 64), (1171, 7, 512, 64), (2048, 6, 60, 4), (2049, 6, 64, 1),
                                     (16384, 1, 2, 1), (16384, 1, 8, 8), (16385, 1, 9, 9), (2048, 8, 64, 64), (1638, 10, 130, 65)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("spread", ["any", "same", "none"])
def test_layout_of_a_workgroup_per_expert(gpu, oracle, T, K, E, R, dtype, spread):
    announce("layout per expert T=%d K=%d E=%d R=%d %s %s" % (T, K, E, R, dtype, spread))
    rng = np.random.default_rng(T + E)
    ids = np.tile(rng.integers(0, E, size=(1, K)), (T, 1)) if spread == "same" else rng.integers(0, E, size=(T, K))
    drop = rng.random((T, K)) < (1.0 if spread == "none" else 0.1)
    ids = np.where(drop, rng.choice([-1, E, 1 << 20], size=(T, K)), ids).astype(np.int64)
    given = ids.copy()
    if dtype == torch.int64:
        given[ids < 0] = 1 << 32    # no expert either, though its lower half is one's id
    got = cam.get_dispatch_layout(torch.from_numpy(given).to(dtype).to(gpu), E, R)
    want = oracle.layout(np.where((ids >= 0) & (ids < E), ids, -1), E, R, skip_out_of_range=True)
    for name, g, w in zip(("per rank", "per expert", "in rank"), got, want):
        assert_bits_equal(to_np(g).astype(np.int32), w.astype(np.int32), name)


@pytest.mark.parametrize("T,K,E,R,launches", [(1025, 8, 256, 1, 1), (16384, 1, 8, 8, 1), (16385, 1, 8, 1, 2), (2048, 8, 64, 64, 1),
                                              (2049, 7, 64, 64, 2)])
def test_launches(gpu, T, K, E, R, launches):
    announce("layout launches T=%d K=%d E=%d R=%d" % (T, K, E, R))
    ids = torch.empty(T, K, dtype=torch.int32, device=gpu)
    assert recorded_kernels(lambda: cam.get_dispatch_layout(ids, E, R)) == launches
