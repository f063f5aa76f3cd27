"""The plan in one launch, a workgroup per expert: the edges of the ids a thread keeps (4, 8, 12, 16) and of its range (16384 ids, one
more), a wave's last round that is not full, one expert and the most, ids that name no expert (64-bit ones whose lower half does
among them), a prefix of active tokens.  All results are whole numbers."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, plan_oracle, recorded_kernels, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (64, 1, 8), (63, 5, 512), (1024, 4, 64), (4097, 1, 7), (1024, 8, 512), (8193, 1, 3),
                                   (1536, 8, 130), (12289, 1, 64), (1365, 12, 256), (2048, 8, 64), (16384, 1, 2), (2341, 7, 16),
                                   (16385, 1, 9)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("same", [False, True])
def test_plan_of_a_workgroup_per_expert(gpu, oracle, T, K, E, dtype, same):
    announce("plan per expert T=%d K=%d E=%d %s same=%d" % (T, K, E, dtype, same))
    rng = np.random.default_rng(T + E)
    ids = np.tile(rng.integers(0, E, size=(1, K)), (T, 1)) if same else rng.integers(0, E, size=(T, K))
    ids = np.where(rng.random((T, K)) < 0.1, rng.choice([-1, E, 1 << 20], size=(T, K)), ids).astype(np.int64)
    given = ids.copy()
    if dtype == torch.int64:
        given[ids < 0] = 1 << 32    # no expert either, though its lower half is one's id
    d = cam.moe_dispatch_plan(torch.from_numpy(given).to(dtype).to(gpu), E)
    cnt, off, pos, _ = plan_oracle(oracle, np.where((ids >= 0) & (ids < E), ids, -1), E, skip_out_of_range=True)
    for name, want in (("num_tokens_per_expert", cnt), ("send_offset", off), ("recv_offset", off), ("recv_count", off + cnt),
                       ("num_recv_tokens_per_expert", cnt)):
        assert_bits_equal(to_np(d[name]).astype(np.int64), np.asarray(want).astype(np.int64), name)
    pos = np.asarray(pos).reshape(T, K)
    row = np.where(pos >= 0, np.asarray(off)[np.clip(ids, 0, E - 1)] + pos, -1)
    assert_bits_equal(to_np(d["send_token_idx"]), pos.astype(np.int32), "ranks")
    assert_bits_equal(to_np(d["slot_row"]), row.astype(np.int32), "rows")
    assert int(d["total"].item()) == int(np.sum(cnt))


@pytest.mark.parametrize("active", [0, 1, 256, 299, 300])
def test_active_prefix(gpu, active):
    """Through a layer of few rows, 2400 ids: what it gives for the active tokens of a mask is what it gives for these tokens alone
    (up to 256 of them, in whose plan no expert has a workgroup)."""
    T, K, E, H, I = 300, 8, 40, 1024, 512
    announce("plan per expert, %d of %d tokens" % (active, T))
    gen = torch.Generator().manual_seed(active)
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=2)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=3)
    dev = [[cam.prepack_weight(w1.to(gpu), True)], [w1s.to(gpu)], [cam.prepack_weight(w2.to(gpu), False)], [w2s.to(gpu)]]
    ids = torch.rand(T, E, generator=gen).topk(K, dim=1).indices.to(torch.int32).to(gpu)
    x, gates = torch.randn(T, H, generator=gen).to(torch.bfloat16).to(gpu), torch.rand(T, K, generator=gen).to(gpu)

    def layer(n, mask):
        return cam.fused_deep_moe(x[:n], ids[:n], *dev, gates[:n], None, mask, "", 1, 0, E, 1, 0, 0, 0)

    out, counts = layer(T, torch.arange(T, device=gpu) < active)
    assert not out[active:].any()
    assert_bits_equal(to_np(counts), np.bincount(ids[:active].reshape(-1).cpu().numpy(), minlength=E), "tokens per expert")
    if active > 0:
        want, want_counts = layer(active, None)
        assert torch.equal(out[:active], want) and torch.equal(counts, want_counts)


@pytest.mark.parametrize("T,launches", [(1, 1), (16384, 1), (16385, 2)])
def test_launches(gpu, T, launches):
    announce("plan launches, %d ids" % T)
    ids = torch.empty(T, 1, dtype=torch.int32, device=gpu)
    assert recorded_kernels(lambda: cam.moe_dispatch_plan(ids, 8)) == launches
