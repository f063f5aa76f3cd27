"""Layers of a handful of tokens in their two launches, int8 bit for bit against the oracle, FP8 within what its sums allow: one slot and the most (8, 16, 32), one row
per expert and as many as tokens (more than are asked for at once), K steps that no wave shares evenly, the shortest and longest rows,
both activation types, weights per expert, experts named twice by a token, ids of no expert, masks down to no token at all, the most
that LDS holds, infinities and NaN; and on which side of its lines a layer takes them."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, recorded_kernels, to_np
from test_gpu_fp8 import _check_layer, _layer_inputs, _u8
from test_gpu_fused import _check, _run
from test_gpu_stream_queues import _check as _check_bits, _ids, _layer as _run_layer, _one_by_one, _weights

pytestmark = pytest.mark.gpu


def _layer(T, H, E, K, I, ids=None):
    g = torch.Generator().manual_seed(T * K + H + I)
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=5)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=6)
    ids = torch.rand(T, max(E, K), generator=g).argsort(dim=1)[:, :K] % E if ids is None else torch.tensor(ids)
    return dict(x=synth.normal_bf16(T, H, seed=7), ids=ids, gates=torch.rand(T, K, generator=g), w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)


@pytest.mark.parametrize("T,H,E,K,I", [
    (1, 512, 1, 1, 512),       # one slot
    (1, 4096, 40, 8, 1536),
    (1, 7168, 16, 12, 640),    # the longest row
    (1, 1152, 3, 8, 3072),     # experts named more than once, the longest products
    (8, 1024, 2, 1, 1152),     # up to eight rows to an expert
    (8, 640, 1, 2, 512),       # eight tokens that all name it twice
    (2, 2048, 64, 8, 1408),
    (4, 4096, 64, 8, 512),     # 32 slots
    (3, 4096, 50, 7, 1024),    # 21 slots
    (5, 2048, 9, 3, 640)])
def test_layer_bit_exact(gpu, oracle, T, H, E, K, I):
    announce("few tokens T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    d = _layer(T, H, E, K, I)
    assert _check(oracle, d, *_run(gpu, d)) == 0
    x = d["x"].half()
    out = cam.fused_deep_moe(x.to(gpu), d["ids"].to(torch.int32).to(gpu), [cam.prepack_weight(d["w1"].to(gpu), True)], [d["w1_scale"].to(gpu)],
                             [cam.prepack_weight(d["w2"].to(gpu), False)], [d["w2_scale"].to(gpu)], d["gates"].to(gpu), None, None, "", 1, 0,
                             E, 1, 0, 0, 0)[0]
    want, _ = oracle.fused_layer_fp16(x.view(torch.int16).numpy().view(np.uint16), d["ids"].numpy(), d["gates"].numpy(), d["w1"].numpy(),
                                      d["w1_scale"].numpy(), d["w2"].numpy(), d["w2_scale"].numpy())
    assert_bits_equal(to_np(out.view(torch.int16)).view(np.uint16), want, "fp16 layer")


@pytest.mark.parametrize("active", [0, 1, 3, 5])
def test_masks_dropped_ids_and_weights_per_expert(gpu, oracle, active):
    announce("few tokens, %d of 5 active" % active)
    d = _layer(5, 1024, 6, 3, 512, ids=[[0, -1, 5], [6, 6, -1], [2, 2, 0], [5, 1, 2], [0, 3, -7]])
    d["x"][2] = 0
    mask = torch.arange(5) < active
    out, etn = _run(gpu, d, mask=mask, per_expert=True)
    # the oracle's layer takes ids that name experts: the others with a weight of nothing, and not counted
    ids = d["ids"].numpy()
    dropped = (ids < 0) | (ids >= 6)
    ok = dict(d, ids=torch.from_numpy(np.where(dropped, 4, ids)), gates=torch.from_numpy(np.where(dropped, 0.0, d["gates"].numpy()).astype(np.float32)))
    want, _ = oracle.fused_layer(synth.bf16_bits(ok["x"]), ok["ids"].numpy(), ok["gates"].numpy(), d["w1"].numpy(), d["w1_scale"].numpy(),
                                 d["w2"].numpy(), d["w2_scale"].numpy(), n_active=active)
    got = to_np(out)
    got, want = np.where(got == 0x8000, 0, got), np.where(want == 0x8000, 0, want)   # (a weight of nothing may leave a zero's sign)
    assert_bits_equal(got, want, "output")
    flat = ids[:active][~dropped[:active]]
    assert_bits_equal(to_np(etn), np.bincount(flat, minlength=6), "tokens per expert")


@pytest.mark.parametrize("T,H,E,K,I,few", [(1, 512, 4, 8, 3072, True), (8, 1024, 4, 1, 512, True), (9, 1024, 4, 1, 512, False),
                                           (2, 768, 32, 4, 3072, False), (8, 896, 32, 1, 3072, False), (4, 512, 32, 2, 2560, False),
                                           (1, 640, 32, 8, 3072, True), (8, 1536, 32, 1, 3072, True), (8, 896, 32, 1, 2048, True), (8, 768, 8, 1, 3072, True),
                                           (4, 5120, 64, 8, 512, False), (4, 4352, 64, 4, 2048, False), (4, 5120, 64, 4, 2048, True),
                                           (8, 6144, 4, 1, 512, True), (8, 6272, 4, 1, 512, False),
                                           (2, 1024, 8, 8, 1024, True), (2, 1024, 8, 8, 1152, False),
                                           (4, 4096, 64, 8, 512, True), (4, 4096, 63, 8, 512, False), (4, 3968, 64, 8, 512, False),
                                           (5, 4096, 64, 4, 512, False), (4, 4096, 64, 8, 1536, True), (4, 4096, 64, 8, 1664, False)])
def test_which_layers(gpu, T, H, E, K, I, few):
    announce("few tokens or not T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    dev = [[cam.prepack_weight(torch.empty(E, H, 2 * I, dtype=torch.int8, device=gpu), True)], [torch.empty(E, 2 * I, device=gpu)],
           [cam.prepack_weight(torch.empty(E, I, H, dtype=torch.int8, device=gpu), False)], [torch.empty(E, H, device=gpu)]]
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, dtype=torch.int32, device=gpu)
    gates = torch.empty(T, K, device=gpu)
    n = recorded_kernels(lambda: cam.fused_deep_moe(x, ids, *dev, gates, None, None, "", 1, 0, E, 1, 0, 0, 0))
    assert n == 2 if few else n > 2


@pytest.mark.parametrize("T,H,E,K,I,active", [(1, 1024, 4, 1, 256, None), (1, 7168, 16, 8, 1280, None), (2, 4096, 40, 8, 1536, None),
                                              (8, 1152, 3, 1, 2176, None),    # as many rows as tokens, K blocks that no wave shares evenly
                                              (5, 2048, 9, 3, 768, 3), (1, 2048, 12, 12, 1024, None)])
def test_fp8_layer(gpu, oracle, T, H, E, K, I, active):
    announce("few tokens FP8 T=%d H=%d E=%d K=%d I=%d active=%s" % (T, H, E, K, I, active))
    ids, w, x, w1, s1, w2, s2 = _layer_inputs(T, H, E, K, I, seed=T + H)
    dev = [cam.prepack_weight(w1.to(gpu), True), s1.to(gpu), cam.prepack_weight(w2.to(gpu), False), s2.to(gpu)]
    mask = None if active is None else (torch.arange(T) < active).to(gpu)
    n = T if active is None else active

    def layer():
        return cam.fused_deep_moe_fp8(x.to(gpu), ids.to(torch.int32).to(gpu), *dev, w.to(gpu), mask)

    out, etn = layer()
    want, dbg = oracle.fp8_fused_layer(synth.bf16_bits(x[:n]), ids[:n].numpy(), w[:n].numpy(), _u8(w1), s1.numpy(), _u8(w2), s2.numpy(),
                                       debug=True)
    assert np.array_equal(etn.cpu().numpy(), dbg["cnt"])
    _check_layer(out[:n].float().cpu().numpy(), want)
    assert not out[n:].any()
    assert torch.equal(layer()[0], out)    # sums in the same order every time


@pytest.mark.parametrize("T,H,E,K,I,few", [(1, 1024, 4, 8, 2048, True), (1, 1024, 4, 8, 2176, False), (2, 4096, 4, 8, 1792, True),
                                           (2, 4096, 4, 8, 1920, False), (4, 1024, 4, 4, 768, True), (4, 1024, 4, 4, 896, False),
                                           (4, 4096, 64, 8, 512, False), (4, 5120, 64, 4, 1536, False), (2, 5120, 64, 5, 1024, True)])
def test_which_fp8_layers(gpu, T, H, E, K, I, few):
    announce("few tokens or not, FP8 T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    f8 = torch.float8_e4m3fn
    dev = [cam.prepack_weight(torch.empty(E, H, 2 * I, dtype=f8, device=gpu), True), torch.empty(E, H // 128, I // 64, dtype=torch.uint8, device=gpu),
           cam.prepack_weight(torch.empty(E, I, H, dtype=f8, device=gpu), False), torch.empty(E, I // 128, H // 128, dtype=torch.uint8, device=gpu)]
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, dtype=torch.int32, device=gpu)
    gates = torch.empty(T, K, device=gpu)
    n = recorded_kernels(lambda: cam.fused_deep_moe_fp8(x, ids, *dev, gates))
    assert n == 2 if few else n > 2


def _device_layer(gpu, fp8, T, H, E, K, I, seed):
    w = _weights(gpu, fp8, E, H, I)
    g = torch.Generator(device=gpu).manual_seed(seed)
    return w, torch.randn(T, H, generator=g, device=gpu).to(torch.bfloat16), torch.rand(T, K, generator=g, device=gpu)


@pytest.mark.parametrize("T,H,E,K,I", [(8, 6144, 16, 2, 2048), (4, 4096, 64, 8, 1536), (2, 7168, 8, 8, 3072)])
def test_largest_rows_in_lds(gpu, T, H, E, K, I):
    """The most bytes of rows in either launch (48 KB, T * H and slots * I), against the operators one by one."""
    announce("few tokens, largest T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    w, x, gates = _device_layer(gpu, False, T, H, E, K, I, T)
    for kind in ("spread", "one", "dropped"):
        ids = _ids(gpu, kind, T, E, K, T)
        assert recorded_kernels(lambda: _run_layer(False, E, w, x, ids, gates)) == 2
        _check_bits(False, E, w, x, ids, gates, _run_layer(False, E, w, x, ids, gates))


def test_largest_fp8_rows_in_lds(gpu, oracle):
    """16 slots of I 3072: 48 KB of rows, whose 384 scales fill their table, beside the sums of all waves."""
    T, H, E, K, I = 2, 7168, 8, 8, 3072
    announce("few tokens FP8, largest")
    ids, w, x, w1, s1, w2, s2 = _layer_inputs(T, H, E, K, I, seed=11)
    dev = [cam.prepack_weight(w1.to(gpu), True), s1.to(gpu), cam.prepack_weight(w2.to(gpu), False), s2.to(gpu)]
    on_gpu = [t.to(gpu) for t in (x, ids.to(torch.int32), w)]
    assert recorded_kernels(lambda: cam.fused_deep_moe_fp8(*on_gpu[:2], *dev, on_gpu[2])) == 2
    out, etn = cam.fused_deep_moe_fp8(*on_gpu[:2], *dev, on_gpu[2])
    want, dbg = oracle.fp8_fused_layer(synth.bf16_bits(x), ids.numpy(), w.numpy(), _u8(w1), s1.numpy(), _u8(w2), s2.numpy(), debug=True)
    assert np.array_equal(etn.cpu().numpy(), dbg["cnt"])
    _check_layer(out.float().cpu().numpy(), want)


@pytest.mark.parametrize("fp8", [False, True])
def test_infinities_and_nan(gpu, fp8):
    """What a token holds stays in its own output: tokens with infinities and NaN are non-finite where the operators one by one make
    them so, the others have the bits they have without them."""
    T, H, E, K, I = 4, 2048, 8, 2, 640
    announce("few tokens, infinities and NaN fp8=%d" % fp8)
    w, x, gates = _device_layer(gpu, fp8, T, H, E, K, I, 5)
    ids = torch.tensor([[0, 1], [1, 2], [0, 1], [1, 0]], dtype=torch.int32, device=gpu)   # rows of one expert side by side
    clean = _run_layer(fp8, E, w, x, ids, gates)[0]
    x[1, H - 1] = float("nan")
    x[2, 0], x[2, 777] = float("inf"), float("-inf")
    assert recorded_kernels(lambda: _run_layer(fp8, E, w, x, ids, gates)) == 2
    got = _run_layer(fp8, E, w, x, ids, gates)[0]
    want = _one_by_one(fp8, E, w, x, ids, gates)[0]
    for t in (0, 3):
        assert torch.equal(got[t].view(torch.int16), clean[t].view(torch.int16))
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
