"""Fused layers of which few tokens go anywhere, under a mask (as many tokens as it has entries set, from the first on) or because their
ids name no expert: what they leave in their workspace, and that the mask counts alike wherever it lies and whatever its bytes are."""
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import _lib, synth
from gpu_util import announce
from test_gpu_fp8 import _layer_inputs

pytestmark = pytest.mark.gpu
T, H, E, I = 8192, 1024, 4, 512


def _weights(gpu, fp8):
    if fp8:
        _, _, _, w1, s1, w2, s2 = _layer_inputs(8, H, E, 1, I, seed=6)
    else:
        (w1, s1), (w2, s2) = synth.absmax_int8_weights(E, H, 2 * I, seed=2), synth.absmax_int8_weights(E, I, H, seed=3)
    return [cam.prepack_weight(w1.to(gpu), True), s1.to(gpu), cam.prepack_weight(w2.to(gpu), False), s2.to(gpu)]


def _mask(gpu, where, tokens, active, offset=0):
    """The first, the last or some entries set, to whatever is not zero; `offset` bytes into an allocation."""
    gen = torch.Generator().manual_seed(tokens + active)
    m = torch.zeros(tokens, dtype=torch.uint8)
    at = {"first": torch.arange(active), "last": torch.arange(tokens - active, tokens),
          "some": torch.randperm(tokens, generator=gen)[:active]}[where]
    m[at] = torch.randint(1, 256, (active,), generator=gen, dtype=torch.uint8)
    room = torch.full((tokens + 48,), 255, dtype=torch.uint8, device=gpu)   # (entries beside it count for nothing)
    room[offset:offset + tokens] = m.to(gpu)
    return room[offset:offset + tokens]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("where", ["first", "last", "some", "ids"])
def test_tokens_that_go_nowhere_leave_nothing(gpu, fp8, where):
    announce("masked rows %s fp8=%s" % (where, fp8))
    active = 5
    x = synth.normal_bf16(T, H, seed=1).to(gpu)
    ids = torch.randint(0, E, (T, 1), generator=torch.Generator().manual_seed(4), dtype=torch.int32)
    mask = None
    if where == "ids":
        ids[active:] = torch.tensor([-1, E])[torch.arange(T - active) % 2].to(torch.int32)[:, None]
    else:
        mask = _mask(gpu, where, T, active)
    w1, s1, w2, s2 = _weights(gpu, fp8)
    out, etn = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(E, dtype=torch.int64, device=gpu)
    gates = torch.ones(T, 1, device=gpu)
    if fp8:
        op, args = "FusedDeepMoeFp8", [x, ids.to(gpu), w1, s1, w2, s2, gates, mask, E, out, etn]
    else:
        op, args = "FusedDeepMoe", [x, ids.to(gpu), [w1], [s1], [w2], [s2], gates, None, mask, "", 1, 0, E, 1, 0, 0, 0, out, etn]
    size = _lib.phase1(op, args)[1]
    ws = torch.full((size,), 0x5a, dtype=torch.uint8, device=gpu)
    _lib.call(op, args, workspace=ws)
    assert int(etn.sum()) == active and not out[active:].any() and bool(out[:active].any(dim=1).all())
    # places and maps 12 bytes a token, a few rows of H + 5 I + 2 H bytes, schedules and histograms: not T rows of H bytes
    assert int((ws != 0x5a).sum()) < T * H // 8


@pytest.mark.parametrize("tokens,active,offset", [(1, 1, 15), (15, 7, 1), (16, 16, 0), (17, 3, 8), (31, 30, 3), (33, 17, 16), (300, 299, 5),
                                                  (1500, 1111, 9), (8192, 4097, 0), (8205, 8205, 13), (16384, 77, 7), (16385, 9000, 2)])
def test_what_a_mask_counts(gpu, tokens, active, offset):
    announce("mask of %d tokens, %d set, at %d" % (tokens, active, offset))
    x = synth.normal_bf16(tokens, H, seed=tokens).to(gpu)
    ids = torch.randint(0, E, (tokens, 1), generator=torch.Generator().manual_seed(5), dtype=torch.int32).to(gpu)
    w1, s1, w2, s2 = _weights(gpu, False)
    gates = torch.ones(tokens, 1, device=gpu)

    def layer(n, mask):
        return cam.fused_deep_moe(x[:n], ids[:n], [w1], [s1], [w2], [s2], gates[:n], None, mask, "", 1, 0, E, 1, 0, 0, 0)

    want, want_etn = layer(active, None)
    for where in ("first", "last", "some"):
        out, etn = layer(tokens, _mask(gpu, where, tokens, active, offset))
        assert torch.equal(etn, want_etn) and not out[active:].any()
        assert torch.equal(out[:active].view(torch.int16), want.view(torch.int16))
