"""Layers whose streaming GEMMs take their last items from queues: every bit as the operators one by one give it, whose items are all
dealt out beforehand.  Spread and uneven ids, ids that leave most queues empty (fewer items than workgroups), dropped ids, inactive
tokens, column groups that do not fill the last block; replays of a graph with other ids in between, so the counts are those of the
replay; and which GEMMs there are queues for, and how wide their items are without."""
import pytest
import torch

import umdk_original_amd as cam
from gpu_util import announce, recorded_names

pytestmark = pytest.mark.gpu


def _weights(gpu, fp8, E, H, I):
    g = torch.Generator(device=gpu).manual_seed(E + H + I)

    def one(kd, n, gate_up):
        if not fp8:
            q = torch.randint(-127, 128, (E, kd, n), generator=g, dtype=torch.int8, device=gpu)
            return cam.prepack_weight(q, gate_up), torch.rand(E, n, generator=g, device=gpu) * 1e-3 + 1e-4
        # bytes of magnitude up to 0x6f: no NaN among them
        q = torch.randint(0, 0x70, (E, kd, n), generator=g, dtype=torch.uint8, device=gpu)
        q |= torch.randint(0, 2, (E, kd, n), generator=g, dtype=torch.uint8, device=gpu) << 7
        scale = torch.randint(114, 118, (E, kd // 128, n // 128), generator=g, dtype=torch.uint8, device=gpu)
        return cam.prepack_weight(q.view(torch.float8_e4m3fn), gate_up), scale

    return one(H, 2 * I, True) + one(I, H, False)


def _ids(gpu, kind, T, E, K, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    score = torch.rand(T, E, generator=g, device=gpu)
    if kind == "uneven":
        score += torch.arange(E, device=gpu) < E // 4
    elif kind == "one":
        score += torch.arange(E, device=gpu) >= E - K
    ids = score.topk(K, dim=1).indices.to(torch.int32)
    if kind == "dropped":
        ids[torch.rand(T, K, generator=g, device=gpu) < 0.3] = -1
    return ids.contiguous()


def _layer(fp8, E, w, x, ids, gates, mask=None):
    if fp8:
        return cam.fused_deep_moe_fp8(x, ids, *w, gates, mask)
    return cam.fused_deep_moe(x, ids, *([t] for t in w), gates, None, mask, "", 1, 0, E, 1, 0, 0, 0)


def _one_by_one(fp8, E, w, x, ids, gates):
    d = cam.moe_dispatch_fused(x, ids, E, quant_mode=4 if fp8 else 2)
    rows = d["recv_count"].to(torch.int64)
    if fp8:
        y, s = cam.grouped_matmul_fp8(d["recv_x"], d["recv_x_scales"], w[0], w[1], rows, out_dtype=torch.float8_e4m3fn)
        y = cam.grouped_matmul_fp8(y, s, w[2], w[3], rows, out_dtype=torch.bfloat16)
    else:
        y, s = cam.grouped_matmul_swiglu_quant(d["recv_x"], d["recv_x_scales"], w[0], w[1], rows)
        y = cam.grouped_matmul_dequant(y, s, w[2], w[3], rows)
    return cam.moe_combine_gather(y, None, d["slot_row"], gates), d["num_recv_tokens_per_expert"]


def _queued(fp8, groups):
    return "stream_gemm_kernelILi4ELb%dELi%dELb0ELb1E" % (fp8, groups)


def _check(fp8, E, w, x, ids, gates, got):
    want, counts = _one_by_one(fp8, E, w, x, ids, gates)
    assert torch.equal(got[0].view(torch.int16), want.view(torch.int16))
    assert torch.equal(got[1], counts)


# T, H, E, K, I, column groups of an item in either GEMM (0: no queue)
SHAPES = [(100, 6144, 64, 4, 2304, 2, 4), (33, 3072, 96, 8, 1920, 2, 4), (32, 2176, 250, 6, 1152, 4, 0)]
SHAPES8 = [(100, 6144, 64, 4, 2304, 4, 4), (340, 3072, 128, 8, 2304, 4, 4), (40, 6784, 80, 8, 2688, 4, 2), (200, 3328, 128, 8, 1152, 4, 4),
           (190, 3328, 128, 8, 1152, 4, 0), (200, 2048, 64, 8, 1408, 0, 0), (200, 2048, 64, 8, 1152, 0, 0)]


@pytest.mark.parametrize("fp8,shape", [(False, s) for s in SHAPES] + [(True, s) for s in SHAPES8])
def test_layer_as_its_operators(gpu, fp8, shape):
    T, H, E, K, I, up, down = shape
    w = _weights(gpu, fp8, E, H, I)
    g = torch.Generator(device=gpu).manual_seed(T)
    x = torch.randn(T, H, generator=g, device=gpu).to(torch.bfloat16)
    gates = torch.rand(T, K, generator=g, device=gpu)
    for kind in ("spread", "uneven", "one", "dropped"):
        announce("queues fp8=%d T=%d H=%d E=%d K=%d I=%d %s" % (fp8, T, H, E, K, I, kind))
        ids = _ids(gpu, kind, T, E, K, T)
        _check(fp8, E, w, x, ids, gates, _layer(fp8, E, w, x, ids, gates))
    names = recorded_names(lambda: _layer(fp8, E, w, x, ids, gates))
    gemms = [n for n in names if "stream_gemm_kernel" in n]
    assert len(gemms) == 2
    assert [_queued(fp8, p) in n if p else "ELb0ELb0E" in n for n, p in zip(gemms, (up, down))] == [True, True], gemms

    active = T // 3
    announce("queues fp8=%d, %d of %d tokens" % (fp8, active, T))
    ids = _ids(gpu, "uneven", T, E, K, 1)
    out, counts = _layer(fp8, E, w, x, ids, gates, torch.arange(T, device=gpu) < active)
    assert not out[active:].any()
    ids[active:] = -1
    _check(fp8, E, w, x, ids, gates, (out, counts))


def test_replays(gpu):
    T, H, E, K, I, _, _ = SHAPES[0]
    w = _weights(gpu, False, E, H, I)
    x = torch.randn(T, H, device=gpu).to(torch.bfloat16)
    gates = torch.rand(T, K, device=gpu)
    ids = _ids(gpu, "spread", T, E, K, 0)
    _layer(False, E, w, x, ids, gates)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _layer(False, E, w, x, ids, gates)
    for i, kind in enumerate(("spread", "one", "uneven", "spread")):
        announce("queues, replay %d: %s" % (i, kind))
        ids.copy_(_ids(gpu, kind, T, E, K, i))
        graph.replay()
        torch.cuda.synchronize()
        _check(False, E, w, x, ids, gates, got)


@pytest.mark.parametrize("H,E,I,up", [(5120, 44, 1536, 2), (5120, 48, 1536, 4), (4096, 40, 1280, 4)])
def test_groups_of_two_rounds(gpu, H, E, I, up):
    """Column groups of an item where there are one to two rounds of four, K over 4096 and not, and the layer with them."""
    T, K = 40, 6
    announce("two rounds H=%d E=%d I=%d" % (H, E, I))
    w = _weights(gpu, False, E, H, I)
    x, gates = torch.randn(T, H, device=gpu).to(torch.bfloat16), torch.rand(T, K, device=gpu)
    ids = _ids(gpu, "uneven", T, E, K, E)
    _check(False, E, w, x, ids, gates, _layer(False, E, w, x, ids, gates))
    gemm = [n for n in recorded_names(lambda: _layer(False, E, w, x, ids, gates)) if "stream_gemm_kernel" in n][0]
    assert "stream_gemm_kernelILi4ELb0ELi%dELb0E" % up in gemm


@pytest.mark.parametrize("T,H,E,K,I,up,down", [(64, 3072, 128, 6, 1536, 2, 0), (4, 3072, 128, 6, 1536, 0, 0),    # few experts reached
                                               (64, 2560, 128, 6, 2048, 4, 4), (64, 2560, 60, 6, 2048, 0, 0),    # rounds of items
                                               (64, 1536, 128, 6, 2048, 0, 0), (90, 5120, 160, 6, 1536, 2, 4)])
def test_which_gemms(gpu, T, H, E, K, I, up, down):
    announce("queues, which T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    w = (cam.prepack_weight(torch.empty(E, H, 2 * I, dtype=torch.int8, device=gpu), True), torch.empty(E, 2 * I, device=gpu),
         cam.prepack_weight(torch.empty(E, I, H, dtype=torch.int8, device=gpu), False), torch.empty(E, H, device=gpu))
    x, ids = torch.empty(T, H, dtype=torch.bfloat16, device=gpu), torch.empty(T, K, dtype=torch.int32, device=gpu)
    names = recorded_names(lambda: _layer(False, E, w, x, ids, torch.empty(T, K, device=gpu)))
    gemms = [n for n in names if "stream_gemm_kernel" in n]
    assert len(gemms) == 2
    for name, p in zip(gemms, (up, down)):
        assert ("ELb0ELb1E" in name) == (p > 0) and (p == 0 or _queued(False, p) in name), name


# rows, experts, K, N, column groups of an item: the wider items where the workgroup with most of them streams as many columns either
# way, the narrower where it streams fewer
@pytest.mark.parametrize("fp8,gate_up,rows,E,kd,n,groups", [
    (False, True, 2048, 128, 4096, 2048, 4), (False, True, 1792, 112, 5120, 1024, 4), (False, True, 1536, 96, 5120, 1024, 2),
    (False, False, 768, 48, 1408, 2048, 8), (False, False, 768, 48, 2048, 4096, 4),
    (True, True, 2048, 128, 1536, 2048, 8), (True, True, 2048, 96, 1280, 3072, 4), (True, False, 2048, 128, 5120, 2048, 4),
    (True, False, 2048, 96, 5120, 1024, 2)])
def test_items_without_queues(gpu, fp8, gate_up, rows, E, kd, n, groups):
    announce("items without queues fp8=%d gate_up=%d rows=%d E=%d K=%d N=%d" % (fp8, gate_up, rows, E, kd, n))
    dtype = torch.float8_e4m3fn if fp8 else torch.int8
    w = cam.prepack_weight(torch.empty(E, kd, n, dtype=dtype, device=gpu), gate_up)
    x, rows_to = torch.empty(rows, kd, dtype=dtype, device=gpu), torch.empty(E, dtype=torch.int64, device=gpu)
    if fp8:
        xs, ws = torch.empty(rows, kd // 128, dtype=torch.uint8, device=gpu), torch.empty(E, kd // 128, n // 128, dtype=torch.uint8, device=gpu)
        out = torch.float8_e4m3fn if gate_up else torch.bfloat16
        names = recorded_names(lambda: cam.grouped_matmul_fp8(x, xs, w, ws, rows_to, out_dtype=out))
    else:
        product = cam.grouped_matmul_swiglu_quant if gate_up else cam.grouped_matmul_dequant
        xs, ws = torch.empty(rows, device=gpu), torch.empty(E, n, device=gpu)
        names = recorded_names(lambda: product(x, xs, w, ws, rows_to))
    gemms = [name for name in names if "stream_gemm_kernel" in name]
    assert len(gemms) == 1 and "stream_gemm_kernelILi4ELb%dELi%dELb0ELb0E" % (fp8, groups) in gemms[0], gemms
