"""The grouped GEMM's streaming form (few rows per expert) against the oracle at the sizes where it can go wrong: edges
of its 32- and 128-row tiles and of their eight-row blocks, a K shorter than one turn of the waves or no multiple of it,
activations in one LDS chunk and in several, column groups that do not fill the last item, the widest items of FP8 products,
both forms of group list."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, recorded_names, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,H,I", [
    ([1], 128, 64),                                # one row, two K steps, one column group
    ([1, 0, 2, 9, 8, 7], 1408, 704),               # K = 22 steps; N = 22 and 22 groups
    ([31, 32, 33], 512, 192),                      # edges of the 32-row tile
    ([127, 1, 0, 128, 129, 3], 1024, 1152),        # edges of the 128-row tile, one tile more
    ([16] * 24, 7168, 512),                        # the longest K, several activation chunks, many column groups
    ([0, 5] * 100 + [40, 0], 256, 1024),           # 201 experts, half of them empty
    ([300, 200], 640, 128),                        # several row tiles per expert, few columns
])
@pytest.mark.parametrize("list_type", [0, 1])
def test_stream_gemm_operators_bit_exact(gpu, oracle, sizes, H, I, list_type):
    announce("stream gemm sizes=%s H=%d I=%d list_type=%d" % (sizes[:8], H, I, list_type))
    G, A = len(sizes), sum(sizes)
    cnt = torch.tensor(sizes, dtype=torch.int64)
    gl = torch.cumsum(cnt, 0)
    given = (gl if list_type == 0 else cnt).to(gpu)
    x = synth.uniform_int8((A, H), A)
    xs = synth.channel_scales((A,), A + 1, lo=0.005, hi=0.05)
    w1, w1s = synth.uniform_int8((G, H, 2 * I), A + 2, -16, 16), synth.channel_scales((G, 2 * I), A + 3)
    w2, w2s = synth.uniform_int8((G, I, H), A + 4, -16, 16), synth.channel_scales((G, H), A + 5)
    y, ys = cam.grouped_matmul_swiglu_quant(x.to(gpu), xs.to(gpu), cam.prepack_weight(w1.to(gpu), True), w1s.to(gpu), given,
                                            list_type)
    c = oracle.gmm_int32(x.numpy(), w1.numpy(), gl.numpy())
    want_y, want_ys = oracle.swiglu_quant(oracle.gmm1_epilogue(c, w1s.numpy(), xs.numpy(), gl.numpy()), rows=A)
    assert_bits_equal(to_np(ys).view(np.uint32), want_ys.view(np.uint32), "y_scale")
    assert_bits_equal(to_np(y), want_y, "y")
    if I % 128 == 0:
        out = cam.grouped_matmul_dequant(y, ys, cam.prepack_weight(w2.to(gpu), False), w2s.to(gpu), given, list_type)
        c = oracle.gmm_int32(want_y, w2.numpy(), gl.numpy())
        assert_bits_equal(to_np(out), oracle.gmm2_epilogue(c, w2s.numpy(), want_ys, gl.numpy()), "rows")


@pytest.mark.parametrize("sizes,K,N", [
    ([1, 33, 0, 128], 640, 768),     # five K blocks: a row's scales are no whole words
    ([9, 2], 4096, 512),             # 32 K blocks, two turns of a chunk
    ([130], 128, 256),               # one K block, two row tiles
    ([0, 34, 62] * 10, 256, 8192),   # 32 rows per expert on average, beyond the limit of int8
])
def test_stream_gemm_fp8_sums(gpu, oracle, sizes, K, N):
    announce("stream fp8 gemm sizes=%s K=%d N=%d" % (sizes, K, N))
    G, A = len(sizes), sum(sizes)
    g = torch.Generator().manual_seed(K + N)
    x = torch.randn((A, K), generator=g).mul(4.0).to(torch.float8_e4m3fn)
    w = torch.randn((G, K, N), generator=g).mul(4.0).to(torch.float8_e4m3fn)
    sx = torch.randint(120, 130, (A, K // 128), generator=g).to(torch.uint8)
    sw = torch.randint(120, 130, (G, K // 128, N // 128), generator=g).to(torch.uint8)
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    got = cam.grouped_matmul_fp8(x.to(gpu), sx.to(gpu), cam.prepack_weight(w.to(gpu), False), sw.to(gpu), gl.to(gpu),
                                 out_dtype=torch.bfloat16).float().cpu()
    xf = x.float() * torch.exp2(sx.float() - 127).repeat_interleave(128, 1)
    wf = w.float() * torch.exp2(sw.float() - 127).repeat_interleave(128, 1).repeat_interleave(128, 2)
    want, r = torch.empty(A, N), 0
    for e, n in enumerate(sizes):
        want[r:r + n] = xf[r:r + n] @ wf[e]
        r += n
    assert (got - want).abs().max() <= 2e-2 * want.abs().max()
    assert ((got - want).norm() / want.norm()).item() <= 5e-3


@pytest.mark.parametrize("K,I", [(2048, 1408), (1280, 1152), (1920, 1664)])   # 5.5, 4.5 and 6.5 items of eight column groups
def test_stream_gemm_fp8_products_of_eight_groups(gpu, K, I):
    """Over 24 rows per expert: the fp32 products against 64-bit sums, the quantised ones bit for bit against those, an expert of three
    row tiles and some of none among them."""
    announce("stream fp8 products of eight groups K=%d I=%d" % (K, I))
    G, N = 64, 2 * I
    sizes = synth.zipf_group_sizes(G, 1700, K)
    assert int(sizes.max()) > 256 and int((sizes == 0).sum()) == 3
    A, g = 1700, torch.Generator(device=gpu).manual_seed(K)
    x = torch.randn(A, K, generator=g, device=gpu).mul(4.0).to(torch.float8_e4m3fn)
    w = torch.randn(G, K, N, generator=g, device=gpu).to(torch.float8_e4m3fn)
    sx = torch.randint(121, 125, (A, K // 128), generator=g, dtype=torch.uint8, device=gpu)
    sw = torch.randint(121, 125, (G, K // 128, N // 128), generator=g, dtype=torch.uint8, device=gpu)
    wp, gl = cam.prepack_weight(w, True), torch.cumsum(sizes, 0).to(gpu)
    for out_dtype in (torch.float32, torch.float8_e4m3fn):
        names = recorded_names(lambda: cam.grouped_matmul_fp8(x, sx, wp, sw, gl, out_dtype=out_dtype))
        assert any("stream_gemm_kernelILi4ELb1ELi8E" in n for n in names), names
    got = cam.grouped_matmul_fp8(x, sx, wp, sw, gl)
    q, s = cam.grouped_matmul_fp8(x, sx, wp, sw, gl, out_dtype=torch.float8_e4m3fn)
    want_q, want_s = cam.quant_rows_fp8(got)
    assert torch.equal(q.view(torch.uint8), want_q.view(torch.uint8)) and torch.equal(s, want_s)
    r = 0
    for e, n in enumerate(sizes.tolist()):
        xf = x[r:r + n].double() * torch.exp2(sx[r:r + n].double() - 127).repeat_interleave(128, 1)
        wf = w[e].double() * torch.exp2(sw[e].double() - 127).repeat_interleave(128, 0).repeat_interleave(128, 1)
        gate, up = (xf @ wf).split(I, 1)
        # fp32 sums of K products, the slope of SiLU at most 1.1, and the roundings of SiLU and of the product
        eg, eu = (xf.abs() @ wf.abs()).mul(K * 2.0 ** -23).split(I, 1)
        silu = gate * torch.sigmoid(gate)
        bound = 1.1 * eg * (up.abs() + eu) + silu.abs() * eu + (silu * up).abs() * 2.0 ** -20
        assert ((got[r:r + n].double() - silu * up).abs() <= bound).all()
        r += n


@pytest.mark.parametrize("experts", [1, 63, 64, 65, 128, 511, 512])
@pytest.mark.parametrize("list_type", [0, 1])
def test_stream_gemm_item_list_at_wave_edges(gpu, oracle, experts, list_type):
    """A wave lists 64 experts at a turn: rows in the first and the last expert of every turn, none in most others."""
    announce("stream item list experts=%d list_type=%d" % (experts, list_type))
    sizes = [(1 + e % 3 if e % 64 in (0, 1, 63) else 0) for e in range(experts)]
    sizes[-1] = 33   # two 32-row tiles at the end of the list
    K, N, A = 128, 64, sum(sizes)
    cnt = torch.tensor(sizes, dtype=torch.int64)
    gl = torch.cumsum(cnt, 0)
    x, xs = synth.uniform_int8((A, K), experts), synth.channel_scales((A,), experts + 1, lo=0.005, hi=0.05)
    w, ws = synth.uniform_int8((experts, K, N), experts + 2, -16, 16), synth.channel_scales((experts, N), experts + 3)
    out = cam.grouped_matmul_dequant(x.to(gpu), xs.to(gpu), cam.prepack_weight(w.to(gpu), False), ws.to(gpu),
                                     (gl if list_type == 0 else cnt).to(gpu), list_type)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    assert_bits_equal(to_np(out), oracle.gmm2_epilogue(c, ws.numpy(), xs.numpy(), gl.numpy()), "rows")
