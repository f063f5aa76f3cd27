"""The tile form of the grouped GEMM through each of its epilogues, at shapes past the limits up to which launches stream
(rows x columns; see stream_gemm_applies): the smallest work that still reaches it.  A test of an operator also checks
that its tiles were scheduled, so that a later change of those limits cannot turn it into a test of the other form."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import _lib, synth
from gpu_util import announce, assert_bits_equal, to_np
from test_gpu_fp8 import _check_layer, _layer_inputs, _rand_e8m0, _rand_fp8, _u8
from test_gpu_fused import _check, _run

pytestmark = pytest.mark.gpu

LIMIT = 32 * 512 * 256  # rows x columns that stream at most (FP8 with up to 32 rows per expert: three times as many)

# Rows per expert: edges of the flat tile (up to 128 rows) and of the tall one (up to 256, in units of 32), several tiles
# per expert, empty experts at the ends and between, one row alone.
MIXED = [0, 1, 33, 128, 129, 0, 160, 161, 255, 256, 257, 64, 31, 600, 0]
FLAT = [0, 96, 1, 128, 127, 32, 33, 0, 65] * 4 + [100, 0]


def _scheduled(op, args, gpu):
    """Runs an operator and returns how many tiles it scheduled (0: it streamed)."""
    ws = torch.zeros(64 << 20, dtype=torch.uint8, device=gpu)
    _lib.call(op, args, workspace=ws)
    return int(ws[:4].view(torch.int32)[0])


def _tiles(sizes, N):
    return sum(((s + 255) // 256) * ((N + 255) // 256) if s > 128 else ((N + 511) // 512 if s > 0 else 0) for s in sizes)


def _int8_case(sizes, K, N, seed, as_list=False, gpu=None, gate_up=False):
    G, A = len(sizes), sum(sizes)
    assert A * N > LIMIT
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    x = synth.uniform_int8((A, K), seed)
    xs = synth.channel_scales((A,), seed + 1, lo=0.005, hi=0.05)
    w, ws = synth.uniform_int8((G, K, N), seed + 2, -16, 16), synth.channel_scales((G, N), seed + 3)
    if as_list:
        wp, wsp = [cam.prepack_weight(w[g].to(gpu), gate_up) for g in range(G)], [ws[g].to(gpu) for g in range(G)]
    else:
        wp, wsp = [cam.prepack_weight(w.to(gpu), gate_up)], [ws.to(gpu)]
    return gl, x, xs, w, ws, wp, wsp


@pytest.mark.parametrize("sizes,H,I,list_type,as_list", [
    (MIXED, 128, 1088, 0, False),      # shortest K; 2176 columns = 8.5 tall and 4.25 flat column blocks
    (MIXED, 640, 1408, 1, False),      # 2816 columns = 11 and 5.5
    (MIXED, 256, 1472, 0, True),       # 2944 columns = 11.5 and 5.75; a weight tensor per expert
    (FLAT, 256, 1216, 1, False),       # flat tiles alone; 2432 columns = 4.75 flat blocks
    ([2100, 0, 5], 2048, 1024, 0, False),
])
def test_swiglu_quant_bit_exact(gpu, oracle, sizes, H, I, list_type, as_list):
    announce("tile form, swiglu: sizes=%s H=%d I=%d list_type=%d as_list=%s" % (sizes[:8], H, I, list_type, as_list))
    A = sum(sizes)
    gl, x, xs, w, ws, wp, wsp = _int8_case(sizes, H, 2 * I, A + I, as_list, gpu, True)
    x[A // 2] = 0
    given = gl.to(gpu) if list_type == 0 else torch.tensor(sizes, dtype=torch.int64, device=gpu)
    y, ys = cam.grouped_matmul_swiglu_quant(x.to(gpu), xs.to(gpu), wp, wsp, given, list_type)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    want, want_s = oracle.swiglu_quant(oracle.gmm1_epilogue(c, ws.numpy(), xs.numpy(), gl.numpy()), rows=A)
    assert_bits_equal(to_np(ys).view(np.uint32), want_s.view(np.uint32), "y_scale")
    assert_bits_equal(to_np(y), want, "y")
    assert (to_np(y)[A // 2] == 0).all()
    assert _scheduled("GroupedMatmulSwigluQuant", [x.to(gpu), xs.to(gpu), wp, wsp, given, list_type, y, ys],
                      gpu) == _tiles(sizes, 2 * I)


@pytest.mark.parametrize("sizes,I,H,list_type,as_list", [
    (MIXED, 128, 2112, 0, False),      # 8.25 tall and 4.125 flat column blocks
    (MIXED, 896, 2816, 1, True),
    (FLAT, 256, 2880, 0, False),
    ([3000], 1536, 1472, 0, False),
])
@pytest.mark.parametrize("kind", ["bf16", "fp16", "wire"])
def test_dequant_bit_exact(gpu, oracle, sizes, I, H, list_type, as_list, kind):
    announce("tile form, %s rows: sizes=%s I=%d H=%d list_type=%d as_list=%s" % (kind, sizes[:8], I, H, list_type, as_list))
    A = sum(sizes)
    gl, x, xs, w, ws, wp, wsp = _int8_case(sizes, I, H, A + H, as_list, gpu)
    given = gl.to(gpu) if list_type == 0 else torch.tensor(sizes, dtype=torch.int64, device=gpu)
    out = cam.grouped_matmul_dequant(x.to(gpu), xs.to(gpu), wp, wsp, given, list_type, wire_rows=kind == "wire",
                                     out_dtype=torch.float16 if kind == "fp16" else torch.bfloat16)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    if kind == "fp16":
        want = oracle.gmm2_epilogue_act(c, ws.numpy(), xs.numpy(), gl.numpy(), True)
        got = out.cpu().view(torch.int16).numpy().view(np.uint16)
    else:
        want = oracle.gmm2_epilogue(c, ws.numpy(), xs.numpy(), gl.numpy())
        got = to_np(out)
    if kind == "wire":
        want, got = oracle.comm_quant_rows(want), out.cpu().numpy().view(np.uint8)
    assert_bits_equal(got, want, kind + " rows")
    assert _scheduled("GroupedMatmulDequant", [x.to(gpu), xs.to(gpu), wp, wsp, given, list_type, out], gpu) == _tiles(sizes, H)


def test_wire_rows_stop_at_the_rows_of_the_list(gpu, oracle):
    """The list ends before the rows do: what is quantised for the wire ends there, too."""
    announce("tile form, wire rows, fewer rows than the input has")
    sizes, I, H = MIXED, 128, 2304
    A, more = sum(sizes), 37
    gl, x, xs, w, ws, wp, wsp = _int8_case(sizes, I, H, 5, False, gpu)
    xx = torch.cat([x, torch.full((more, I), 3, dtype=torch.int8)])
    xxs = torch.cat([xs, torch.ones(more)])
    out = torch.full((A + more, H + H // 4), 77, dtype=torch.int8, device=gpu)
    assert _scheduled("GroupedMatmulDequant", [xx.to(gpu), xxs.to(gpu), wp, wsp, gl.to(gpu), 0, out], gpu) == _tiles(sizes, H)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    want = oracle.comm_quant_rows(oracle.gmm2_epilogue(c, ws.numpy(), xs.numpy(), gl.numpy()))
    assert_bits_equal(out[:A].cpu().numpy().view(np.uint8), want, "wire rows")
    assert (out[A:] == 77).all()


FP8_FLAT = [0, 1, 62, 33] * 10 + [64, 0, 31, 32]   # 25 rows per expert on average: past three times the limit of int8


def _fp8_case(sizes, K, N, gpu, gate_up):
    G, A = len(sizes), sum(sizes)
    assert A * N > (3 * LIMIT if A <= 32 * G else LIMIT)
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    seed = K + N
    a, sa = _rand_fp8((A, K), seed, 2.0), _rand_e8m0((A, K // 128), seed + 1, -6, 2)
    w, sw = _rand_fp8((G, K, N), seed + 2), _rand_e8m0((G, K // 128, N // 128), seed + 3, -6, 2)
    return gl, a, sa, w, sw, cam.prepack_weight(w.to(gpu), gate_up)


@pytest.mark.parametrize("sizes,K,N,gate_up", [
    (MIXED, 128, 2176, False),       # one K block; ragged column blocks
    (MIXED, 640, 2304, False),       # five K blocks: a row's scales are no whole words
    (MIXED, 640, 2304, True),
    (MIXED, 1024, 2816, True),
    ([700, 130, 1, 1000], 4096, 2560, False),
    (FP8_FLAT, 256, 13312, True),
    (FP8_FLAT, 384, 13440, False),
])
def test_fp8_sums(gpu, oracle, sizes, K, N, gate_up):
    """fp32 sums and bf16 rows of the scaled FP8 products against double accumulation.  Tolerance as in test_gpu_fp8: |diff|
    <= 1e-3 |want| + 2e-4 max|want| for the sums (the matrix core aligns the products of an instruction before adding
    them), and one rounding to bf16 (2^-8) more for the rows."""
    announce("tile form, fp8 sums: sizes=%s K=%d N=%d gate_up=%s" % (sizes[:8], K, N, gate_up))
    gl, a, sa, w, sw, wp = _fp8_case(sizes, K, N, gpu, gate_up)
    c = oracle.fp8_gemm(_u8(a), sa.numpy(), _u8(w), sw.numpy(), gl.numpy())
    want = oracle.fp8_swiglu(c) if gate_up else c
    biggest = np.abs(want).max()
    args = (a.to(gpu), sa.to(gpu), wp, sw.to(gpu), gl.to(gpu))
    got = cam.grouped_matmul_fp8(*args)   # SwiGLU products; plain sums, which are tiles at any size
    assert (np.abs(got.cpu().numpy() - want) <= 1e-3 * np.abs(want) + 2e-4 * biggest).all()
    if not gate_up:
        got = cam.grouped_matmul_fp8(*args, out_dtype=torch.bfloat16)
        assert (np.abs(got.float().cpu().numpy() - want) <= (2.0 ** -8 + 1e-3) * np.abs(want) + 2e-4 * biggest).all()
    assert _scheduled("GroupedMatmulFp8", [args[0], args[1], wp, args[3], 1 if gate_up else 0, args[4], 0, got, None],
                      gpu) == _tiles(sizes, N)


@pytest.mark.parametrize("sizes,K,N", [
    (MIXED, 256, 2304),              # 9 tall and 4.5 flat column blocks: the last two waves of the last flat item have no columns
    (MIXED, 640, 2816),              # 5.5 flat blocks; scales that are no whole words
    ([700, 130, 1, 1000], 4096, 2560),
    (FP8_FLAT, 256, 13568),          # flat tiles alone, 26.5 blocks
])
def test_fp8_quantised_product_bit_exact(gpu, oracle, sizes, K, N):
    """The epilogue that quantises the SwiGLU product against the product followed by QuantRowsFp8: the same sums, so the
    same bits (the products themselves: test_fp8_sums)."""
    announce("tile form, fp8 quantised product: sizes=%s K=%d N=%d" % (sizes[:8], K, N))
    gl, a, sa, w, sw, wp = _fp8_case(sizes, K, N, gpu, True)
    args = (a.to(gpu), sa.to(gpu), wp, sw.to(gpu), gl.to(gpu))
    want_q, want_s = cam.quant_rows_fp8(cam.grouped_matmul_fp8(*args))
    q, s = cam.grouped_matmul_fp8(*args, out_dtype=torch.float8_e4m3fn)
    assert torch.equal(s, want_s)
    assert np.array_equal(_u8(q), _u8(want_q))
    assert _scheduled("GroupedMatmulFp8", [args[0], args[1], wp, args[3], 1, args[4], 0, q, s], gpu) == _tiles(sizes, N)


def _layer(T, H, E, K, I, seed):
    ids, gates = synth.sigmoid_zipf_routing(T, E, K, seed=seed) if K > 2 else synth.softmax_topk_routing(T, E, K, seed=seed)
    w1, w1s = synth.absmax_int8_weights(E, H, 2 * I, seed=seed + 1)
    w2, w2s = synth.absmax_int8_weights(E, I, H, seed=seed + 2)
    x = synth.normal_bf16(T, H, seed=seed + 3)
    x[T // 3] = 0
    return dict(x=x, ids=ids, gates=gates, w1=w1, w1_scale=w1s, w2=w2, w2_scale=w2s)


@pytest.mark.parametrize("T,H,E,K,I,active,as_list,dropped", [
    (500, 512, 8, 2, 2176, None, False, False),     # 1000 ids: plan of one workgroup
    (512, 1152, 16, 4, 1152, None, False, False),   # 2048 ids: the most that plan and permute share a launch for where
                                                    # there are no schedules; ragged column blocks
    (513, 1024, 16, 4, 1152, None, False, True),    # 2052 ids, some dropped
    (700, 1024, 16, 4, 768, 601, True, False),      # masked tokens, a weight tensor per expert
    (2100, 512, 4, 1, 1152, 1000, False, False),    # most tokens masked
    (1021, 1024, 64, 6, 768, None, False, False),   # most experts flat
])
def test_layer_bit_exact(gpu, oracle, T, H, E, K, I, active, as_list, dropped):
    """Layers whose schedules are built in the plan."""
    announce("tile form, layer T=%d H=%d E=%d K=%d I=%d active=%s as_list=%s dropped=%s" % (T, H, E, K, I, active, as_list,
                                                                                          dropped))
    assert T * K * 2 * I > LIMIT
    d = _layer(T, H, E, K, I, T + I)
    if dropped:
        d["ids"][::7, 1] = -1
    mask = None if active is None else torch.arange(T) < active
    out, etn = _run(gpu, d, mask=mask, per_expert=as_list, via_torch_ops=not as_list)
    assert _check(oracle, d, out, etn, n_active=active) == 0
    if active is not None:
        assert (out[active:] == 0).all()


@pytest.mark.parametrize("T,H,E,K,I", [(700, 1152, 16, 4, 1408), (1500, 512, 8, 2, 768)])
def test_layer_fp16_bit_exact(gpu, oracle, T, H, E, K, I):
    announce("tile form, fp16 layer T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    assert T * K * 2 * I > LIMIT
    d = _layer(T, H, E, K, I, T)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).half()
    d["x"] = x
    out, etn = _run(gpu, d)
    assert out.dtype == torch.float16
    want, cnt = oracle.fused_layer_fp16(x.view(torch.int16).numpy().view(np.uint16), d["ids"].numpy(), d["gates"].numpy(),
                                        d["w1"].numpy(), d["w1_scale"].numpy(), d["w2"].numpy(), d["w2_scale"].numpy())
    assert_bits_equal(to_np(etn), cnt.astype(np.int64), "expert_token_nums")
    assert_bits_equal(out.cpu().view(torch.int16).numpy().view(np.uint16), want, "fp16 layer output")


@pytest.mark.parametrize("T,H,E,K,I,active", [(700, 1024, 16, 4, 1024, None), (901, 1152, 8, 2, 1280, 650)])
def test_fp8_layer(gpu, oracle, T, H, E, K, I, active):
    announce("tile form, fp8 layer T=%d H=%d E=%d K=%d I=%d active=%s" % (T, H, E, K, I, active))
    assert T * K * 2 * I > LIMIT and T * K > 32 * E
    ids, w, x, w1, s1, w2, s2 = _layer_inputs(T, H, E, K, I, seed=T)
    mask = None if active is None else (torch.arange(T) < active).to(gpu)
    out, etn = cam.fused_deep_moe_fp8(x.to(gpu), ids.to(torch.int32).to(gpu), cam.prepack_weight(w1.to(gpu), True), s1.to(gpu),
                                      cam.prepack_weight(w2.to(gpu), False), s2.to(gpu), w.to(gpu), mask)
    n = T if active is None else active
    want, dbg = oracle.fp8_fused_layer(synth.bf16_bits(x)[:n], ids.numpy()[:n], w.numpy()[:n], _u8(w1), s1.numpy(), _u8(w2),
                                       s2.numpy(), debug=True)
    assert np.array_equal(etn.cpu().numpy(), dbg["cnt"])
    _check_layer(out[:n].float().cpu().numpy(), want)
    assert (out[n:] == 0).all()


@pytest.mark.parametrize("seed", range(6))
def test_random_shapes_bit_exact(gpu, oracle, seed):
    """Both int8 operators on seeded shapes that nobody picked by hand."""
    rng = np.random.default_rng(7000 + seed)
    G = int(rng.choice([1, 3, 8, 24, 64, 130]))
    H = 128 * int(rng.integers(1, 9))
    I = 128 * int(rng.integers(8, 16))
    N2 = 64 * int(rng.integers(20, 40))
    A = LIMIT // min(2 * I, N2) + int(rng.integers(1, 700))
    cut = np.sort(rng.integers(0, A + 1, size=G - 1))
    sizes = np.diff(np.concatenate([[0], cut, [A]])).tolist()
    list_type = int(rng.integers(0, 2))
    announce("tile form, random: seed=%d G=%d A=%d H=%d I=%d N2=%d list_type=%d" % (seed, G, A, H, I, N2, list_type))
    gl, x, xs, w, ws, wp, wsp = _int8_case(sizes, H, 2 * I, seed, False, gpu, True)
    given = gl.to(gpu) if list_type == 0 else torch.tensor(sizes, dtype=torch.int64, device=gpu)
    y, ys = cam.grouped_matmul_swiglu_quant(x.to(gpu), xs.to(gpu), wp, wsp, given, list_type)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    want, want_s = oracle.swiglu_quant(oracle.gmm1_epilogue(c, ws.numpy(), xs.numpy(), gl.numpy()), rows=A)
    assert_bits_equal(to_np(ys).view(np.uint32), want_s.view(np.uint32), "y_scale")
    assert_bits_equal(to_np(y), want, "y")
    w2, w2s = synth.uniform_int8((G, I, N2), seed + 9, -16, 16), synth.channel_scales((G, N2), seed + 10)
    out = cam.grouped_matmul_dequant(y, ys, cam.prepack_weight(w2.to(gpu), False), w2s.to(gpu), given, list_type)
    c = oracle.gmm_int32(want, w2.numpy(), gl.numpy())
    assert_bits_equal(to_np(out), oracle.gmm2_epilogue(c, w2s.numpy(), want_s, gl.numpy()), "rows")


# Rows per expert at the edges of every number of row fragments a narrow tile has, and column counts for which the items of a
# launch are more than the CUs (256) and at most two for each, and at most three with the flat ones cut in two.
NARROW = [1, 31, 32, 33, 64, 65, 96, 97, 127, 128] * 4 + [0]


def _narrow_tiles(sizes, N, gpu):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    cut = sum((s + 255) // 256 for s in sizes) * ((N + 255) // 256)
    wide = _tiles(sizes, N)
    if cus == 256:
        assert cus < wide <= 2 * cus and cut <= 3 * cus
    return cut if cus < wide <= 2 * cus and cut <= 3 * cus else wide


@pytest.mark.parametrize("list_type", [0, 1])
def test_narrow_int8_bit_exact(gpu, oracle, list_type):
    H, I, N2 = 256, 1984, 4032   # 31 groups of 128 columns gate and up, 63 of 64: the last column block is ragged
    announce("tile form, narrow tiles, int8: H=%d I=%d N2=%d list_type=%d" % (H, I, N2, list_type))
    gl, x, xs, w, ws, wp, wsp = _int8_case(NARROW, H, 2 * I, 31, False, gpu, True)
    given = gl.to(gpu) if list_type == 0 else torch.tensor(NARROW, dtype=torch.int64, device=gpu)
    y, ys = cam.grouped_matmul_swiglu_quant(x.to(gpu), xs.to(gpu), wp, wsp, given, list_type)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    want, want_s = oracle.swiglu_quant(oracle.gmm1_epilogue(c, ws.numpy(), xs.numpy(), gl.numpy()), rows=x.size(0))
    assert_bits_equal(to_np(ys).view(np.uint32), want_s.view(np.uint32), "y_scale")
    assert_bits_equal(to_np(y), want, "y")
    assert _scheduled("GroupedMatmulSwigluQuant", [x.to(gpu), xs.to(gpu), wp, wsp, given, list_type, y, ys],
                      gpu) == _narrow_tiles(NARROW, 2 * I, gpu)
    gl, x, xs, w, ws, wp, wsp = _int8_case(NARROW, 384, N2, 37, False, gpu)
    c = oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy())
    for fp16 in (False, True):
        out = cam.grouped_matmul_dequant(x.to(gpu), xs.to(gpu), wp, wsp, given, list_type,
                                         out_dtype=torch.float16 if fp16 else torch.bfloat16)
        want = oracle.gmm2_epilogue_act(c, ws.numpy(), xs.numpy(), gl.numpy(), fp16)
        assert_bits_equal(out.cpu().view(torch.int16).numpy().view(np.uint16), want, "rows")
        assert _scheduled("GroupedMatmulDequant", [x.to(gpu), xs.to(gpu), wp, wsp, given, list_type, out],
                          gpu) == _narrow_tiles(NARROW, N2, gpu)


@pytest.mark.parametrize("K", [128, 384, 512])   # scales that are no whole words, and words
def test_narrow_fp8(gpu, oracle, K):
    """Tolerances of test_fp8_sums; the quantised product bit for bit, as above."""
    announce("tile form, narrow tiles, fp8: K=%d" % K)
    for N, gate_up in ((3840, True), (3968, False)):
        gl, a, sa, w, sw, wp = _fp8_case(NARROW, K, N, gpu, gate_up)
        c = oracle.fp8_gemm(_u8(a), sa.numpy(), _u8(w), sw.numpy(), gl.numpy())
        want = oracle.fp8_swiglu(c) if gate_up else c
        biggest = np.abs(want).max()
        args = (a.to(gpu), sa.to(gpu), wp, sw.to(gpu), gl.to(gpu))
        got = cam.grouped_matmul_fp8(*args)
        assert (np.abs(got.cpu().numpy() - want) <= 1e-3 * np.abs(want) + 2e-4 * biggest).all()
        s = None
        if gate_up:
            want_q, want_s = cam.quant_rows_fp8(got)
            got, s = cam.grouped_matmul_fp8(*args, out_dtype=torch.float8_e4m3fn)
            assert torch.equal(s, want_s) and np.array_equal(_u8(got), _u8(want_q))
        else:
            got = cam.grouped_matmul_fp8(*args, out_dtype=torch.bfloat16)
            assert (np.abs(got.float().cpu().numpy() - want) <= (2.0 ** -8 + 1e-3) * np.abs(want) + 2e-4 * biggest).all()
        assert _scheduled("GroupedMatmulFp8", [args[0], args[1], wp, args[3], 1 if gate_up else 0, args[4], 0, got, s],
                          gpu) == _narrow_tiles(NARROW, N, gpu)


def test_narrow_layer_bit_exact(gpu, oracle):
    """The narrow schedule as the plan builds it."""
    T, H, E, K, I = 1021, 512, 64, 6, 1152
    announce("tile form, narrow tiles, layer T=%d H=%d E=%d K=%d I=%d" % (T, H, E, K, I))
    d = _layer(T, H, E, K, I, 5)
    out, etn = _run(gpu, d)
    assert _check(oracle, d, out, etn) == 0
    _narrow_tiles(etn.tolist(), 2 * I, gpu)
