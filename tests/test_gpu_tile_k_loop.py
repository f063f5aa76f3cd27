"""The K loop of the tile GEMM at its edges: every number of row fragments of both tile shapes (the last with one row, or one
short of full), K of fewer 128-byte stages than the ring, odd and even numbers of them, column blocks of which the last is
ragged."""
import numpy as np
import pytest
import torch

import umdk_original_amd as cam
from umdk_original_amd import synth
from gpu_util import announce, assert_bits_equal, to_np

pytestmark = pytest.mark.gpu

FLAT = [1, 31, 32, 33, 64, 65, 96, 97, 127, 128]
TALL = [129, 160, 161, 191, 193, 224, 225, 256, 257, 300]


@pytest.mark.parametrize("Kd", [128, 256, 384, 512, 640, 1152])
@pytest.mark.parametrize("name,sizes,N,gate_up", [("flat", FLAT, 9 * 64, False), ("tall", TALL, 9 * 64, False),
                                                  ("flat", FLAT, 11 * 128, True), ("tall", TALL, 5 * 128, True)])
def test_int32_sums_bit_exact(gpu, oracle, name, sizes, N, gate_up, Kd):
    announce("tile form, K loop: %s tiles, K=%d N=%d gate_up=%s" % (name, Kd, N, gate_up))
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    x = synth.uniform_int8((sum(sizes), Kd), Kd)   # no row behind the last tile's
    w = synth.uniform_int8((len(sizes), Kd, N), Kd + N)
    got = cam.grouped_matmul_int32(x.to(gpu), cam.prepack_weight(w.to(gpu), gate_up), gl.to(gpu))
    assert_bits_equal(to_np(got), oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy()), "int32 sums")


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("sizes,Kd,N,gate_up", [
    (FLAT * 4, 128, 63 * 64, False), (FLAT * 4, 384, 31 * 128, True), (FLAT * 3 + [0] + TALL, 640, 31 * 128, False)])
def test_narrow_items(gpu, oracle, sizes, Kd, N, gate_up, fp8):
    """Between one and two items per workgroup: experts of few rows in 256-column blocks.  Tolerance of fp8 as below."""
    from test_gpu_gemm import _schedule_items
    from umdk_original_amd import _lib
    announce("tile form, narrow items: %d experts, K=%d N=%d gate_up=%s fp8=%s" % (len(sizes), Kd, N, gate_up, fp8))
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    A, G = sum(sizes), len(sizes)
    x, w = synth.uniform_int8((A, Kd), Kd), synth.uniform_int8((G, Kd, N), Kd + N)
    if fp8:
        N = N // 128 * 128
        x, w = (x.float() / 32).to(torch.float8_e4m3fn), (w[:, :, :N].float() / 64).to(torch.float8_e4m3fn).contiguous()
        gen = torch.Generator().manual_seed(Kd)
        xs = torch.randint(121, 130, (A, Kd // 128), generator=gen, dtype=torch.uint8)
        ws = torch.randint(121, 130, (G, Kd // 128, N // 128), generator=gen, dtype=torch.uint8)
        got = cam.grouped_matmul_fp8(x.to(gpu), xs.to(gpu), cam.prepack_weight(w.to(gpu), False), ws.to(gpu), gl.to(gpu),
                                     out_dtype=torch.float32).cpu().numpy()
        want = oracle.fp8_gemm(x.view(torch.uint8).numpy(), xs.numpy(), w.view(torch.uint8).numpy(), ws.numpy(), gl.numpy())
        assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 2e-4 * np.abs(want).max()).all()
        return
    out = torch.empty((A, N), dtype=torch.int32, device=gpu)
    packed = cam.prepack_weight(w.to(gpu), gate_up)
    scratch = _lib.call("GroupedMatmulInt32", [x.to(gpu), [packed], int(gate_up), gl.to(gpu), 0, out])
    assert_bits_equal(to_np(out), oracle.gmm_int32(x.numpy(), w.numpy(), gl.numpy()), "int32 sums")
    items, starts, queues, _ = _schedule_items(scratch)
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    wide, tiles = (-(-N // 512), -(-N // 256)), [-(-s // 256) for s in sizes]
    wide = sum(t * wide[s > 128] for s, t in zip(sizes, tiles))
    narrow = sum(tiles) * -(-N // 256)
    if cus < wide <= 2 * cus and narrow <= 3 * cus:
        wide = narrow
    assert len(items) == wide and starts[-1] == wide and queues == cus
    assert cus != 256 or not (items[:, 5] & 0xffff).any()


@pytest.mark.parametrize("Kd", [128, 256, 384, 1024])
@pytest.mark.parametrize("sizes", [FLAT, TALL])
def test_fp8_sums(gpu, oracle, sizes, Kd):
    """Tolerance as in test_gpu_fp8.py: the matrix core aligns the 64 products of an instruction before it adds them."""
    N = 640
    announce("tile form, fp8 K loop: sizes=%s K=%d" % (sizes[:3], Kd))
    gen = torch.Generator().manual_seed(Kd)
    gl = torch.tensor(np.cumsum(sizes), dtype=torch.int64)
    x = torch.randn(sum(sizes), Kd, generator=gen).mul_(2).to(torch.float8_e4m3fn)
    w = torch.randn(len(sizes), Kd, N, generator=gen).to(torch.float8_e4m3fn)
    xs = torch.randint(121, 130, (sum(sizes), Kd // 128), generator=gen, dtype=torch.uint8)
    ws = torch.randint(121, 130, (len(sizes), Kd // 128, N // 128), generator=gen, dtype=torch.uint8)
    got = cam.grouped_matmul_fp8(x.to(gpu), xs.to(gpu), cam.prepack_weight(w.to(gpu), False), ws.to(gpu), gl.to(gpu),
                                 out_dtype=torch.float32).cpu().numpy()
    want = oracle.fp8_gemm(x.view(torch.uint8).numpy(), xs.numpy(), w.view(torch.uint8).numpy(), ws.numpy(), gl.numpy())
    assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 2e-4 * np.abs(want).max()).all(), float(np.abs(got - want).max())
