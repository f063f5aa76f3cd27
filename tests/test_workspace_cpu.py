"""What phase 1 asks for where a GEMM streams (few rows): its rows and the plan's scratch, not the schedules of the tile form,
which alone are over 60 KB on any device."""
import pytest
import torch

from umdk_original_amd import _lib
from test_abi_cpu import _fused_args, _packed, _t

SLACK = 16384  # the plan's histograms, metadata, alignment to 256 bytes


@pytest.mark.parametrize("bs,K,E,H,I", [(4, 2, 4, 1024, 512), (1, 8, 128, 4096, 1536), (16, 8, 16, 7168, 2048)])
def test_layers(bs, K, E, H, I):
    st, ws, msg = _lib.phase1("FusedDeepMoe", _fused_args(bs=bs, K=K, E=E, H=H, I=I))
    assert st == _lib.CAM_OK, msg
    row = 8 + max(2 * H, H + 4 * I) + 4 + I + 4 + 2 * H   # (the last where GMM2 reads the products while it writes)
    assert ws <= bs * K * row + SLACK


@pytest.mark.parametrize("rows,G,K,N", [(8, 4, 1024, 1024), (1, 128, 512, 2048)])
def test_operators(rows, G, K, N):
    x, xs, gl = _t((rows, K), torch.int8), _t((rows,), torch.float32), _t((G,), torch.int64)
    w, ws = [_packed((G, K, N))], [_t((G, N), torch.float32)]
    st, swiglu, msg = _lib.phase1("GroupedMatmulSwigluQuant", [x, xs, w, ws, gl, 0, _t((rows, N // 2), torch.int8), xs])
    assert st == _lib.CAM_OK, msg
    assert swiglu <= rows * N // 2 * 4 + 1024
    st, dequant, msg = _lib.phase1("GroupedMatmulDequant", [x, xs, w, ws, gl, 0, _t((rows, N), torch.bfloat16)])
    assert st == _lib.CAM_OK, msg
    assert dequant <= 1024
    # the raw sums always take the tiles
    st, sums, msg = _lib.phase1("GroupedMatmulInt32", [x, w, 0, gl, 0, _t((rows, N), torch.int32)])
    assert st == _lib.CAM_OK and sums > 60000, msg
