"""The permute on both sides of the line between all rows of a token asked for at once and one by one (152 MiB of 8-bit rows; int8 29 to 63
MiB of tokens), with dropped ids: every copy of a token in its row, with its scale and its triple.  Each token quantised once by a dispatch to one expert is the reference."""
import pytest
import torch

import umdk_original_amd as cam
from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", [2, 4, 0])
@pytest.mark.parametrize("T,H,E,K", [(1389, 7168, 64, 16), (1390, 7168, 64, 16), (2222, 7168, 32, 10), (2224, 7168, 32, 10), (2501, 1024, 512, 1),
                                     (3711, 4096, 64, 2), (3712, 4096, 64, 2), (4607, 7168, 12, 1), (4608, 7168, 12, 1),
                                     (257, 4096, 300, 8)])
def test_copies(gpu, quant, T, H, E, K):
    announce("permute rows quant=%d T=%d H=%d E=%d K=%d" % (quant, T, H, E, K))
    g = torch.Generator(device=gpu).manual_seed(T)
    x = torch.randn(T, H, generator=g, device=gpu).to(torch.bfloat16)
    ids = torch.rand(T, E, generator=g, device=gpu).topk(K, dim=1).indices.to(torch.int32)
    ids[torch.rand(T, K, generator=g, device=gpu) < 0.05] = -1
    once = cam.moe_dispatch_fused(x, torch.zeros(T, 1, dtype=torch.int32, device=gpu), 1, quant_mode=quant)
    d = cam.moe_dispatch_fused(x, ids, E, quant_mode=quant)
    t, k = (ids >= 0).nonzero(as_tuple=True)
    rows = d["slot_row"][t, k].long()
    assert torch.equal(rows.sort().values, torch.arange(len(t), device=gpu))
    raw = torch.int16 if quant == 0 else torch.int8
    for i in range(0, len(t), 4096):
        some = slice(i, i + 4096)
        assert torch.equal(d["recv_x"].view(raw)[rows[some]], once["recv_x"].view(raw)[t[some]])
        if quant:
            assert torch.equal(d["recv_x_scales"][rows[some]], once["recv_x_scales"][t[some]])
    info = d["expand_idx"].view(-1, 3)[rows]
    assert torch.equal(info, torch.stack([torch.zeros_like(t), t, k], dim=1).to(torch.int32))
