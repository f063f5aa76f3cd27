"""The counts per expert that moe_dispatch_prefill brings to the host: stored by the plan kernel into host memory of the
calling thread.  Several threads on streams of their own, one expert and the most there can be, ids that name no expert."""
import threading

import pytest
import torch

import umdk_original_amd as cam
from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (37, 2, 512), (1500, 3, 17)])
def test_prefill_counts_from_several_threads(gpu, T, K, E):
    announce("prefill counts T=%d K=%d E=%d" % (T, K, E))
    wrong = []

    def work(seed):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            g = torch.Generator().manual_seed(seed)
            for i in range(20):
                ids = torch.randint(-1 if i % 2 else 0, E, (T, K), generator=g)
                x = torch.randn(T, 1024, generator=g).bfloat16().to(gpu)
                w = torch.rand(T, K, device=gpu)
                dev = ids.to(torch.int32).to(gpu)
                want = torch.bincount(ids[ids >= 0].flatten(), minlength=E)
                for fn in (torch.ops.umdk_cam_op_lib.moe_dispatch_prefill, cam.moe_dispatch_prefill):
                    r, e, in_rank = cam.get_dispatch_layout(dev, E, 1)
                    rows, info, _, counts = fn(x, dev, w, r, in_rank, e, 0, "", 0, 1)
                    if not torch.equal(counts, want) or rows.size(0) not in (int(want.sum()), max(int(want.sum()), 1)):
                        wrong.append((seed, i))
                    elif want.sum() > 0 and not torch.equal(rows, x[info.view(-1, 3)[:, 1].long()]):
                        wrong.append((seed, i, "rows"))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
