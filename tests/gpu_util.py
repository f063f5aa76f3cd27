"""Helpers shared by the GPU parity tests (which call the HIP path through the C ABI)."""
import ctypes

import numpy as np
import torch

from umdk_original_amd import synth


def announce(msg):
    # Names the case before any GPU work so a lost box still tells which test was running.
    print("[gpu-case] " + msg, flush=True)


def to_np(t):
    if t.dtype == torch.bfloat16:
        return synth.bf16_bits(t.cpu())
    return t.cpu().numpy()


def plan_oracle(oracle, idx_np, E, skip_out_of_range=False):
    T = idx_np.shape[0]
    _, cnt, _ = oracle.layout(idx_np, E, 1, skip_out_of_range=skip_out_of_range)
    off, trip = oracle.offsets(cnt, T)
    pos = oracle.send_token_idx(idx_np, E)
    return cnt, off, pos, trip


def assert_bits_equal(got, want, what):
    got = np.asarray(got)
    want = np.asarray(want)
    assert got.shape == want.shape, (what, got.shape, want.shape)
    if not np.array_equal(got, want):
        bad = np.argwhere(got != want)
        raise AssertionError("%s: %d of %d elements differ; first at %s: got %s want %s" % (
            what, len(bad), got.size, bad[0].tolist(), got[tuple(bad[0])], want[tuple(bad[0])]))


def _recorded(call):
    """The runtime, the graph that a call records and its nodes; nothing of it runs."""
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    hip = ctypes.CDLL(path)
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        keep = call()
    raw, n = ctypes.c_void_p(g.raw_cuda_graph()), ctypes.c_size_t()
    assert keep is not None and hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    return hip, g, nodes


def recorded_kernels(call):
    """How many launches a call records."""
    return len(_recorded(call)[2])


class _KernelNode(ctypes.Structure):   # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint * 3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def recorded_names(call):
    """The mangled names of the kernels that a call records."""
    hip, g, nodes = _recorded(call)
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    names = []
    for node in nodes:
        p = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        names.append(hip.hipKernelNameRefByPtr(ctypes.c_void_p(p.func), None).decode())
    return names
