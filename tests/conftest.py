import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "comfyui-hy-nomas_amd")
for p in (ROOT, PKG):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


@pytest.fixture(scope="session")
def dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def seeded(seed=0):
    import torch

    return torch.Generator().manual_seed(seed)


def recorded_kernels(call):
    """(workgroups, threads of one) of each kernel that a call records into a graph, in order."""
    import ctypes

    import torch
    from hy_nomas import _lib

    class Params(ctypes.Structure):  # hipKernelNodeParams
        _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                    ("grid", ctypes.c_uint32 * 3), ("args", ctypes.c_void_p), ("lds", ctypes.c_uint)]

    call()
    torch.cuda.synchronize()
    graph, n, lib = torch.cuda.CUDAGraph(keep_graph=True), ctypes.c_size_t(), _lib.lib()
    with torch.cuda.graph(graph):
        call()
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    assert lib.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes, out = (ctypes.c_void_p * n.value)(), []
    assert lib.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    for node in nodes:
        p = Params()
        assert lib.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        out.append((p.grid[0] * p.grid[1] * p.grid[2], p.block[0] * p.block[1] * p.block[2]))
    return out
