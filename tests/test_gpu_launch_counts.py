"""What the queries say about the launches of a call, against the kernels that a capture of the call records."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def kernels_recorded(torch, call):
    """Kernel nodes of a captured call."""
    hip = C.CDLL("libamdhip64.so")
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        call()
    raw, n = C.c_void_p(graph.raw_cuda_graph()), C.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, C.byref(n)) == 0
    nodes, kind, kernels = (C.c_void_p * n.value)(), C.c_int(0), 0
    assert hip.hipGraphGetNodes(raw, nodes, C.byref(n)) == 0
    for node in nodes:
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        kernels += kind.value == 0  # hipGraphNodeTypeKernel
    return kernels


# 1024: column blocks shared by several programs; 256: every block lies in one program's run, so no launch finishes them
@pytest.mark.parametrize("rows", [1, 8, 16, 17, 40, 64])
@pytest.mark.parametrize("k,wide", [(1024, 3), (256, 2)])
def test_group_launches(rows, k, wide):
    import torch
    from ferrite_amd import exl3, synth
    kern = exl3.Kernels.load()
    lins = [exl3.Linear.new(kern, exl3.DeviceExl3.upload_strips(synth.exl3_tensor(k, n, 4, n)), 256) for n in (384, 256)]
    ws = exl3.Workspace(lins, 64)
    x = torch.from_numpy(synth.activations(rows, k, 3).view(np.int16)).cuda()
    ys = [torch.zeros((rows, l.n), dtype=torch.bfloat16, device="cuda") for l in lins]
    call = lambda: exl3.forward_group(lins, x, exl3.Dtype.Bf16, ys, exl3.Dtype.Bf16, rows, ws)
    got = exl3.forward_group_launches(lins, rows, ws)
    assert got == kernels_recorded(torch, call) and (rows <= 16 or got == wide)
