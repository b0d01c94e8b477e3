"""NVFP4 at 17 to 65 rows: one pass of the GEMV up to 48, the GEMM beyond; both weight layouts the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(128, 256), (640, 1280), (1152, 2304)])
def test_rows_at_the_edges_of_a_pass(n, k):
    import torch
    from ferrite_amd import fp4, synth
    kern = fp4.Kernels.load()
    host = synth.fp4_linear(n, k, 3, input_scale=0.7)
    lin = host.upload()
    view = fp4.PromptLinear.from_view("view", n, k, torch.from_numpy(host.codes).cuda(), torch.from_numpy(host.sf).cuda(), torch.from_numpy(host.alpha).cuda(), host.g)
    x = torch.from_numpy((np.random.default_rng(n).normal(size=(65, k)) * 20).astype(np.float32)).cuda().to(torch.bfloat16)
    ws = fp4.Workspace(65, k)

    def run(l, m, strips=1):
        kern.set_option("gemv_strips", strips)
        y = torch.full((m + 1, n), 5.0, dtype=torch.bfloat16, device="cuda")
        l.forward(kern, ws, y, n, x, k, m)
        torch.cuda.synchronize()
        assert (y[m] == 5.0).all()
        return y[:m]

    whole = run(lin, 65)
    for m in (17, 33, 48, 49, 64):
        got, passes = run(lin, m), run(lin, m, strips=0)
        assert torch.equal(got.view(torch.int16), run(view, m).view(torch.int16))
        assert torch.equal(passes.view(torch.int16), run(view, m, strips=0).view(torch.int16))
        assert m > 48 or torch.equal(got.view(torch.int16), passes.view(torch.int16))
        for other in (passes, whole[:m]):  # exact products, f32 sums in another order: a bf16 step where a sum lies between two, f32's own error where one nearly cancels
            a, b = got.double(), other.double()
            assert ((a - b).abs() <= b.abs() / 128 + b.abs().amax(dim=1, keepdim=True) * 1e-6).all()


# one K split and several; the last weight tile's columns; groups of rows partly empty; both layouts; a linear whose rows from 33 on take the GEMM
@pytest.mark.parametrize("inter,k", [(128, 256), (640, 1280), (2304, 4096)])
def test_swiglu_in_the_gemv_gives_the_bits_of_its_parts(inter, k):
    import ctypes as C
    import torch
    from ferrite_amd import _lib, fp4, route, synth
    kern = fp4.Kernels.load()
    a, b = (synth.fp4_linear(inter, k, seed, input_scale=0.7) for seed in (3, 4))
    fused = fp4.HostLinear.fuse([("gate", a.codes, a.sf, 0.01, 1.4), ("up", b.codes, b.sf, 0.02, 1.4)])
    inter_host = fused.into_swiglu()
    down = synth.fp4_linear(128, inter, 5, input_scale=0.9).upload()
    plain, lin = fused.upload(), inter_host.upload()
    view = fp4.PromptLinear.from_view("view", 2 * inter, k, torch.from_numpy(inter_host.codes).cuda(), torch.from_numpy(inter_host.sf).cuda(),
                                      torch.from_numpy(inter_host.alpha).cuda(), inter_host.g)
    x = torch.from_numpy((np.random.default_rng(k).normal(size=(48, k + 8)) * 20).astype(np.float32)).cuda().to(torch.bfloat16)
    x[0, 3], x[16, 5] = float("inf"), float("nan")
    kern.set_option("gemv_strips", 0)  # the parts through the GEMV over weight tiles at every row count

    def left(ws, m):
        torch.cuda.synchronize()
        ptr, op = C.c_uint64(), np.empty((m, inter), np.uint16)
        _lib.check(_lib.lib().fe_fp4_workspace_operand(ws.h, C.byref(ptr)))
        _lib.check(_lib.lib().fe_hip_memcpy_dtoh(op.ctypes.data_as(C.c_void_p), ptr.value, op.nbytes))
        return (*ws.read(m, inter), op)

    try:
        for m in (1, 16, 17, 32, 33, 48):
            ws, want, act = fp4.Workspace(m, max(k, inter)), fp4.Workspace(m, inter), torch.empty((m, inter), dtype=torch.bfloat16, device="cuda")
            big = torch.empty((m, 2 * inter), dtype=torch.bfloat16, device="cuda")
            plain.forward(kern, ws, big, 2 * inter, x, k + 8, m)
            route.silu_mul(act, big.data_ptr(), big.data_ptr() + 2 * inter, 2 * inter, inter, m)
            down.quantize(kern, want, act, inter, m)
            for l in (lin, view):
                got = fp4.Workspace(m, inter)
                l.forward_swiglu(kern, ws, got, x, k + 8, m, down.g)
                g, w = left(got, m), left(want, m)
                assert np.array_equal(g[0], w[0]) and np.array_equal(g[2], w[2]), m
                rows = range(m)
                assert np.array_equal(_scales(g[1], rows, inter), _scales(w[1], rows, inter)), m
    finally:
        kern.set_option("gemv_strips", 1)


def _scales(tiled, rows, k):
    """The block scales of the rows that exist: the tiles also hold rows that no call writes."""
    import oracle
    return oracle.untile_scales(tiled, max(rows) + 1, k // 16)
