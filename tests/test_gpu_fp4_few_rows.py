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
