"""The FP8 GEMV of few rows: a row's bits whatever the batch, the width of a program and the weights' layout; against the GEMM over the same codes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# One step of K for one wavefront alone, quarters of unequal length, one step more than stages; the last program partly past n, columns of two weight tiles; K past the line
# of 40 rows; programs of fewer columns than their octets
@pytest.mark.parametrize("n,k", [(128, 128), (384, 640), (640, 2944), (256, 17408), (4992, 640)])
def test_every_form_gives_the_same_bits(n, k):
    import torch
    from ferrite_amd import fp4
    kern = fp4.Kernels.load()
    rng = np.random.default_rng(n + k)
    codes = torch.from_numpy(rng.normal(size=(n, k)).astype(np.float32) * 32).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    host = fp4.HostLinear.fuse_fp8([("l", codes.numpy(), 1.0 / (32.0 * k ** 0.5), 0.25)])
    host.alpha[:] = host.alpha * np.linspace(0.5, 2.0, n).astype(np.float32)
    lin = host.upload()
    dc, da = codes.cuda(), torch.from_numpy(host.alpha).cuda()
    view = fp4.PromptLinear.from_view("v", n, k, dc, None, da, host.g)
    x = torch.from_numpy(rng.normal(size=(64, k)).astype(np.float32) * 4).cuda().to(torch.bfloat16)
    res = torch.from_numpy(rng.normal(size=(64, n)).astype(np.float32)).cuda().to(torch.bfloat16)
    ws = fp4.Workspace(64, k)

    def run(l, m, cols=0, gemv=1, r=None):
        kern.set_option("gemv_cols", cols)
        kern.set_option("gemv", gemv)
        try:
            y = torch.full((m + 1, n + 8), 5.0, dtype=torch.bfloat16, device="cuda")
            l.forward(kern, ws, y, n + 8, x, k, m, res=r)
            torch.cuda.synchronize()
        finally:
            kern.set_option("gemv_cols", 0)
            kern.set_option("gemv", 1)
        assert (y[m] == 5.0).all() and (y[:, n:] == 5.0).all()
        return y[:m, :n]

    most = 64 if k <= 14336 else 40
    want = run(lin, most)
    for m in (1, 8, 9, 16, 17, 33, most):
        for cols in (0, 8, 16, 24, 32, 40, 48, 72):
            assert torch.equal(run(lin, m, cols).view(torch.int16), want[:m].view(torch.int16)), (m, cols)
        assert torch.equal(run(view, m).view(torch.int16), want[:m].view(torch.int16))
        big = torch.zeros((m, n + 8), dtype=torch.bfloat16, device="cuda")
        big[:, :n] = res[:m]
        assert torch.equal(run(lin, m, r=big), (want[:m].float() + res[:m].float()).to(torch.bfloat16))
        a, b = want[:m].double(), run(lin, m, gemv=0).double()  # exact products, f32 sums in another order
        assert ((a - b).abs() <= b.abs() / 128 + b.abs().amax(dim=1, keepdim=True) * 1e-6).all()
    a, b = run(lin, 64).double()[:most], want.double()  # past the line: the GEMM
    assert ((a - b).abs() <= b.abs() / 128 + b.abs().amax(dim=1, keepdim=True) * 1e-6).all()
