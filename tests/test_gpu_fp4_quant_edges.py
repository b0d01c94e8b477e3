"""The NVFP4 quantizer where g / (block scale) is zero, not finite or not a number: codes and block scales as the oracle's, by its own launch and inside the GEMV."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [1.0, 1e-38, 1e-44, 0.0, float("inf"), float("nan")])
@pytest.mark.parametrize("inside", [0, 32768])
def test_infinities_against_every_multiplier(oracle, g, inside):
    import torch
    from ferrite_amd import fp4, synth
    n, k, m = 128, 256, 2
    host = synth.fp4_linear(n, k, 1)
    kern, ws = fp4.Kernels.load(), fp4.Workspace(m, k)
    dev = [torch.from_numpy(a).cuda() for a in (host.codes, host.sf, host.alpha)]
    lin = fp4.PromptLinear.from_view("view", n, k, *dev, g)
    x = np.zeros((m, k), np.float32)
    x[:] = np.random.default_rng(3).normal(size=(m, k)).astype(np.float32) * 10
    x[0, :16:2], x[0, 1:16:4] = np.inf, -np.inf  # infinities; one among finite values; with a NaN; no value at all; zeros; the smallest and the largest
    x[0, 20], x[0, 40], x[0, 41], x[1, :16], x[1, 16:32], x[1, 32:48], x[1, 50] = np.inf, -np.inf, np.nan, np.nan, 0.0, 1e-40, 3e38
    xd = torch.from_numpy(x).cuda().to(torch.bfloat16)
    kern.set_option("gemv_quant", inside)
    lin.forward(kern, ws, torch.zeros((m, n), dtype=torch.bfloat16, device="cuda"), n, xd, k, m)
    torch.cuda.synchronize()
    codes, tiled = ws.read(m, k)
    want, sf = oracle.quant_fp4(xd.view(torch.int16).cpu().numpy().view(np.uint16), g)
    assert np.array_equal(oracle.untile_scales(tiled, m, k // 16).reshape(m, k // 16), sf)
    # (a NaN that the product makes has no sign of its own: a code of magnitude 0 is one, whatever its sign)
    plain = lambda c: np.where(c & 7, c, 0)
    for a, b in ((codes & 15, want & 15), (codes >> 4, want >> 4)):
        assert np.array_equal(plain(a), plain(b))


@pytest.mark.parametrize("n,k,m", [(128, 256, 1), (640, 2304, 3), (256, 17408, 1), (1152, 4096, 8)])
def test_the_option_says_where_the_quantizer_runs(n, k, m):
    """One kernel where the GEMV's programs quantize, two with the quantizer's own launch: the two sides that the comparisons of bits set against each other."""
    import torch
    from ferrite_amd import fp4, synth
    from test_gpu_launch_counts import kernels_recorded
    kern, ws, lin = fp4.Kernels.load(), fp4.Workspace(m, k), synth.fp4_linear(n, k, 1).upload()
    x, y = torch.zeros((m, k), dtype=torch.bfloat16, device="cuda"), torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
    for limit, kernels in ((32768, 1), (0, 2)):
        kern.set_option("gemv_quant", limit)
        assert kernels_recorded(torch, lambda: lin.forward(kern, ws, y, n, x, k, m)) == kernels
