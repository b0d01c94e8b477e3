"""The GEMVs and the GEMMs that run in their place at few rows, both against sums in 64 bits over the operands that they multiply: each value within one rounding to bf16 and the f32 sum's
own error, and the GEMV as a whole no further off than the GEMM."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def distances(torch, x, w, alpha, got, other):
    """x, w, alpha: float64 operands; got: the GEMV's result, other: the GEMM's."""
    want, size, k = x @ w.T * alpha, x.abs() @ w.abs().T * alpha, x.shape[1]
    out = []
    for y in (got, other):
        off = (y.double() - want).abs()
        # half a bf16 step of what is rounded (8 bits), which the f32 sum has moved by at most (k + 1) 2^-24 of the terms' magnitudes; alpha's product rounds once more
        moved = (k + 1) * 2.0 ** -24 * size + 2.0 ** -24 * want.abs()
        assert (off <= 2.0 ** -8 * (want.abs() + moved) + moved).all()
        out.append((off.norm() / want.norm()).item())
    # Both round almost the same sums, so their distances are those of the rounding, about 2^-9 of a value. The f32 parts, k sums of 2^-24 each at most and of either sign, move that
    # by 2^-15 sqrt(k) of itself for one value and by the square root of their count less for all; four times that is allowed.
    assert out[0] <= out[1] * (1 + 4 * 2.0 ** -15 * (k / got.numel()) ** 0.5), out


@pytest.mark.parametrize("n,k", [(128, 128), (640, 2944), (5120, 2048), (1024, 5120), (384, 14464), (256, 17408)])
def test_fp8(n, k):
    import torch
    from ferrite_amd import fp4
    kern, ws = fp4.Kernels.load(), fp4.Workspace(64, k)
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    codes = (torch.randn((n, k), generator=gen, device="cuda") * 32).clamp(-448, 448).to(torch.float8_e4m3fn)
    host = fp4.HostLinear.fuse_fp8([("l", codes.view(torch.uint8).cpu().numpy(), 1.0 / (32.0 * k ** 0.5), 0.25)])
    lin, x = host.upload(), (torch.randn((64, k), generator=gen, device="cuda") * 4).to(torch.bfloat16)
    alpha = torch.from_numpy(host.alpha).cuda().double()
    for m in (1, 2, 8, 9, 16, 17, 24, 32, 33, 48, 64):
        y = [torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        for gemv in (1, 0):
            kern.set_option("gemv", gemv)
            lin.forward(kern, ws, y[1 - gemv], n, x, k, m)
        torch.cuda.synchronize()
        q = torch.from_numpy(ws.read_fp8(m, k)).view(torch.float8_e4m3fn).cuda().double()
        distances(torch, q, codes.double(), alpha, *y)


@pytest.mark.parametrize("n,k", [(64, 256), (640, 2816), (5120, 2048), (1024, 5120), (256, 17408)])
def test_bf16(n, k):
    import torch
    from ferrite_amd import bf16
    kern = bf16.Kernels.load()
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    w, x = (torch.randn((n, k), generator=gen, device="cuda") * k ** -0.5).to(torch.bfloat16), torch.randn((64, k), generator=gen, device="cuda").to(torch.bfloat16)
    for m in (1, 2, 8, 9, 16, 17, 24, 32, 33, 48, 64):
        y = [torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        bf16.forward(kern, y[0], n, x, k, w, m, dec=m)
        bf16.gemm(kern, y[1], n, x, k, w, m)
        torch.cuda.synchronize()
        distances(torch, x[:m].double(), w.double(), 1.0, *y)


@pytest.mark.parametrize("n,k", [(128, 256), (640, 2304), (1152, 4096), (12416, 2048), (1024, 5120), (256, 17408)])
def test_nvfp4(oracle, n, k):
    import torch
    from ferrite_amd import fp4, synth
    host = synth.fp4_linear(n, k, 11, input_scale=0.7)
    kern, ws, lin = fp4.Kernels.load(), fp4.Workspace(48, k), host.upload()
    x = torch.from_numpy((np.random.default_rng(k).normal(size=(48, k)) * 20).astype(np.float32)).cuda().to(torch.bfloat16)

    def values(codes, scales):  # e2m1 codes [r][k / 2] times e4m3 scales [r][k / 16]
        table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
        c = torch.from_numpy(codes).cuda().long()
        s = torch.from_numpy(np.ascontiguousarray(scales)).view(torch.float8_e4m3fn).cuda().double()
        return torch.stack((table[c & 15], table[c >> 4]), -1).reshape(len(codes), -1) * s.repeat_interleave(16, 1)

    w, alpha = values(host.codes, host.sf.reshape(n, k // 16)), torch.from_numpy(host.alpha).cuda().double()
    for m in (1, 2, 3, 5, 9, 16, 17, 33, 48):
        y = [torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        for gemv in (1, 0):
            kern.set_option("gemv", gemv)
            lin.forward(kern, ws, y[1 - gemv], n, x, k, m)
        torch.cuda.synchronize()
        codes, tiled = ws.read(m, k)
        distances(torch, values(codes, oracle.untile_scales(tiled, m, k // 16).reshape(m, k // 16)), w, alpha, *y)
