"""Gate, up and SwiGLU of decode rows over plain bf16 weights in one launch: the bits of two GEMVs and fe_silu_mul."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# One step a wavefront (fewer than stages in flight), fewer steps in all than stages, as many as stages, many; the last program partly past the columns; every row form and
# width of a program, also of fewer columns than its octets; rows by their count and as decode rows, prompt rows that are few enough and one more
@pytest.mark.parametrize("hidden,inter", [(256, 320), (512, 1216), (1792, 576), (2048, 1344), (5120, 192), (256, 5184)])
def test_one_launch_gives_the_bits_of_three(hidden, inter):
    import torch
    from ferrite_amd import bf16, route
    kern = bf16.Kernels.load()
    gen = torch.Generator(device="cuda").manual_seed(hidden + inter)

    def rand(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)

    g, u, dn = rand(inter, hidden, scale=2 / hidden ** 0.5), rand(inter, hidden, scale=2 / hidden ** 0.5), rand(hidden, inter, scale=inter ** -0.5)
    ctx = route.LinCtx()
    ctx.set_bf16(kern)
    gate_up = route.Proj([(route.Linear("gate", inter, hidden, w=g), [inter]), (route.Linear("up", inter, hidden, w=u), [inter])])
    down = route.Linear("down", hidden, inter, w=dn)
    for m, dec in ((1, 0), (2, 0), (8, 0), (9, 0), (16, 0), (17, 17), (20, 0), (32, 0), (33, 0), (33, 40), (48, 48), (64, 64), (65, 65), (20, 4)):
        xn = rand(m, hidden)
        xn[0, 3], xn[m - 1, hidden - 1] = float("inf"), float("nan")
        big, act = rand(m, 2 * inter), torch.zeros((m, inter), dtype=torch.bfloat16, device="cuda")
        yg, yu = torch.empty((m, inter), dtype=torch.bfloat16, device="cuda"), torch.empty((m, inter), dtype=torch.bfloat16, device="cuda")
        want = torch.empty_like(act)
        kern.set_option("nc", -1)
        bf16.forward(kern, yg, inter, xn, hidden, g, m, dec=dec)
        bf16.forward(kern, yu, inter, xn, hidden, u, m, dec=dec)
        route.silu_mul(want, yg.data_ptr(), yu.data_ptr(), inter, inter, m)
        ctx.dec = dec
        for nc in (-1, 8, 16, 24, 32, 40, 48, 72):
            kern.set_option("nc", nc)
            act.fill_(3.0)
            x = torch.zeros((m, hidden), dtype=torch.bfloat16, device="cuda")
            route.mlp_forward(ctx, gate_up, down, x, xn, big, act, m, hidden, inter)
            torch.cuda.synchronize()
            assert torch.equal(act.view(torch.int16), want.view(torch.int16)), (m, dec, nc)
    kern.set_option("nc", -1)


def test_act_over_the_input(dim=512):
    """act in the input's memory: what the separate launches give, which read all of the input first."""
    import torch
    from ferrite_amd import bf16, route
    kern = bf16.Kernels.load()
    w = [(torch.randn((dim, dim), device="cuda") * 0.05).to(torch.bfloat16) for _ in range(3)]
    ctx = route.LinCtx()
    ctx.set_bf16(kern)
    gate_up = route.Proj([(route.Linear("gate", dim, dim, w=w[0]), [dim]), (route.Linear("up", dim, dim, w=w[1]), [dim])])
    down = route.Linear("down", dim, dim, w=w[2])
    xn = torch.randn((4, dim), device="cuda").to(torch.bfloat16)
    got = []
    for over in (False, True):
        xi, big = xn.clone(), torch.empty((4, 2 * dim), dtype=torch.bfloat16, device="cuda")
        x = torch.zeros((4, dim), dtype=torch.bfloat16, device="cuda")
        route.mlp_forward(ctx, gate_up, down, x, xi, big, xi if over else torch.empty_like(xi), 4, dim, dim)
        torch.cuda.synchronize()
        got.append(x.view(torch.int16).cpu().numpy())
    assert np.array_equal(*got)
