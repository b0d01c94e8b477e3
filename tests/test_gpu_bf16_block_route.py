"""Which launches an MLP block over plain bf16 weights takes: gate, up and SwiGLU in one GEMV, the GEMM over interleaved weights, or the separate linears. Told apart by whether
`big`, which only the separate linears write, is still what it was, and by the bits of act, which differ between the GEMV's and the GEMM's order of sums."""
import pytest

pytestmark = pytest.mark.gpu

PAIR, GEMM, PARTS = "one GEMV", "GEMM with SwiGLU", "separate linears"


# rows, decode rows, hidden, inter, interleaved weights given, what the decode rows (all rows where dec is None) and the prompt rows take
@pytest.mark.parametrize("rows,dec,hidden,inter,fused,first,rest", [
    (1, None, 5120, 320, False, PAIR, PAIR), (16, None, 5120, 320, True, PAIR, PAIR),
    (17, None, 2048, 320, True, PAIR, PAIR), (32, None, 2048, 1344, True, PAIR, PAIR), (32, None, 5120, 12288, True, PAIR, PAIR), (20, 4, 2048, 320, True, PAIR, PAIR),
    (17, None, 5120, 320, True, GEMM, GEMM), (32, None, 5120, 320, True, GEMM, GEMM), (26, None, 7168, 320, True, GEMM, GEMM),  # the GEMM with SwiGLU is ahead of it
    (26, None, 5120, 320, False, PAIR, PAIR), (32, None, 5120, 320, False, PAIR, PAIR),  # no interleaved weights: against three launches
    (33, None, 5120, 320, True, GEMM, GEMM), (33, None, 5120, 320, False, PARTS, PARTS),
    (23, None, 14848, 64, False, PARTS, PARTS), (23, None, 14848, 64, True, GEMM, GEMM),  # the linears' own line
    (64, 64, 5120, 320, True, PAIR, PAIR), (65, 65, 5120, 320, False, PARTS, PARTS), (40, 4, 5120, 320, True, PAIR, GEMM),
])
def test_a_block_takes(rows, dec, hidden, inter, fused, first, rest):
    import torch
    from ferrite_amd import bf16, route
    kern = bf16.Kernels.load()
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden + inter)

    def rand(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)

    g, u, dn = rand(inter, hidden, scale=2 / hidden ** 0.5), rand(inter, hidden, scale=2 / hidden ** 0.5), rand(hidden, inter, scale=inter ** -0.5)
    wi = bf16.interleave_gu(kern, g, u)
    ctx = route.LinCtx()
    ctx.set_bf16(kern)
    ctx.dec = d = dec or 0
    gate_up = route.Proj([(route.Linear("gate", inter, hidden, w=g), [inter]), (route.Linear("up", inter, hidden, w=u), [inter])])
    xn, x = rand(rows, hidden), torch.zeros((rows, hidden), dtype=torch.bfloat16, device="cuda")
    empty = lambda: torch.empty((rows, inter), dtype=torch.bfloat16, device="cuda")

    def parts(decode_rows):
        yg, yu, out = empty(), empty(), empty()
        bf16.forward(kern, yg, inter, xn, hidden, g, rows, dec=decode_rows)
        bf16.forward(kern, yu, inter, xn, hidden, u, rows, dec=decode_rows)
        route.silu_mul(out, yg.data_ptr(), yu.data_ptr(), inter, inter, rows)
        return out

    want = {PAIR: parts(rows), PARTS: parts(d), GEMM: empty()}
    bf16.gemm_swiglu(kern, want[GEMM], xn, hidden, wi, rows)
    if GEMM in (first, rest):
        assert not torch.equal(want[PAIR].view(torch.int16), want[GEMM].view(torch.int16))  # or the bits would tell nothing
        if d:
            bf16.gemm_swiglu(kern, want[GEMM][d:], xn[d:], hidden, wi, rows - d)
    big, act = torch.full((rows, 2 * inter), 3.0, dtype=torch.bfloat16, device="cuda"), torch.full((rows, inter), 3.0, dtype=torch.bfloat16, device="cuda")
    route.mlp_forward(ctx, gate_up, route.Linear("down", hidden, inter, w=dn), x, xn, big, act, rows, hidden, inter, swiglu_w=wi if fused else None)
    torch.cuda.synchronize()
    assert bool((big == 3.0).all()) == (PARTS not in (first, rest))
    assert torch.equal(act[:d].view(torch.int16), want[first][:d].view(torch.int16)) and torch.equal(act[d:].view(torch.int16), want[rest][d:].view(torch.int16))
