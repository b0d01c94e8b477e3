"""The epilogues of the prompt GEMMs. With a residual: bf16(bf16(sum) + res) of the very sums that the call without one rounds, bit for bit, in every tile (whole ones, rows and columns that
end inside one), in place and from another buffer, with rows that lie further apart than they are wide; nothing is written past a row's columns or past the last row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _calls(torch, form, n, k, m, x):
    """(kernels, y, ldy, res -> None)"""
    from ferrite_amd import bf16, fp4, synth
    if form == "bf16":
        kern = bf16.Kernels.load()
        w = (torch.from_numpy(np.random.default_rng(7).normal(size=(n, k)).astype(np.float32)) / k ** 0.5).to(torch.bfloat16).cuda()
        return kern, lambda y, ldy, res: bf16.gemm(kern, y, ldy, x, k, w, m, res=res)
    kern = fp4.Kernels.load()
    lin = (synth.fp4_linear(n, k, 5) if form == "nvfp4" else synth.fp8_linear(n, k, 6, input_scale=0.05)).upload()
    ws = fp4.Workspace(m, k)
    ws.lin = lin
    return kern, lambda y, ldy, res: lin.forward(kern, ws, y, ldy, x, k, m, res=res)


# (tile 1: 256 x 256, 2: 128 x 256, 3: 128 x 128, 4..6: 224, 192, 160 x 256; bf16's columns may end at any multiple of 8, its rows be 8-byte aligned only)
@pytest.mark.parametrize("form,m,n,k,gap", [("bf16", 256, 512, 256, 0), ("bf16", 129, 264, 256, 4), ("bf16", 301, 776, 512, 12), ("nvfp4", 256, 512, 512, 0),
                                            ("nvfp4", 143, 384, 512, 8), ("nvfp4", 337, 640, 256, 64), ("fp8", 256, 512, 512, 0), ("fp8", 143, 384, 512, 8), ("fp8", 337, 640, 256, 64)])
def test_residual(form, m, n, k, gap):
    import torch
    from ferrite_amd import synth
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda().view(torch.bfloat16)
    x, old = dev(synth.activations(m, k, 3)), dev(synth.activations(m, n, 4))
    kern, run = _calls(torch, form, n, k, m, x)
    ldy = n + gap

    def call(in_place, adds):
        y = torch.full((m + 1, ldy), 1.5, dtype=torch.bfloat16, device="cuda")
        res = y if in_place else torch.full((m + 1, ldy), 2.5, dtype=torch.bfloat16, device="cuda")
        if adds:
            res[:m, :n] = old
        run(y, ldy, res if adds else None)
        torch.cuda.synchronize()
        assert (y[m:] == 1.5).all() and (y[:, n:] == 1.5).all(), (form, in_place)
        return y[:m, :n].clone()

    settings = [("gemm_tile", t) for t in (1, 2, 3, 4, 5, 6)] + ([] if form == "bf16" else [("gemm_sk", 2)])
    try:
        kern.set_option("gemm_splits", 1)
        kern.set_option("gemm_pieces", 1)
        for name, value in settings:
            kern.set_option("gemm_tile", value if name == "gemm_tile" else 1)
            if name == "gemm_sk":
                kern.set_option("gemm_sk", value)
            want = (call(False, False).float() + old.float()).to(torch.bfloat16)
            for in_place in (False, True):
                assert torch.equal(call(in_place, True), want), (name, value, in_place)
    finally:
        kern.set_option("gemm_splits", 8)
        kern.set_option("gemm_tile", 0)
        kern.set_option("gemm_pieces", 0)
        if form != "bf16":
            kern.set_option("gemm_sk", 1)


@pytest.mark.parametrize("inter,k,m", [(128, 512, 70), (640, 256, 300), (384, 512, 256)])
def test_nvfp4_swiglu_of_exact_sums(inter, k, m):
    """The NVFP4 SwiGLU front on operands whose sums are exact in f32 in any order: the tiles' epilogue (registers, lane by lane) and the reduce launch of cut tiles (rows through
    LDS) leave the same codes, scales and fp16 operand, the last seen through the linear that reads it."""
    import torch
    from ferrite_amd import fp4, synth
    kern = fp4.Kernels.load()
    rng = np.random.default_rng(11)
    part = lambda n, kk: (rng.integers(0, 256, (n, kk // 2), dtype=np.uint8), np.full((n, kk // 16), 0x38, np.uint8))  # any codes, scales of 1
    g, u, d = part(inter, k), part(inter, k), part(256, inter)
    fused = fp4.HostLinear.fuse([("gate", *g, 2.0 ** -7, 1.0), ("up", *u, 2.0 ** -7, 1.0)])
    sw = fused.into_swiglu().upload()
    down = fp4.HostLinear.fuse([("down", *d, 2.0 ** -5, 1.0)]).upload()
    x = rng.choice([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], (m, k)) * rng.choice([-1.0, 1.0], (m, k))
    x[:, ::16] = 6.0  # (every block's scale is 1)
    x = torch.from_numpy(x).to(torch.bfloat16).cuda()
    ws, act = fp4.Workspace(m, k), fp4.Workspace(m, inter)

    def call(tile, pieces):
        kern.set_option("gemm_tile", tile)
        kern.set_option("gemm_pieces", pieces)
        sw.forward_swiglu(kern, ws, act, x, k, m, 0.5)
        kern.set_option("gemm_tile", 1)
        y = torch.zeros((m, 256), dtype=torch.bfloat16, device="cuda")
        down.gemm(kern, act, y, 256, m)
        torch.cuda.synchronize()
        return [a.copy() for a in act.read(m, inter)] + [y.view(torch.int16).cpu().numpy()]

    try:
        kern.set_option("gemm_splits", 1)
        want = call(2, 2)  # cut: the reduce launch
        assert np.unique(want[0]).size > 64 and np.unique(want[1]).size > 4
        for tile, pieces in [(1, 1), (2, 1), (3, 1), (3, 2), (4, 1), (5, 1), (6, 1)]:
            for a, b in zip(call(tile, pieces), want):
                assert np.array_equal(a, b), (tile, pieces)
    finally:
        kern.set_option("gemm_splits", 8)
        kern.set_option("gemm_tile", 0)
        kern.set_option("gemm_pieces", 0)
