"""The GEMMs' epilogues with a residual: bf16(bf16(sum) + res) of the very sums that the call without one rounds, bit for bit, in every tile (whole ones, rows and columns that
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
