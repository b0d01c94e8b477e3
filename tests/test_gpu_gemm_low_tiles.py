"""The prompt GEMMs on tiles of 224, 192 and 160 rows (option gemm_tile 4, 5, 6) against the 256 x 256 form: K uncut the same bits in every
weight form and epilogue (same k order), K cut within the rounding of the result, rows past m untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LOW = (4, 5, 6)


def nvfp4_swiglu(k, n, m):
    """(kernels, run() -> codes and scales) of the fused front of a gate|up pair of n / 2 columns each."""
    import torch
    from ferrite_amd import fp4, synth
    kern = fp4.Kernels.load()
    inter = n // 2
    g, u = synth.fp4_linear(inter, k, 1, name="gate"), synth.fp4_linear(inter, k, 2, name="up")
    fused = fp4.HostLinear.fuse([("gate", g.codes, g.sf, 1.0, 1.0), ("up", u.codes, u.sf, 1.0, 1.0)])
    fused.alpha[:] = fused.alpha * np.float32(0.02)
    sw = fused.into_swiglu().upload()
    ws, act = fp4.Workspace(m, k), fp4.Workspace(m, inter)
    x = torch.from_numpy(synth.activations(m, k, 9).view(np.int16)).cuda()

    def run():
        sw.forward_swiglu(kern, ws, act, x, k, m, 0.5)
        torch.cuda.synchronize()
        return [a.copy() for a in act.read(m, inter)]
    return kern, run


# the last tile full, one row over, one group of 16 rows, a group and a row; one, two and three tiles; an odd count of 128-column tiles
@pytest.mark.parametrize("m,n,k", [(97, 512, 512), (160, 384, 256), (225, 768, 1024), (400, 512, 1280), (481, 1152, 512)])
def test_low_tiles(m, n, k):
    import torch
    from test_gpu_gemm_tiles import forms
    for name, (kern, run, cols) in forms(torch, k, n, m).items():
        if name.startswith("trellis") or name == "kept":
            continue

        def call(tile, splits):
            kern.set_option("gemm_tile", tile)
            kern.set_option("gemm_splits", splits)
            y = torch.full((m + 1, cols), 1.5, dtype=torch.bfloat16, device="cuda")
            run(y)
            torch.cuda.synchronize()
            assert (y[m:] == 1.5).all(), name
            return y[:m].clone()

        try:
            want = call(1, 1)
            rms = want.float().square().mean().sqrt()
            for tile in LOW:
                assert torch.equal(call(tile, 1), want), (name, tile)
                got = call(tile, 8).float()  # (few tiles: each in as many pieces as K has eighths of a kilobyte)
                # (a step of the sum before the residual or the SwiGLU product shows in a smaller result)
                assert ((got - want.float()).abs() <= want.float().abs() / 64 + 2e-2 * rms).all(), (name, tile)
                assert (got != want.float()).float().mean() < 0.05, (name, tile)
        finally:
            kern.set_option("gemm_splits", 8)
            kern.set_option("gemm_tile", 0)


@pytest.mark.parametrize("m,n,k", [(225, 768, 1024), (400, 256, 512)])
def test_low_tiles_of_the_nvfp4_swiglu_front(m, n, k):
    kern, run = nvfp4_swiglu(k, n, m)
    try:
        kern.set_option("gemm_splits", 1)
        kern.set_option("gemm_tile", 1)
        codes, sf = run()
        for tile in LOW:
            kern.set_option("gemm_tile", tile)
            kern.set_option("gemm_splits", 1)
            c, s = run()
            assert np.array_equal(c, codes) and np.array_equal(s, sf), tile
            kern.set_option("gemm_splits", 8)
            c, s = run()
            assert (c != codes).mean() < 1e-2 and (s != sf).mean() < 5e-3, tile
    finally:
        kern.set_option("gemm_splits", 8)
        kern.set_option("gemm_tile", 0)
