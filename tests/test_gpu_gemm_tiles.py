"""The GEMMs on their smaller output tiles (128 x 256 and 128 x 128, options gemm_tile and gemm_pieces) against the 256 x 256
form, which other tests hold to the oracle: K uncut the same bits in every weight form and epilogue (same k order), K cut
within the rounding of the result, rows past m untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def forms(torch, k, n, m):
    """name -> (kernels, run(y [m + 1][n] bf16), columns) of every GEMM; run writes rows 0 .. m - 1."""
    from ferrite_amd import bf16, exl3, fp4, synth
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda()
    xb = synth.activations(m, k, 3)
    x = dev(xb).view(torch.bfloat16)
    res = dev(synth.activations(m, n, 4)).view(torch.bfloat16)
    out = {}
    x3 = exl3.Kernels.load()
    for bits in (2, 3, 5, 8):
        lin = exl3.Linear.new(x3, exl3.DeviceExl3(synth.exl3_tensor(k, n, bits, bits), bits != 3), 256)
        ws = exl3.Workspace([lin], m)
        dt = exl3.Dtype.Bf16Add if bits == 5 else exl3.Dtype.Bf16
        out["trellis %d" % bits] = (x3, lambda y, l=lin, w=ws, d=dt: l.forward(x, exl3.Dtype.Bf16, y, d, m, w), n)
    kept = exl3.Linear.new(x3, exl3.DeviceExl3(synth.exl3_tensor(k, n, 4, 4), True), 256)
    kept.keep_decoded()
    kws = exl3.Workspace([kept], m)
    out["kept"] = (x3, lambda y: kept.forward(x, exl3.Dtype.Bf16, y, exl3.Dtype.Bf16, m, kws), n)
    k4 = fp4.Kernels.load()
    ws4 = fp4.Workspace(m, k)
    for name, host in (("nvfp4", synth.fp4_linear(n, k, 5)), ("fp8", synth.fp8_linear(n, k, 6, input_scale=0.05))):
        l4 = host.upload()
        out[name] = (k4, lambda y, l=l4: l.forward(k4, ws4, y, n, x, k, m, res=res), n)
    kb = bf16.Kernels.load()
    w = (torch.from_numpy(np.random.default_rng(7).normal(size=(n, k)).astype(np.float32)) / k ** 0.5).to(torch.bfloat16).cuda()
    out["bf16"] = (kb, lambda y: bf16.gemm(kb, y, n, x, k, w, m, res=res), n)
    out["bf16 swiglu"] = (kb, lambda y: bf16.gemm_swiglu(kb, y, x, k, w, m), n // 2)
    return out


@pytest.mark.parametrize("m,n,k", [(70, 384, 512), (129, 640, 1280), (300, 256, 1024)])
def test_small_tiles(m, n, k):
    import torch
    for name, (kern, run, cols) in forms(torch, k, n, m).items():
        def call(tile, pieces):
            kern.set_option("gemm_tile", tile)
            kern.set_option("gemm_pieces", pieces)
            y = torch.full((m + 1, cols), 1.5, dtype=torch.bfloat16, device="cuda")
            run(y)
            torch.cuda.synchronize()
            assert (y[m:] == 1.5).all(), name
            return y[:m].clone()

        try:
            kern.set_option("gemm_splits", 1)
            want = call(1, 0)
            for tile in (2, 3):
                assert torch.equal(call(tile, 1), want), (name, tile)
                for pieces in (2, 3):
                    got = call(tile, pieces).float()
                    rms = want.float().square().mean().sqrt()
                    # (a step of the sum before the residual or the SwiGLU product shows in a smaller result)
                    assert ((got - want.float()).abs() <= want.float().abs() / 64 + 2e-2 * rms).all(), (name, tile, pieces)
                    assert (got != want.float()).float().mean() < 0.05, (name, tile, pieces)
        finally:
            kern.set_option("gemm_splits", 8)
            kern.set_option("gemm_tile", 0)
            kern.set_option("gemm_pieces", 0)


@pytest.mark.parametrize("inter,k,m", [(128, 512, 70), (640, 1280, 300)])
def test_small_tiles_of_the_nvfp4_swiglu_front(inter, k, m):
    import torch
    from ferrite_amd import fp4, synth
    kern = fp4.Kernels.load()
    g, u = synth.fp4_linear(inter, k, 1, name="gate"), synth.fp4_linear(inter, k, 2, name="up")
    fused = fp4.HostLinear.fuse([("gate", g.codes, g.sf, 1.0, 1.0), ("up", u.codes, u.sf, 1.0, 1.0)])
    fused.alpha[:] = fused.alpha * np.float32(0.02)
    sw = fused.into_swiglu().upload()
    ws, act = fp4.Workspace(m, k), fp4.Workspace(m, inter)
    x = torch.from_numpy(synth.activations(m, k, 9).view(np.int16)).cuda()

    def call(tile, pieces):
        kern.set_option("gemm_tile", tile)
        kern.set_option("gemm_pieces", pieces)
        sw.forward_swiglu(kern, ws, act, x, k, m, 0.5)
        torch.cuda.synchronize()
        return [a.copy() for a in act.read(m, inter)]

    try:
        kern.set_option("gemm_splits", 1)
        codes, sf = call(1, 0)
        for tile in (2, 3):
            c, s = call(tile, 1)
            assert np.array_equal(c, codes) and np.array_equal(s, sf), tile
            c, s = call(tile, 2)
            assert (c != codes).mean() < 1e-2 and (s != sf).mean() < 5e-3, tile
    finally:
        kern.set_option("gemm_splits", 8)
        kern.set_option("gemm_tile", 0)
        kern.set_option("gemm_pieces", 0)
