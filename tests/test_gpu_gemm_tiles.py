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


@pytest.mark.parametrize("strips", [True, False])
def test_trellis_of_4_gb_and_more(strips):
    """Byte offsets into a trellis of 2^32 bytes and a few column blocks: every tile of the prefill GEMM, both schedules, and the decode into
    tiles give the first, a middle and the last column blocks the bits of linears that hold these blocks alone. The decode GEMV, which
    addresses a trellis by 32 bits, refuses it, one linear, a group or an MLP block."""
    import torch
    from ferrite_amd import exl3
    from ferrite_amd._lib import FeError
    k, n, bits, m = 16384, 262144 + 384, 8, 70
    kt, nb, tile = k // 16, n // 128, 8 * 8 * bits  # words of the 8 tiles of a column block and k step
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    words = torch.empty(k * n // 32 * bits, dtype=torch.int32, device="cuda")
    for part in words.chunk(8):
        part.random_(-(1 << 31), 1 << 31, generator=gen)
    assert words.numel() * 4 > 1 << 32
    suh = torch.ones(k, dtype=torch.float16, device="cuda")
    svh = (torch.rand(n, generator=gen, device="cuda") + 0.5).to(torch.float16) / 128
    x = torch.randn(m, k, generator=gen, device="cuda").to(torch.bfloat16)
    kern = exl3.Kernels.load()

    def linear(w, cols, sv):
        view = exl3.Exl3View(k, cols, bits, w.data_ptr(), suh.data_ptr(), sv.data_ptr(), strips)
        lin = exl3.Linear.from_view(kern, "w", view, exl3.Linear.plan_for(k, cols, bits, exl3.default_blocks(exl3.cu_count())))
        lin.keep = (w, sv)
        return lin

    def forward(lin, out=exl3.Dtype.Bf16):
        y = torch.zeros((m, lin.n), dtype=torch.bfloat16, device="cuda")
        lin.forward(x, exl3.Dtype.Bf16, y, out, m, exl3.Workspace([lin], m))
        torch.cuda.synchronize()
        return y

    whole = linear(words, n, svh)
    try:
        for option, value in (("gemm_tile", 1), ("gemm_tile", 2), ("gemm_tile", 3), ("hat_rows", 65)):
            kern.set_option("gemm_splits", 1)
            kern.set_option("gemm_sk", 0)
            kern.set_option(option, value)
            y = forward(whole)
            for b0, b1 in ((0, 2), (1024, 1026), (nb - 3, nb)):
                w = words.view(nb, kt * tile)[b0:b1] if strips else words.view(kt, nb, tile)[:, b0:b1]
                want = forward(linear(w.contiguous(), 128 * (b1 - b0), svh[128 * b0:128 * b1].contiguous()))
                assert want.float().abs().amax(dim=0).min() > 0  # (no column of zeros: what reads past a wrapped size give)
                assert torch.equal(y[:, 128 * b0:128 * b1], want), (option, value, b0)
    finally:
        for option, value in (("gemm_tile", 0), ("hat_rows", 2304), ("gemm_splits", 8), ("gemm_sk", 1)):
            kern.set_option(option, value)
    down = linear(words, n, svh)
    ws = exl3.Workspace([whole, down], m)
    y = torch.full((m, n), 2.0, dtype=torch.bfloat16, device="cuda")
    for rows in (1, 8, 17, 64):
        with pytest.raises(FeError, match="4 GB"):
            whole.forward(x, exl3.Dtype.Bf16, y, exl3.Dtype.Bf16, rows, ws)
        with pytest.raises(FeError, match="4 GB"):
            exl3.forward_group([whole, down], x, exl3.Dtype.Bf16, [y, y], exl3.Dtype.Bf16, rows, ws)
    torch.cuda.synchronize()
    assert (y == 2.0).all()
