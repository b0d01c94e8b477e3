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
    from ferrite_amd import fp4
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


def _exact(torch, form, n, k, m):
    """(kernels, x, y, ldy, res -> None) on operands whose sums are exact in f32 in any order: halves and whole numbers up to 6, K at most 2560."""
    from ferrite_amd import bf16, fp4
    rng = np.random.default_rng(13)
    values = np.array([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], np.float32)
    draw = lambda r, c: rng.choice(values, (r, c)) * rng.choice(np.array([-1.0, 1.0], np.float32), (r, c))
    x = draw(m, k)
    x[:, ::16] = 6.0  # (NVFP4: every block's scale is 1)
    x = torch.from_numpy(x).to(torch.bfloat16).cuda()
    if form == "bf16":
        kern, w = bf16.Kernels.load(), torch.from_numpy(draw(n, k)).to(torch.bfloat16).cuda()
        return kern, lambda y, ldy, res: bf16.gemm(kern, y, ldy, x, k, w, m, res=res)
    kern, ws = fp4.Kernels.load(), fp4.Workspace(m, k)
    if form == "nvfp4":
        host = fp4.HostLinear.fuse([("a", rng.integers(0, 256, (n, k // 2), dtype=np.uint8), np.full((n, k // 16), 0x38, np.uint8), 2.0 ** -7, 1.0)])
    else:
        host = fp4.HostLinear.fuse_fp8([("a", torch.from_numpy(draw(n, k)).to(torch.float8_e4m3fn).view(torch.uint8).numpy(), 2.0 ** -7, 1.0)])
    lin = host.upload()
    return kern, lambda y, ldy, res: lin.forward(kern, ws, y, ldy, x, k, m, res=res)


# two to nine pieces of K (up to eight are asked for at once, 128 x 128 the first, then four, two, one); rows and columns that end inside a workgroup's 16 (8) x 128
@pytest.mark.parametrize("form,m,n,gap", [("bf16", 143, 328, 4), ("bf16", 301, 264, 0), ("nvfp4", 143, 384, 8), ("nvfp4", 301, 256, 0), ("fp8", 143, 384, 8), ("fp8", 301, 256, 0)])
def test_cut_tiles_of_exact_sums(form, m, n, gap):
    """The reduce launches: the very bits of the launch without a cut, and with a residual bf16(bf16(sum) + res) of them, in place and from another buffer."""
    import torch
    k, ldy = 2560, n + gap
    kern, run = _exact(torch, form, n, k, m)
    old = torch.from_numpy(np.random.default_rng(17).normal(size=(m, n)) * 40).to(torch.bfloat16).cuda()

    def call(in_place, adds):
        y = torch.full((m + 1, ldy), 1.5, dtype=torch.bfloat16, device="cuda")
        res = y if in_place else torch.full((m + 1, ldy), 2.5, dtype=torch.bfloat16, device="cuda")
        if adds:
            res[:m, :n] = old
        run(y, ldy, res if adds else None)
        torch.cuda.synchronize()
        assert (y[m:] == 1.5).all() and (y[:, n:] == 1.5).all(), (form, in_place)
        return y[:m, :n].clone()

    def options(tile, pieces, splits):
        for name, value in (("gemm_tile", tile), ("gemm_pieces", pieces), ("gemm_splits", splits)):
            kern.set_option(name, value)

    try:
        options(1, 1, 1)
        want = call(False, False)
        added = (want.float() + old.float()).to(torch.bfloat16)
        assert want.unique().numel() > 500
        for s in [(t, p, 1) for t in (2, 3) for p in (2, 3, 5, 8, 9)] + [(t, 0, p) for t in (1, 4, 5, 6) for p in (2, 5, 8)]:
            options(*s)
            assert torch.equal(call(False, False), want), s
            for in_place in (False, True):
                assert torch.equal(call(in_place, True), added), (s, in_place)
    finally:
        options(0, 0, 8)


def test_nvfp4_swiglu_of_infinities():
    """Sums that leave f32 or meet an infinite or absent scale: the tiles' epilogue and the reduce launch of cut tiles leave the same codes and block scales."""
    import torch
    from ferrite_amd import fp4
    inter, k, m = 384, 512, 143
    kern, rng = fp4.Kernels.load(), np.random.default_rng(19)
    part = lambda name: (name, rng.integers(0, 256, (inter, k // 2), dtype=np.uint8), np.full((inter, k // 16), 0x38, np.uint8), 2.0 ** -7, 1.0)
    fused = fp4.HostLinear.fuse([part("gate"), part("up")])
    for i, odd in enumerate((3e38, np.inf, -np.inf, np.nan, 1e-40, 0.0)):  # in blocks of their own, and all in the last one
        fused.alpha[16 * i + i], fused.alpha[inter + 16 * i + 2 * i] = odd, odd
        fused.alpha[inter - 16 + i], fused.alpha[2 * inter - 2 - i] = odd, odd
    sw = fused.into_swiglu().upload()
    x = rng.choice([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], (m, k)) * rng.choice([-1.0, 1.0], (m, k))
    x[:, ::16] = 6.0
    x[5] = 0.0
    x = torch.from_numpy(x).to(torch.bfloat16).cuda()
    ws, act = fp4.Workspace(m, k), fp4.Workspace(m, inter)

    def call(tile, pieces):
        kern.set_option("gemm_tile", tile)
        kern.set_option("gemm_pieces", pieces)
        sw.forward_swiglu(kern, ws, act, x, k, m, 0.5)
        torch.cuda.synchronize()
        codes, sf = (a.copy() for a in act.read(m, inter))
        plain = lambda c: np.where(c & 7, c, 0)  # (a NaN that the product makes has no sign of its own: a code of magnitude 0 is one, whatever its sign)
        return plain(codes & 15), plain(codes >> 4), sf

    try:
        kern.set_option("gemm_splits", 1)
        want = call(2, 2)
        assert (want[2] == 0x7e).any() and np.unique(want[0]).size > 8
        for tile, pieces in [(1, 1), (2, 1), (3, 1), (3, 2), (4, 1), (5, 1), (6, 1)]:
            for a, b in zip(call(tile, pieces), want):
                assert np.array_equal(a, b), (tile, pieces)
    finally:
        kern.set_option("gemm_splits", 8)
        kern.set_option("gemm_tile", 0)
        kern.set_option("gemm_pieces", 0)


@pytest.mark.parametrize("inter,m", [(184, 143), (640, 301)])
def test_bf16_swiglu_of_exact_sums(inter, m):
    """The bf16 SwiGLU front: tiles finished in registers and the reduce launch of cut tiles leave the same values, infinities and NaN among them."""
    import torch
    from ferrite_amd import bf16
    k, kern, rng = 2560, bf16.Kernels.load(), np.random.default_rng(23)
    whole = lambda r, c: torch.from_numpy(rng.integers(-2, 3, (r, c)).astype(np.float32)).to(torch.bfloat16).cuda()
    x, w = whole(m, k), bf16.interleave_gu(kern, whole(inter, k), whole(inter, k))
    x[3, 7], x[17, 100], x[17, 2000], x[40, 2559], x[m - 1, 0] = np.inf, np.inf, -np.inf, np.nan, -np.inf

    def call(tile, pieces, splits):
        for name, value in (("gemm_tile", tile), ("gemm_pieces", pieces), ("gemm_splits", splits)):
            kern.set_option(name, value)
        act = torch.full((m + 1, inter), 1.5, dtype=torch.bfloat16, device="cuda")
        bf16.gemm_swiglu(kern, act, x, k, w, m)
        torch.cuda.synchronize()
        assert (act[m:] == 1.5).all()
        return act[:m].float().cpu().numpy()

    try:
        want = call(1, 1, 1)
        assert np.isnan(want).any() and np.isinf(want).any()
        for s in [(t, p, 1) for t in (2, 3) for p in (1, 2, 5, 9)] + [(t, 0, p) for t in (1, 4, 5, 6) for p in (1, 5)]:
            assert np.array_equal(call(*s), want, equal_nan=True), s
    finally:
        call(0, 0, 8)
