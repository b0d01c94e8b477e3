"""The prompt GEMM that decodes the trellis into registers (exl3_rgemm_b*): every width, one and two column blocks a program (option
rgemm_form), tiles whole, cut and dealt as runs that cross from one tile to the next (rgemm_pieces), against the oracle's product over the
GPU's own rotated inputs, and against the GEMM that passes the decoded weights through LDS (rgemm = 0)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def setup(k, n, bits, m, strips=True):
    import torch
    from ferrite_amd import exl3, synth
    kern = exl3.Kernels.load()
    t = synth.exl3_tensor(k, n, bits, 40 + bits)
    lin = exl3.Linear.new(kern, exl3.DeviceExl3(t, strips), 64)
    x = torch.from_numpy(synth.activations(m, k, 3, outliers=True).view(np.int16)).cuda()
    return torch, exl3, kern, t, lin, x


def options(kern, **o):
    for name, default in (("rgemm", 1), ("rgemm_form", 0), ("rgemm_pieces", 0)):
        kern.set_option(name, o.get(name, default))


# rows at the edges of the row groups (32 rows a step of the kernels' sizes), of one tile and of two; an odd count of column blocks; the
# shortest K, K of an odd count of steps; trellis layouts
@pytest.mark.parametrize("bits,k,n,m,strips", [(2, 256, 128, 65, True), (3, 384, 384, 96, False), (4, 1024, 384, 97, True), (5, 640, 640, 160, True),
                                               (6, 512, 256, 255, False), (8, 1152, 384, 256, True), (4, 512, 640, 257, False),
                                               (3, 1024, 256, 449, True), (8, 384, 384, 513, True), (4, 256, 384, 1100, True), (3, 256, 256, 2303, True)])
def test_against_the_oracle(oracle, bits, k, n, m, strips):
    torch, exl3, kern, t, lin, x = setup(k, n, bits, m, strips)
    ws = exl3.Workspace([lin], m)

    def run(dt, fill, **o):
        options(kern, **o)
        f32 = dt in (exl3.Dtype.F32, exl3.Dtype.F32Add)
        y = torch.full((m + 2, n), fill, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
        lin.forward(x, exl3.Dtype.Bf16, y, dt, m, ws)
        torch.cuda.synchronize()
        assert (y[m:] == fill).all()
        return y[:m].float().cpu().numpy().astype(np.float64)

    try:
        lds = run(exl3.Dtype.F32, 3.0, rgemm=0)
        rows = sorted({0, 15, 16, 31, 32, 63, 64, m // 2, m - 17, m - 2, m - 1})
        o = oracle.Exl3(t.k, t.n, t.bits, t.trellis, t.suh, t.svh)
        ref = oracle.gemv_ref(o, oracle.w_hat_f16(o), ws.xh(m, k)[rows])
        rms = np.sqrt((lds ** 2).mean())
        for form in (0, 1, 2):
            for pieces in ((0,) if not form else (1, 2, 3, 5)):
                how = dict(rgemm_form=form, rgemm_pieces=pieces)
                got = run(exl3.Dtype.F32, 3.0, **how)
                # f32 sums of up to 1152 products in another order: a few times sqrt(K) 2^-24 of the rms (4e-6 at most here)
                assert np.abs(got - lds).max() < 1e-5 * rms, how
                assert np.abs(got[rows] - ref).max() < 1e-4 * rms, how
                assert np.array_equal(got, run(exl3.Dtype.F32, 3.0, **how)), how  # whatever program comes first
                plus = got + 0.25
                assert (np.abs(run(exl3.Dtype.F32Add, 0.25, **how) - plus) <= (np.abs(plus) + np.abs(got)) * 2.0 ** -23).all(), how
                assert (np.abs(run(exl3.Dtype.Bf16, 7.0, **how) - got) <= np.abs(got) / 256 + 1e-6 * rms).all(), how
                added = got + 1.5
                assert (np.abs(run(exl3.Dtype.Bf16Add, 1.5, **how) - added) <= np.abs(added) / 256 + 1e-6 * rms).all(), how
    finally:
        options(kern)


@pytest.mark.parametrize("bits,k,n,m,form,pieces", [(4, 2560, 256, 70, 1, 9), (3, 2560, 128, 130, 1, 10), (5, 2560, 384, 200, 2, 17), (4, 2560, 256, 66, 1, 20), (8, 2432, 128, 129, 2, 38)])
def test_many_pieces_of_a_tile(oracle, bits, k, n, m, form, pieces):
    """Tiles cut into more pieces than the reduce launch loads at once, a step each at most."""
    torch, exl3, kern, t, lin, x = setup(k, n, bits, m)
    ws = exl3.Workspace([lin], m)
    got = []
    try:
        for _ in range(2):
            options(kern, rgemm_form=form, rgemm_pieces=pieces)
            y = torch.full((m + 1, n), 3.0, dtype=torch.float32, device="cuda")
            lin.forward(x, exl3.Dtype.Bf16, y, exl3.Dtype.F32, m, ws)
            torch.cuda.synchronize()
            assert (y[m] == 3.0).all()
            got.append(y[:m].cpu().numpy().astype(np.float64))
    finally:
        options(kern)
    o = oracle.Exl3(t.k, t.n, t.bits, t.trellis, t.suh, t.svh)
    rows = sorted({0, 1, 15, 16, 63, m // 2, m - 2, m - 1})
    ref = oracle.gemv_ref(o, oracle.w_hat_f16(o), ws.xh(m, k)[rows])
    assert np.abs(got[0][rows] - ref).max() < 1e-4 * np.sqrt((ref ** 2).mean())
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("m,form", [(70, 1), (203, 1), (203, 2), (203, -1), (40, 0)])
def test_infinities_and_nans_stay_in_their_rows(m, form):
    """Rows that hold infinities and NaN among ordinary rows of one tile: the others keep their bits (through both GEMMs, form -1 the one
    that decodes into LDS, and the decode GEMV)."""
    torch, exl3, kern, t, lin, x = setup(640, 384, 4, m)
    ws = exl3.Workspace([lin], m)
    bad = [0, 5, 17, 31, m // 2, m - 1]
    x2 = x.clone().view(torch.bfloat16)
    for i, r in enumerate(bad):
        x2[r, 7 * i + 3] = (float("inf"), float("-inf"), float("nan"))[i % 3]
    got = []
    try:
        options(kern, rgemm=0 if form < 0 else 1, rgemm_form=max(form, 0), rgemm_pieces=3 if form > 0 else 0)
        for inp in (x, x2):
            y = torch.zeros((m, 384), dtype=torch.float32, device="cuda")
            lin.forward(inp, exl3.Dtype.Bf16, y, exl3.Dtype.F32, m, ws)
            torch.cuda.synchronize()
            got.append(y)
    finally:
        options(kern)
    fine = [r for r in range(m) if r not in bad]
    assert torch.equal(got[0][fine], got[1][fine]) and torch.isfinite(got[0]).all()
    assert not torch.isfinite(got[1][bad]).all(dim=1).any()


@pytest.mark.parametrize("m", [70, 300])
def test_gate_and_up_in_one_launch(m):
    """The routing layer's prompt over two trellis linears of one input: one launch, the members' own results up to the order of the sums,
    with a workspace too small for both rotated inputs as well (member by member), captured and replayed."""
    import torch
    from ferrite_amd import exl3, route, synth
    kern = exl3.Kernels.load()
    k, n = 1024, 640
    x3 = [exl3.Linear.new(kern, exl3.DeviceExl3(synth.exl3_tensor(k, n, 4, s), True), 64) for s in (1, 2)]
    down = exl3.Linear.new(kern, exl3.DeviceExl3(synth.exl3_tensor(n, k, 4, 3), True), 64)
    deep = exl3.Linear.new(kern, exl3.DeviceExl3(synth.exl3_tensor(2 * k, n, 4, 4), True), 64)
    x = torch.from_numpy(synth.activations(m, k, 5).view(np.int16)).cuda().view(torch.bfloat16)
    proj = route.Proj([(route.Linear("gate", n, k, q=x3[0]), [n]), (route.Linear("up", n, k, q=x3[1]), [n])])
    for ws in (exl3.Workspace(x3 + [deep], m), exl3.Workspace(x3 + [down], m)):
        ctx = route.LinCtx(x3=(kern, ws))
        out = torch.zeros((2, m, n), dtype=torch.bfloat16, device="cuda")
        proj.forward(ctx, out, x, k, m)
        torch.cuda.synchronize()
        for lin, got in zip(x3, out):
            y = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
            lin.forward(x, exl3.Dtype.Bf16, y, exl3.Dtype.Bf16, m, ws)
            torch.cuda.synchronize()
            d = (got.float() - y.float()).abs()
            assert (d <= y.float().abs() / 128 + 1e-5 * y.float().square().mean().sqrt()).all() and (d > 0).float().mean() < 0.02
    want = out.clone()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        captured = route.LinCtx(x3=(kern, ws))
        proj.forward(captured, out, x, k, m)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
