"""9..64 rows: the launch that finishes gate and up also forms down's rotated input. The MLP block against its parts, bit for bit: the
grouped launch of gate and up, fe_silu_mul, down's own forward; programs singly and in pairs (option gemv_pairs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,hidden,inter,strips", [(2, 256, 128, True), (4, 1024, 640, True), (5, 384, 2816, False), (8, 640, 384, True)])
def test_mlp_block_has_the_bits_of_its_parts(bits, hidden, inter, strips):
    import torch
    from ferrite_amd import exl3, route, synth
    kern = exl3.Kernels.load()
    shapes = ((hidden, inter), (hidden, inter), (inter, hidden))
    g, u, d = (exl3.Linear.new(kern, exl3.DeviceExl3(synth.exl3_tensor(k, n, bits, 60 + i), strips), 256) for i, (k, n) in enumerate(shapes))
    ws = exl3.Workspace([g, u, d], 64)
    x = torch.from_numpy(synth.activations(64, hidden, 7).view(np.int16)).cuda()
    bf = lambda *shape: torch.full(shape, 1.5, dtype=torch.bfloat16, device="cuda")
    B = exl3.Dtype.Bf16
    try:
        for rows in (9, 15, 16, 17, 32, 33, 47, 48, 64):
            yg, yu, act, want = bf(rows, inter), bf(rows, inter), bf(rows, inter), bf(rows, hidden)
            kern.set_option("gemv_pairs", 0)
            exl3.forward_group([g, u], x, B, [yg, yu], B, rows, ws)
            route.silu_mul(act, yg.data_ptr(), yu.data_ptr(), inter, inter, rows)
            d.forward(act, B, want, exl3.Dtype.Bf16Add, rows, ws)
            for pairs in (0, 2):
                kern.set_option("gemv_pairs", pairs)
                og, ou, y = bf(rows + 1, inter), bf(rows + 1, inter), bf(rows + 1, hidden)
                for _ in range(2):  # (a second call on the same workspace)
                    y.fill_(1.5)
                    exl3.mlp_forward(g, u, d, x, B, og, ou, y, exl3.Dtype.Bf16Add, rows, ws)
                torch.cuda.synchronize()
                for got, ref in ((og, yg), (ou, yu), (y, want)):
                    assert torch.equal(got[:rows].view(torch.int16), ref.view(torch.int16)), (rows, pairs)
                    assert (got[rows:] == 1.5).all(), (rows, pairs)
    finally:
        kern.set_option("gemv_pairs", 1)


# runs that are whole column blocks (one, several; in pairs of programs), runs that cut some of the blocks, a run over all of them; runs of two
# blocks and more over a full chip, where the programs finish the blocks that lie in one run and the launch behind the others
@pytest.mark.parametrize("bits,k,n,plan", [(4, 128, 384, None), (3, 256, 2048, None), (2, 512, 1024, (8, 4, 4, 0)), (8, 384, 1536, (9, 1, 4, 0)), (5, 256, 1280, (10, 1, 4, 0)),
                                           (6, 1024, 512, (8, 1, 4, 0)), (4, 640, 640, (7, 1, 4, 0)), (4, 384, 384, (1, 1, 4, 0)), (2, 256, 140800, (1024, 1, 4, 0))])
def test_blocks_finished_by_their_program(bits, k, n, plan):
    """17..64 rows: a column block that lies in one run is finished by its program, the others by the launch behind. Every row has the bits
    of the single-row call, in every output mode, alone and grouped with a linear whose blocks are cut."""
    import torch
    from ferrite_amd import exl3, synth
    kern = exl3.Kernels.load()
    dev = exl3.DeviceExl3.upload_strips(synth.exl3_tensor(k, n, bits, 9))
    lin = exl3.Linear.with_plan(kern, dev, exl3.Plan(*plan)) if plan else exl3.Linear.new(kern, dev, 256)
    cut = exl3.Linear.with_plan(kern, exl3.DeviceExl3.upload_strips(synth.exl3_tensor(k, 256, bits, 10)), exl3.Plan(2 * (k // 128), 1, 4, 0))
    ws = exl3.Workspace([lin, cut], 64)
    x = torch.from_numpy(synth.activations(64, k, 7, outliers=True).view(np.int16)).cuda()
    D = exl3.Dtype
    one = [torch.zeros((64, l.n), dtype=torch.float32, device="cuda") for l in (lin, cut)]
    for l, y in zip((lin, cut), one):
        for r in range(64):
            l.forward(x[r:r + 1], D.Bf16, y[r:r + 1], D.F32, 1, ws)
    try:
        for rows in (17, 32, 33, 50, 64):
            for pairs in (0, 2):
                kern.set_option("gemv_pairs", pairs)
                for dt, fill, want in ((D.F32, 3.0, one[0]), (D.F32Add, 0.25, one[0] + 0.25), (D.Bf16, 3.0, one[0].bfloat16()),
                                       (D.Bf16Add, 1.5, (one[0] + 1.5).bfloat16())):
                    y = torch.full((65, n), fill, dtype=want.dtype, device="cuda")
                    for _ in range(2):
                        y[:rows] = fill
                        lin.forward(x, D.Bf16, y, dt, rows, ws)
                    torch.cuda.synchronize()
                    assert torch.equal(y[:rows], want[:rows]) and (y[rows:] == fill).all(), (rows, pairs, dt)
                ys = [torch.full((65, l.n), 3.0, device="cuda") for l in (lin, cut)]
                exl3.forward_group([lin, cut], x, D.Bf16, ys, D.F32, rows, ws)
                torch.cuda.synchronize()
                for y, want in zip(ys, one):
                    assert torch.equal(y[:rows], want[:rows]) and (y[rows:] == 3.0).all(), (rows, pairs)
    finally:
        kern.set_option("gemv_pairs", 1)
