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
