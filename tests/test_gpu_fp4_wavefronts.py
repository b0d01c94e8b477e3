"""The NVFP4 GEMV of up to 16 rows where it sums eighths of K, by eight wavefronts or by four: the same bits in every form, and the sums of the GEMV over weight tiles in
another order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# Eighths of one step, of unequal length, of nine steps; the last program partly past n; as many columns as there may be, and a block more (quarters); k below the
# rule's (quarters). Programs of 8 to 72 columns, rows of every form, the quantizer inside and with its own launch.
@pytest.mark.parametrize("n,k", [(128, 2048), (640, 2304), (1152, 4096), (256, 17408), (12288, 2048), (12416, 2048), (384, 1792)])
def test_every_form_of_the_eighths_gives_the_same_bits(n, k):
    import torch
    from ferrite_amd import fp4, synth
    kern = fp4.Kernels.load()
    lin = synth.fp4_linear(n, k, 7, input_scale=0.7).upload()
    rng = np.random.default_rng(n + k)
    x = torch.from_numpy((rng.normal(size=(16, k + 8)) * 30).astype(np.float32)).cuda().to(torch.bfloat16)
    ws = fp4.Workspace(16, k)

    def run(m, cols=0, quant=0, strips=1):
        for name, v in (("gemv_cols", cols), ("gemv_quant", quant), ("gemv_strips", strips)):
            kern.set_option(name, v)
        y = torch.full((m + 1, n), 5.0, dtype=torch.bfloat16, device="cuda")
        lin.forward(kern, ws, y, n, x, k + 8, m)
        torch.cuda.synchronize()
        assert (y[m] == 5.0).all()
        return y[:m]

    want = run(16)
    a, b = want.double(), run(16, strips=0).double()
    assert ((a - b).abs() <= b.abs() / 128.0 + 1e-30).all()  # exact products, f32 sums: a bf16 step where a sum lies between two
    for m in (1, 2, 3, 4, 5, 8, 9, 16):
        for cols in (0, 8, 16, 24, 32, 40, 48, 72):
            for quant in (0, 10240, 32768):
                assert torch.equal(run(m, cols, quant).view(torch.int16), want[:m].view(torch.int16)), (m, cols, quant)
