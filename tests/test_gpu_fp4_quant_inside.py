"""The NVFP4 GEMV that quantizes its own activations against the quantizer's launch followed by the GEMV: the same bits in the output and in
what the call leaves in the workspace (codes, block scales, fp16 operand)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from ferrite_amd import fp4
    assert torch.cuda.is_available()
    return torch, fp4, fp4.Kernels.load()


def operand(fp4, ws, m, k):
    import ctypes as C
    from ferrite_amd import _lib
    ptr = C.c_uint64()
    _lib.check(_lib.lib().fe_fp4_workspace_operand(ws.h, C.byref(ptr)))
    out = np.empty((m, k), np.uint16)
    _lib.check(_lib.lib().fe_hip_memcpy_dtoh(out.ctypes.data_as(C.c_void_p), ptr.value, out.nbytes))
    return out


def both(env, lin, kern, x, lda, m, res=None, in_place=False):
    """(output, codes, scales, operand) with the quantizer inside and with its own launch."""
    torch, fp4, _ = env
    got = []
    for limit in (32768, 0):
        kern.set_option("gemv_quant", limit)
        try:
            ws = fp4.Workspace(m, lin.k)
            xi = x.clone()
            y = xi if in_place else torch.full((m, lin.n + 8), 7.0, dtype=torch.bfloat16, device="cuda")
            lin.forward(kern, ws, y, lda if in_place else lin.n + 8, xi, lda, m, res=res)
            torch.cuda.synchronize()
            got.append((y.view(torch.int16).cpu().numpy(), *ws.read(m, lin.k), operand(fp4, ws, m, lin.k)))
        finally:
            kern.set_option("gemv_quant", 10240)
    return got


# One step of K for one wavefront alone, quarters of unequal length, an odd count of (step, row) units, a quarter of the largest length; columns
# that fill their programs and not
@pytest.mark.parametrize("n,k,m", [(n, k, m) for n, k in [(128, 256), (384, 1280), (640, 2304), (1152, 4096), (256, 17408)]
                                   for m in (1, 2, 3, 4, 5, 8) if m * k <= 32768])
def test_same_bits_as_the_quantizers_launch(env, n, k, m):
    torch, fp4, kern = env
    from ferrite_amd import synth
    lin = synth.fp4_linear(n, k, 5, input_scale=0.7).upload()
    rng = np.random.default_rng(n + k + m)
    lda = k + 24
    x = torch.from_numpy((rng.normal(size=(m, lda)) * 50).astype(np.float32)).cuda().to(torch.bfloat16)
    x[0, :16] = 0.0  # an all-zero block
    x[m - 1, k - 1], x[m - 1, 33], x[0, 70] = float("nan"), float("inf"), -3e38
    res = torch.from_numpy(rng.normal(size=(m, n + 8)).astype(np.float32)).cuda().to(torch.bfloat16)
    inside, launch = both(env, lin, kern, x, lda, m, res)
    for a, b in zip(inside, launch):
        assert np.array_equal(a, b)


def test_output_over_the_activations(env):
    torch, fp4, kern = env
    from ferrite_amd import synth
    k = 1024
    lin = synth.fp4_linear(k, k, 9).upload()
    x = torch.from_numpy(np.random.default_rng(1).normal(size=(2, k)).astype(np.float32)).cuda().to(torch.bfloat16)
    inside, launch = both(env, lin, kern, x, k, 2, in_place=True)
    for a, b in zip(inside, launch):
        assert np.array_equal(a, b)
