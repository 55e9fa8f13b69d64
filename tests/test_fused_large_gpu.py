"""The fused c2r -> operation -> r2c planes at 96 and 128, which the CCC runs and ettk_fft3 does not offer: called by the
C++ name of what stands behind ettk_fft3, against the FP64 composition, with the bars of test_fft_gpu.py (5e-6 over the
whole half spectrum and over its k = 0 and k = n/2 planes)."""
import ctypes as C

import numpy as np
import pytest

from test_fft_gpu import _check_half, _checker

MASK, SQUARE = 2, 3


def run(ctx, n, batch, kind, d_in, d_out, d_aux=None):
    fn = getattr(ctx.lib, "_ZN4ettk8fft3_runEP8ettk_ctxiiiPKvPvPKf")
    fn.argtypes, fn.restype = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p], None
    fn(ctx.h, n, batch, kind, d_in.data_ptr(), d_out.data_ptr(), d_aux.data_ptr() if d_aux is not None else None)


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch,hermitian", [(96, 2, True), (96, 1, False), (128, 1, True), (128, 1, False)])
def test_fused_planes_match_numpy(torch_gpu, ctx, n, batch, hermitian):
    """A spectrum that is not Hermitian on the k = 0 and k = n/2 planes keeps only its real part there, as FFTW's c2r."""
    torch = torch_gpu
    g = np.random.default_rng(n + hermitian)
    shape = (batch, n, n, n // 2 + 1)
    if hermitian:
        X = np.fft.rfftn(g.standard_normal((batch, n, n, n)), axes=(1, 2, 3)).astype(np.complex64)
    else:
        X = (g.standard_normal(shape) + 1j * g.standard_normal(shape)).astype(np.complex64)
    m = g.uniform(0.0, 1.0, (n, n, n)).astype(np.float32)
    r = np.fft.irfftn(X.astype(np.complex128), s=(n, n, n), axes=(1, 2, 3)) * float(n) ** 3
    dX, dm = torch.from_numpy(X).cuda(), torch.from_numpy(m).cuda()
    out = torch.empty_like(dX)
    torch.cuda.synchronize()
    run(ctx, n, batch, MASK, dX, out, dm)
    _check_half(out.cpu().numpy(), np.fft.rfftn(r * m.astype(np.float64), axes=(1, 2, 3)))
    run(ctx, n, batch, SQUARE, dX, out)
    _check_half(out.cpu().numpy(), np.fft.rfftn(r * r * _checker(n), axes=(1, 2, 3)))
    assert np.array_equal(dX.cpu().numpy(), X)
