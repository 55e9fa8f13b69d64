"""Particle means (launch_vol_mean, refine.hip): one workgroup per particle at 16 and 32, partial sums above.  Called by its C++
name.  FP64 sums of FP32 voxels, rounded to FP32 once: equal to numpy's rounded mean up to one unit in the last place."""
import ctypes as C

import numpy as np
import pytest

from conftest import to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("N,count", [(16, 1), (16, 300), (32, 1), (32, 65), (48, 3), (64, 2)])
def test_means_match_numpy(torch_gpu, ctx, N, count):
    fn = getattr(ctx.lib, "_ZN4ettk15launch_vol_meanEPKfiiPdPfP12ihipStream_t")
    fn.argtypes, fn.restype = [C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p], None
    g = np.random.default_rng(N + count)
    vols = (g.standard_normal((count, N, N, N)) * g.uniform(1, 100, (count, 1, 1, 1)) + 7).astype(np.float32)
    d = to_dev(torch_gpu, vols)
    part = torch_gpu.zeros((count, (N ** 3 + 8191) // 8192), dtype=torch_gpu.float64, device="cuda")
    mean = torch_gpu.full((count + 1,), -5.0, dtype=torch_gpu.float32, device="cuda")
    torch_gpu.cuda.synchronize()
    fn(d.data_ptr(), count, N, part.data_ptr(), mean.data_ptr(), None)
    torch_gpu.cuda.synchronize()
    got = mean.cpu().numpy()
    want = vols.reshape(count, -1).astype(np.float64).mean(1).astype(np.float32)
    assert np.abs(got[:count] - want).max() <= np.spacing(np.abs(want)).max()
    assert got[count] == -5.0
