"""Extraction far along a long axis, where an FP32 coordinate has few bits left for the fraction."""
import numpy as np
import pytest

from conftest import to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("nx,N", [(3000, 24), (9990, 40), (20000, 24)])
def test_extract_far_along_an_axis(torch_gpu, ctx, nx, N):
    """Boxes near the far end of an axis against the FP64 oracle.  Along x the offset, the sum and the floor tolerance are
    rounded, half a unit in the last place of nx each (the other axes are short: 1e-5 voxels); the gradient of a
    volume smoothed by 1.5 voxels is at most 1 / 1.5 of its maximum per voxel, and the subtracted mean moves by as much
    again: 2 units of the maximum, and 4e-5."""
    from scipy import ndimage

    from ettk_amd.abi import Particle
    from ettk_amd.synth import random_rotation
    from oracle_lib import extract

    g = np.random.default_rng(nx)
    tomo = ndimage.gaussian_filter(g.standard_normal((36, 40, nx)), 1.5).astype(np.float32)
    n = 8
    pos = np.stack([g.uniform(nx - 700, nx - 100, n), g.uniform(10, 30, n), g.uniform(10, 26, n)], 1)
    descs = []
    for _ in range(n):
        t = np.eye(4)
        t[:3, :3] = random_rotation(g)
        descs.append(Particle(matrix=t, normal=tuple(g.uniform(-40, 40, 3))))
    out = torch_gpu.full((n, N, N, N), 9.0, dtype=torch_gpu.float32, device="cuda")
    torch_gpu.cuda.synchronize()
    ctx.extract(to_dev(torch_gpu, tomo), pos, descs, N, out)
    got, want = out.cpu().numpy(), extract(tomo, pos, descs, N)
    both = (got != 0) & (want != 0)
    err = np.abs(got - want)[both].max() / np.abs(tomo).max()
    print(f"[far] extract nx={nx} N={N}: {both.sum()} valid voxels, {err:.2e} of the maximum", flush=True)
    assert both.sum() > 0.3 * n * N ** 3
    assert np.count_nonzero((got != 0) != (want != 0)) <= 0.0005 * n * N ** 3
    assert err <= 2 * np.spacing(np.float32(nx)) + 4e-5
