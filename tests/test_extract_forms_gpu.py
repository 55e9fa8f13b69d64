"""The two forms of the extraction: tiles, and runs of voxels for maps that magnify 2.25 times and more."""
import numpy as np
import pytest

from conftest import to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("N", [1, 7, 17, 32])
def test_forms_mixed_in_one_call(torch_gpu, ctx, N):
    """Boxes of both forms in one call, whose workgroups per box differ (1 tile and 2 runs at 7, 27 and 20 at 17, 64 and 128
    at 32), equal those cut alone, bit for bit, and the FP64 oracle's.  Offsets below 256 are rounded by 7.6e-6 voxels,
    four times on each of three axes, at a gradient of at most 1 / 1.5 of the maximum per voxel: 6e-5 of the maximum,
    and the subtracted mean moves by as much at most."""
    from scipy import ndimage

    from ettk_amd.abi import Particle
    from ettk_amd.synth import random_rotation
    from oracle_lib import extract

    g = np.random.default_rng(40 + N)
    tomo = ndimage.gaussian_filter(g.standard_normal((64, 80, 96)), 1.5).astype(np.float32)
    scales = [1.0, 2.2, 3.0, 2.3, 1.0, 6.0]
    pos = np.stack([g.uniform(20, 76, 6), g.uniform(20, 60, 6), g.uniform(15, 49, 6)], 1)
    descs = []
    for s in scales:
        t = np.eye(4)
        t[:3, :3] = random_rotation(g) * s
        descs.append(Particle(matrix=t, normal=tuple(g.uniform(-40, 40, 3))))
    d_tomo = to_dev(torch_gpu, tomo)

    def cut(which):
        out = torch_gpu.full((len(which), N, N, N), 9.0, dtype=torch_gpu.float32, device="cuda")
        torch_gpu.cuda.synchronize()
        ctx.extract(d_tomo, pos[which], [descs[i] for i in which], N, out)
        return out.cpu().numpy()

    got = cut(list(range(6)))
    for i in range(6):
        assert np.array_equal(got[i], cut([i])[0]), scales[i]
    want = extract(tomo, pos, descs, N)
    both = (got != 0) & (want != 0)
    print(f"[forms] N={N}: {both.sum()} valid voxels", flush=True)
    assert np.count_nonzero((got != 0) != (want != 0)) <= 0.0005 * 6 * N ** 3
    if both.any():
        assert np.abs(got - want)[both].max() <= 1.2e-4 * np.abs(tomo).max()
