"""Kernels at the edges of their launch shapes: sizes that leave remainders in a workgroup's share, the smallest and
the largest of a range, and every branch of a choice made by size."""
import numpy as np
import pytest

from conftest import to_dev
from ettk_amd.abi import default_params
from ettk_amd.synth import blob_reference, make_particles


@pytest.mark.gpu
@pytest.mark.parametrize("N", [16, 48, 96])
def test_particle_mean_blocks(torch_gpu, ctx, N):
    """The particle mean summed over workgroups: half a block at 16, 13.5 at 48, an exact number at 96.  The score takes
    the particle minus its mean, so a constant added to the volume leaves it as it was up to the rounding of the
    shifted voxels: 2^-24 of 128 per voxel is 8e-6 of a unit-variance volume, and the score moves by at most twice
    the relative change of its spectrum.  A block left out of the sum would move the mean by units."""
    from ettk_amd.lib import Plan

    ref = blob_reference(N, seed=3)
    ps = make_particles(ref, 2, seed=4, half_wedge=(50, 60), snr=(0.5, 0.5), max_shift=1.0)
    vols = ps.vols / ps.vols.std()
    plan = Plan(ctx, default_params(N, 8, mask_radius=N / 2 - 3, square_mask=2))
    try:
        plan.set_reference(to_dev(torch_gpu, ref))
        x = np.zeros((2, 6))
        s0, _ = plan.ccc_grad(to_dev(torch_gpu, vols), ps.descs, [0, 1], ps.truth, x)
        s1, _ = plan.ccc_grad(to_dev(torch_gpu, vols + np.float32(100.0)), ps.descs, [0, 1], ps.truth, x)
        print(f"[edges] N={N} score {s0} shifted {s1}", flush=True)
        assert np.abs(s0).min() > 0.1
        assert np.abs(s1 - s0).max() < 5e-5
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("N", [16, 48, 96])
def test_average_transposed_tiles(torch_gpu, ctx, N):
    """The average's output tiles: half a 32-wide tile at 16, one and a half at 48, three at 96.  One particle averaged at
    the identity against the FP64 oracle, whose interpolator moves a sample by the same 2^-17 voxel: the spectrum is
    divided by the amplitude it was multiplied by, in FP64, so FP32 transforms (2^-24 times their log2(N^3) <= 20
    levels, forward and back, 3e-6 at most) set the difference, and a factor of 8 is left."""
    from ettk_amd.abi import Particle, particle_array
    from ettk_amd.lib import Plan
    from oracle_lib import OraclePlan, oracle, vp

    g = np.random.default_rng(N)
    v = g.standard_normal((1, N, N, N)).astype(np.float32)
    p = default_params(N, 8, mask_radius=N / 2 - 3, square_mask=2)
    plan, orc = Plan(ctx, p), OraclePlan(p)
    try:
        out = torch_gpu.full((N, N, N), 7.0, dtype=torch_gpu.float32, device="cuda")
        torch_gpu.cuda.synchronize()
        plan.average(to_dev(torch_gpu, v), [Particle()], [1.0], [np.eye(4)], out)
        want, one, eye = np.zeros((N, N, N)), np.ones(1, np.float32), np.eye(4).reshape(1, 16)
        oracle().orc_average(orc.h, 1, vp(v), particle_array([Particle()]), vp(one), vp(eye), vp(want))
        err = np.abs(out.cpu().numpy() - want).max()
        print(f"[edges] average N={N} err {err:.2e}", flush=True)
        assert err < 2.4e-5
    finally:
        plan.close()
