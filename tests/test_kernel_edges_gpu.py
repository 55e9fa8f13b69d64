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


@pytest.mark.gpu
@pytest.mark.parametrize("N,scale", [(1, 1.0), (7, 1.0), (8, 1.0), (17, 1.0), (33, 1.0), (20, 1.7)])
def test_extract_tiles(torch_gpu, ctx, N, scale):
    """Extraction by 8^3 tiles: boxes smaller than a tile, exactly one, one voxel more than two or four, and a map that
    magnifies 1.7 times, whose input box exceeds the staged one.  Positions in FP32 (coordinates below 128: 7.6e-6 per
    operation) move a sample by about 1e-5 voxels, times a gradient of at most 1 / 1.5 of the maximum per voxel of a
    volume smoothed by 1.5 voxels, along three axes: 2e-5 of the maximum."""
    from scipy import ndimage

    from ettk_amd.abi import Particle
    from ettk_amd.synth import random_rotation
    from oracle_lib import extract

    g = np.random.default_rng(N)
    tomo = ndimage.gaussian_filter(g.standard_normal((64, 80, 96)), 1.5).astype(np.float32)
    n = 9
    pos = np.stack([g.uniform(0, 95, n), g.uniform(0, 79, n), g.uniform(0, 63, n)], 1)
    descs = []
    for _ in range(n):
        t = np.eye(4)
        t[:3, :3] = random_rotation(g) * scale
        descs.append(Particle(matrix=t, normal=tuple(g.uniform(-40, 40, 3)), cut_offset=float(g.uniform(-1, 1))))
    out = torch_gpu.full((n, N, N, N), 9.0, dtype=torch_gpu.float32, device="cuda")
    torch_gpu.cuda.synchronize()
    ctx.extract(to_dev(torch_gpu, tomo), pos, descs, N, out)
    got, want = out.cpu().numpy(), extract(tomo, pos, descs, N)
    both = (got != 0) & (want != 0)
    print(f"[edges] extract N={N} x{scale}: {both.sum()} valid voxels", flush=True)
    assert np.count_nonzero((got != 0) != (want != 0)) <= 0.0005 * n * N ** 3
    if both.any():
        assert np.abs(got - want)[both].max() <= 2e-5 * np.abs(tomo).max()


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(96, 1), (96, 3), (128, 1), (192, 1), (256, 1)])
def test_register_pencils(torch_gpu, ctx, n, batch):
    """Transforms whose strided passes hold their pencils in registers: at 96 (64 pencils a workgroup) a pass ends in half a
    workgroup of pencils for an odd batch, the other lengths have their own factorisation.  Forward and back against
    numpy in FP64; 3 log2(n) <= 24 levels of 2^-24 each way leave 1.5e-6, 5e-6 are allowed as for the other sizes."""
    g = np.random.default_rng(n + batch)
    v = g.standard_normal((batch, n, n, n)).astype(np.float32)
    F = torch_gpu.empty((batch, n, n, n // 2 + 1), dtype=torch_gpu.complex64, device="cuda")
    b = torch_gpu.empty((batch, n, n, n), dtype=torch_gpu.float32, device="cuda")
    d = to_dev(torch_gpu, v)
    ctx.fft3(ctx.FFT_R2C, n, batch, d, F)
    want = np.fft.rfftn(v.astype(np.float64), axes=(1, 2, 3))
    rel = np.linalg.norm(F.cpu().numpy() - want) / np.linalg.norm(want)
    ctx.fft3(ctx.FFT_C2R, n, batch, F, b)
    back = np.linalg.norm(b.cpu().numpy() / n ** 3 - v) / np.linalg.norm(v)
    print(f"[edges] fft {n} x{batch}: {rel:.2e} {back:.2e}", flush=True)
    assert rel < 5e-6 and back < 5e-6


@pytest.mark.gpu
@pytest.mark.parametrize("N,window", [(16, 3.0), (32, -1.0), (48, 1.0), (64, 0.0), (64, -1.0), (96, 19.5), (128, 11.0)])
def test_ccc_windows(torch_gpu, ctx, N, window):
    """The search window of the upsampled correlation at its ends: a single point (0), 3 x 3 x 3 half voxels (1), the
    whole doubled box (-1, at 32 and 64), the widest windows that 96 and 128 accept, and the smallest box.  Against the
    FP64 oracle with the bounds of the other comparisons of this chain: FP32 transforms and sums leave 1e-6 of the two
    norms whose difference the distance is, and the distance is above 1e-3 of them; the shift is an index, equal unless
    two half-voxel points tie within that."""
    from ettk_amd.lib import Plan
    from oracle_lib import OraclePlan
    from parity import DIST_RTOL, peak_tie

    p = default_params(N, 8, mask_radius=N / 2 - 3, square_mask=2, trans_restrict=window)
    ref = blob_reference(N, seed=5)
    n = 3 if N <= 64 else 1
    ps = make_particles(ref, n, seed=6, half_wedge=(50, 60), snr=(0.3, 0.3), max_shift=2.0)
    plan, orc = Plan(ctx, p), OraclePlan(p)
    try:
        plan.set_reference(to_dev(torch_gpu, ref))
        orc.set_reference(ref)
        t = ps.truth.copy()
        t[:, :3, 3] = 0.0
        dist, out = plan.ccc(to_dev(torch_gpu, ps.vols), ps.descs, list(range(n)), t)
        for i in range(n):
            want, m = orc.ccc(ps.vols[i], ps.descs[i], t[i])
            print(f"[edges] ccc N={N} window {window}: {dist[i]:.6e} {want:.6e}", flush=True)
            assert abs(dist[i] - want) <= DIST_RTOL * abs(want) + 1e-7
            assert np.abs(out[i] - m).max() < 1e-9 or peak_tie(orc, ps.vols[i], ps.descs[i], t[i], out[i])[0]
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("N,band,mask", [(16, (0.0, 0.5), True), (48, (0.0, 0.5), False), (96, (0.1, 0.3), True),
                                         (128, (0.0, 0.5), True)])
def test_projection_box_sizes(torch_gpu, ctx, N, band, mask):
    """The padded spectrum at every pencil shape (the smallest box, 4 threads and 24 elements per pencil, the
    largest with the narrower column steps), with a band that leaves most of it out and without the mask.  FP32
    transforms of (2N)^3 elements: 2^-24 per level, at most 24 levels, is 1.5e-6 of the rms magnitude per
    element; the 4..128 shells of one ray add to at least their mean, so 1e-5 of the largest value leaves a factor of 6."""
    from ettk_amd.lib import Plan
    from oracle_lib import OraclePlan

    p = default_params(N, 8, mask_radius=(N / 2 - 3) if mask else 0.0, square_mask=2, bp_lo=band[0], bp_hi=band[1])
    g = np.random.default_rng(N)
    ps = make_particles(blob_reference(N, seed=3), 2, seed=4, half_wedge=(50, 60), snr=(0.5, 0.5), max_shift=1.0)
    vols = (ps.vols / ps.vols.std() + g.standard_normal(ps.vols.shape) + 1.0).astype(np.float32)
    plan, orc = Plan(ctx, p), OraclePlan(p)
    try:
        pp = plan.project(to_dev(torch_gpu, vols), ps.descs)
        err = 0.0
        for i in range(2):
            want = orc.project(vols[i], ps.descs[i])
            err = max(err, np.abs(pp[i] - want).max() / np.abs(want).max())
        print(f"[edges] projection N={N} band {band} mask {mask} err {err:.2e}", flush=True)
        assert err < 1e-5
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("B,pairs", [(16, 8), (16, 11), (32, 5)])
def test_correlations_in_pieces(torch_gpu, ctx, B, pairs):
    """Results that fill one piece of the download exactly, leave a remainder in the second, and use the first slot
    again, against the same pairs one call each.  FP64 sums whose order may depend on the batch: 2B x 2B x B terms,
    1e-12 of the largest value."""
    from ettk_amd.lib import Plan

    g = np.random.default_rng(B + pairs)
    sig, pat = g.standard_normal((2, pairs, 2 * B, 2 * B))
    plan = Plan(ctx, default_params(32, B))
    try:
        got = plan.so3_correlate(sig, pat)
        for i in range(pairs):
            one = plan.so3_correlate(sig[i], pat[i])[0]
            err = np.abs(got[i] - one).max() / np.abs(one).max()
            assert err < 1e-12, (i, err)
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("N", [32, 96])
def test_wedge_at_lattice_rotations(torch_gpu, ctx, N):
    """Rotations by multiples of 45 degrees put the tilt axis along lattice directions, where a line of samples lies on
    both wedge planes and the last bit of the plane values decides: the distances are pinned to those the 27-sample
    stencil gave when every element evaluated its own.  FP32 transforms, 2^-24 per level of at most 24: 1.4e-6 of a
    score of at most 1; samples on the other side move these distances by 1e-5 and more."""
    import json
    import math
    from pathlib import Path

    from ettk_amd.lib import Plan

    def turn(axis, deg):
        a, r, (i, j) = math.radians(deg), np.eye(3), [(1, 2), (2, 0), (0, 1)][axis]
        r[i, i] = r[j, j] = math.cos(a)
        r[i, j], r[j, i] = -math.sin(a), math.sin(a)
        return r

    want = np.array(json.loads((Path(__file__).parent / "golden" / "wedge_lattice.json").read_text())[str(N)])
    rots = [turn(2, a) @ turn(0, b) @ turn(2, g) for a in (0, 45, 90, 135) for b in (0, 45, 90) for g in (0, 45, 270)]
    ref = blob_reference(N, seed=3)
    ps = make_particles(ref, 2, seed=4, half_wedge=(50, 60), snr=(0.5, 0.5), max_shift=1.0)
    t = np.tile(np.eye(4), (len(rots), 1, 1))
    t[:, :3, :3] = rots
    plan = Plan(ctx, default_params(N, 8, mask_radius=N / 2 - 3, square_mask=2))
    try:
        plan.set_reference(to_dev(torch_gpu, ref))
        d, _ = plan.ccc(to_dev(torch_gpu, ps.vols), ps.descs, np.arange(len(rots), dtype=np.int32) % 2, t)
        print(f"[edges] wedge N={N} err {np.abs(d - want).max():.2e}", flush=True)
        assert np.abs(d - want).max() < 2e-6
    finally:
        plan.close()
