"""The work that a program has this library do, as cases to be timed: each public block of the alignment path and two
whole calls, over the box sizes 32 .. 128 of the alignment, refinement and classification workloads.

A case is a dict of plain values; `op` names the entry point it calls:

  ccc       Plan.ccc: constrained CCC of (particle, transform) pairs, the inner step of every search and of Powell
  score     autograd.ccc_score, forward and backward: the score and pose gradient of one refinement step
  project   Plan.project: the S^2 projections of a batch of particles
  so3       Plan.so3_correlate: the SO(3) correlation of spherical images held on the host
  average   Plan.average: the wedge-weighted average of aligned particles
  extract   Context.extract: sub-volumes cut from a tomogram
  align     Plan.align, batched + adjoint: search, candidates, refinement, final CCC (a whole call)
  classify  Plan.mra_iteration, search only: alignment to K references, assignment, class averages (a whole call)

Particles are noisy, rotated, shifted copies of a sum of Gaussian blobs with a missing wedge, as the benchmark's.
"""
import math

import numpy as np
import torch

from ettk_amd.abi import Particle, default_params
from ettk_amd.autograd import ccc_score
from ettk_amd.lib import Context, Plan

TOL = 7.62939453125e-06  # the interpolator's floor tolerance, 2^-17


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one evaluation, as the plain form asks for them one after another: latency and launches
        dict(name="ccc_one_64", op="ccc", N=64, n=1, evals=1, mcf=True, wedge=True, window=8.0),
        # a peak round of a search over a small set: most of an alignment's time
        dict(name="ccc_64", op="ccc", N=64, n=24, evals=240, mcf=True, wedge=True, window=8.0),
        # a ragged last chunk of the smaller box of a mixed-size list, without the amplitude equalisation
        dict(name="ccc_48_ragged", op="ccc", N=48, n=7, evals=37, mcf=False, wedge=True, window=6.0),
        # the classification workload's box
        dict(name="ccc_128", op="ccc", N=128, n=6, evals=36, mcf=True, wedge=True, window=8.0),
        # one refinement step of the headline box: score, and its gradient through the adjoint
        dict(name="score_64", op="score", N=64, n=96),
        # the same at the box of the local-refinement workload
        dict(name="score_96", op="score", N=96, n=40),
        # the search's first half: projections of a chunk and a half of particles
        dict(name="project_64", op="project", N=64, B=32, n=48, mcf=True),
        # spherical correlation called on host buffers, as a program with its own spherical images does
        dict(name="so3_32", op="so3", B=32, pairs=6),
        # a class average
        dict(name="average_64", op="average", N=64, n=150),
        # cutting a list of picked positions out of a tomogram
        dict(name="extract_64", op="extract", N=64, n=60, nx=200, ny=256, nz=120),
        # the headline call on a small set
        dict(name="align_64", op="align", N=64, B=32, n=64),
        # one classification iteration
        dict(name="classify_64", op="classify", N=64, B=16, n=24, K=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["ccc", "ccc", "score", "project", "so3", "average", "extract", "align", "classify"])
    vox = 64 ** 3
    if op == "ccc":
        N = rng.choice([32, 48, 64, 96, 128])
        evals = _log(rng, 1, max(2, min(300, 240 * vox // N ** 3)))
        return dict(op=op, N=N, n=min(evals, rng.randint(1, 12)), evals=evals, mcf=rng.random() < 0.7,
                    wedge=rng.random() < 0.8, window=rng.choice([3.0, 4.0, 6.0, 8.0]))
    if op == "score":
        N = rng.choice([32, 48, 64, 96, 128])
        return dict(op=op, N=N, n=_log(rng, 1, max(2, min(200, 120 * vox // N ** 3))))
    if op == "project":
        N = rng.choice([32, 48, 64])
        return dict(op=op, N=N, B=rng.choice([8, 16, 32]), n=_log(rng, 1, min(64, 48 * vox // N ** 3)),
                    mcf=rng.random() < 0.7)
    if op == "so3":
        return dict(op=op, B=rng.choice([8, 16, 32]), pairs=rng.randint(1, 7))
    if op == "average":
        N = rng.choice([32, 48, 64, 96, 128])
        return dict(op=op, N=N, n=_log(rng, 2, min(300, 200 * vox // N ** 3)))
    if op == "extract":
        return dict(op=op, N=rng.randint(20, 72), n=_log(rng, 1, 50), nx=rng.randint(90, 260), ny=rng.randint(90, 260),
                    nz=rng.randint(60, 140))
    if op == "align":
        return dict(op=op, N=rng.choice([48, 64]), B=rng.choice([16, 32]), n=_log(rng, 1, 48))
    return dict(op=op, N=rng.choice([32, 48, 64]), B=rng.choice([8, 16]), n=rng.randint(8, 20), K=rng.randint(2, 3))


# ---------------------------------------------------------------------------------------------------- inputs
def _rotation(g):
    u1, u2, u3 = g.random(3)
    x, y = math.sqrt(1 - u1) * math.sin(2 * math.pi * u2), math.sqrt(1 - u1) * math.cos(2 * math.pi * u2)
    z, w = math.sqrt(u1) * math.sin(2 * math.pi * u3), math.sqrt(u1) * math.cos(2 * math.pi * u3)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])


def _turn(g, deg):
    """A rotation by `deg` degrees about a random axis."""
    a = g.standard_normal(3)
    a /= np.linalg.norm(a)
    K = np.array([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]])
    t = math.radians(deg)
    return np.eye(3) + math.sin(t) * K + (1 - math.cos(t)) * K @ K


def _blobs(g, N):
    d = g.standard_normal((40, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r = 24.0 * N / 64 * g.random(40) ** (1 / 3)
    return d * r[:, None], g.uniform(1.5, 4.0, 40), g.uniform(0.5, 1.0, 40)


def _volumes(centres, sigma, amp, N):
    """(n, N, N, N) [z, y, x]: sums of Gaussians at (n, 40, 3) centres (x, y, z)."""
    c = torch.from_numpy(np.asarray(centres)).cuda()
    s = torch.from_numpy(sigma).cuda()
    ar = torch.arange(N, dtype=torch.float64, device="cuda")
    e = torch.exp(-((ar - c[..., None]) ** 2) / (2 * s[:, None, None] ** 2))  # (n, 40, axis, N)
    a = torch.from_numpy(amp).cuda()
    out = torch.empty((c.shape[0], N, N, N), dtype=torch.float32, device="cuda")
    for q in range(c.shape[0]):
        x, y, z = e[q, :, 0], e[q, :, 1], e[q, :, 2] * a[:, None]
        zy = (z[:, :, None] * y[:, None, :]).reshape(z.shape[0], N * N)
        out[q] = (zy.T @ x).reshape(N, N, N)
    return out


class _Held:
    """What a program keeps: its context and plan, closed with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for h in (getattr(self, "plan", None), getattr(self, "ctx", None)):
            if h is not None:
                h.close()


def _particles(g, seed, blobs, N, n, wedge=True):
    """Particles of one blob model: volumes, limits of the missing wedges, true transforms."""
    centres, sigma, amp = blobs
    c = N / 2.0
    moved, truth, limits, snr = [], [], [], []
    for _ in range(n):
        R, s = _rotation(g), g.uniform(-4.0, 4.0, 3) * N / 64
        moved.append(c + s + centres @ R.T)
        T = np.eye(4)
        T[:3, :3], T[:3, 3] = R, s
        truth.append(T)
        h = float(np.float32(g.uniform(45.0, 70.0)))
        limits.append((-h, h) if wedge else (-90.0, 90.0))
        snr.append(g.uniform(0.05, 0.2))
    vols = _volumes(np.array(moved), sigma, amp, N)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    f = torch.fft.fftfreq(N, device="cuda", dtype=torch.float32) * N
    fx = torch.arange(N // 2 + 1, device="cuda", dtype=torch.float32)
    kz, kx = f[:, None, None], fx[None, None, :]
    for q in range(n):
        v = vols[q]
        if limits[q] != (-90.0, 90.0):
            n1, n2 = _normals(*limits[q])
            keep = (n1[0] * kx + n1[2] * kz) * (n2[0] * kx + n2[2] * kz) <= 0
            v = torch.fft.irfftn(torch.fft.rfftn(v) * keep, s=(N, N, N))
        noise = torch.randn((N, N, N), generator=gen, device="cuda", dtype=torch.float32)
        vols[q] = v + noise * torch.sqrt(v.var() / snr[q])
    return vols, limits, np.array(truth)


def _normals(lo, hi):
    lo, hi = max(lo, -90.0), min(hi, 90.0)
    if hi - lo >= 180:
        return None
    return [np.array([math.cos(-math.radians(90 - a)), 0.0, -math.sin(-math.radians(90 - a))]) for a in (hi, lo)]


def _inputs(case, seed):
    """The inputs of a case, from the seed alone."""
    g = np.random.default_rng(seed)
    op = case["op"]
    if op == "so3":
        n, B = case["pairs"], case["B"]
        # projections of noisy particles are positive and smooth: a few low orders, and noise
        th = (2 * np.arange(2 * B) + 1) * np.pi / (4 * B)
        ph = np.arange(2 * B) * np.pi / B
        img = np.zeros((2, n, 2 * B, 2 * B))
        for a in range(2):
            for q in range(n):
                v = 40.0 + g.standard_normal((2 * B, 2 * B))
                for _ in range(12):
                    l, m = g.integers(1, 9), g.integers(0, 6)
                    v = v + g.normal(0, 4) * np.sin(th[:, None]) ** m * np.cos(th[:, None] * l) * np.cos(
                        m * ph[None, :] + g.uniform(0, 6.28))
                img[a, q] = v
        return dict(sig=img[0], pat=img[1])
    if op == "extract":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        d = (case["nz"], case["ny"], case["nx"])
        tomo = torch.randn(d, generator=gen, device="cuda", dtype=torch.float32)
        k = torch.fft.rfftn(tomo)
        fz, fy = (torch.fft.fftfreq(m, device="cuda") for m in d[:2])
        fx = torch.fft.rfftfreq(d[2], device="cuda")
        r2 = fz[:, None, None] ** 2 + fy[None, :, None] ** 2 + fx[None, None, :] ** 2
        tomo = torch.fft.irfftn(k * torch.exp(-r2 * 20.0), s=d) * 30.0 + tomo  # blurred structure and noise
        lim = np.array([case["nx"], case["ny"], case["nz"]], dtype=float)
        # picked positions, some close enough to the border that their boxes reach outside
        pos = g.uniform(0.08, 0.92, (case["n"], 3)) * lim
        normal = np.stack([g.uniform(0, 180, case["n"]), g.uniform(-180, 180, case["n"]),
                           g.uniform(-180, 180, case["n"])], 1).astype(np.float32)
        cut = g.uniform(-4, 4, case["n"]).astype(np.float32)
        return dict(tomo=tomo.contiguous(), pos=pos, normal=normal, cut=cut)
    N, n = case["N"], case["n"]
    K = case.get("K", 1)
    models = [_blobs(g, N) for _ in range(K)]
    refs = torch.cat([_volumes((N / 2.0 + m[0])[None], m[1], m[2], N) for m in models])
    got = [_particles(g, seed * 16 + k, m, N, (n + K - 1 - k) // K, case.get("wedge", True))
           for k, m in enumerate(models)]
    vols = torch.cat([v[0] for v in got])
    limits = [x for v in got for x in v[1]]
    truth = np.concatenate([v[2] for v in got])
    more = {}
    if op == "ccc":
        e = case["evals"]
        idx = np.arange(e) % n
        t = np.tile(np.eye(4), (e, 1, 1))
        for q in range(e):  # candidates near the true rotation and their mirrored or false competitors
            t[q, :3, :3] = truth[idx[q], :3, :3] @ _turn(g, g.uniform(0, 8)) if q % 2 == 0 else _rotation(g)
        more = dict(idx=idx.astype(np.int32), t=t)
    elif op == "score":
        seeds = truth.copy()
        for q in range(n):  # poses as a coarse search leaves them
            seeds[q, :3, :3] = truth[q, :3, :3] @ _turn(g, 3.0)
            seeds[q, :3, 3] += g.uniform(-1, 1, 3)
        more = dict(seeds=seeds, x=g.uniform(-0.5, 0.5, (n, 6)).astype(np.float32),
                    up=g.uniform(0.5, 1.5, n).astype(np.float32))
    elif op == "average":
        w = g.uniform(0.5, 1.5, n).astype(np.float32)
        w[g.random(n) < 0.05] = 0.0
        w[0] = 1.0
        mats = truth.copy()
        for q in range(n):
            mats[q, :3, :3] = truth[q, :3, :3] @ _turn(g, 1.0)
        more = dict(w=w, mats=mats)
    return dict(refs=refs, vols=vols, limits=limits, truth=truth, **more)


def _params(case):
    N = case.get("N", 32)
    B = case.get("B", {32: 16, 48: 16, 64: 32, 96: 32, 128: 64}[N])
    return default_params(N, B, mcf=int(case.get("mcf", True)), missing_wedge=int(case.get("wedge", True)),
                          trans_restrict=case.get("window", 8.0))


def prepare(case, seed):
    x = _inputs(case, seed)
    op = case["op"]
    ctx = Context(0)
    if op == "so3":
        return _Held(op=op, ctx=ctx, plan=Plan(ctx, default_params(32, case["B"])), x=x)
    if op == "extract":
        descs = [Particle(normal=tuple(float(v) for v in x["normal"][q]), cut_offset=float(x["cut"][q]))
                 for q in range(case["n"])]
        out = torch.empty((case["n"],) + (case["N"],) * 3, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        return _Held(op=op, ctx=ctx, x=x, descs=descs, out=out, N=case["N"])
    plan = Plan(ctx, _params(case))
    descs = [Particle(lwedge=a, uwedge=b) for a, b in x["limits"]]
    torch.cuda.synchronize()  # the library's streams do not wait for torch's
    if op in ("ccc", "score", "align"):
        plan.set_reference(x["refs"][0])
    out = torch.empty_like(x["refs"][0])
    torch.cuda.synchronize()
    return _Held(op=op, ctx=ctx, plan=plan, x=x, descs=descs, out=out)


def run(s):
    x, op = s.x, s.op
    if op == "ccc":
        dist, t = s.plan.ccc(x["vols"], s.descs, x["idx"], x["t"])
        return {"distance": dist, "transform": t}
    if op == "score":
        p = torch.from_numpy(x["x"]).requires_grad_(True)
        val = ccc_score(s.plan, x["vols"], s.descs, np.arange(len(s.descs)), x["seeds"], p)
        val.backward(torch.from_numpy(x["up"]))
        return {"score": val.detach(), "gradient": p.grad}
    if op == "project":
        return s.plan.project(x["vols"], s.descs)
    if op == "so3":
        return s.plan.so3_correlate(x["sig"], x["pat"])
    if op == "average":
        s.plan.average(x["vols"], s.descs, x["w"], x["mats"], s.out)
        return s.out
    if op == "extract":
        s.ctx.extract(x["tomo"], x["pos"], s.descs, s.N, s.out)
        return s.out
    if op == "align":
        res = s.plan.align(x["vols"], s.descs, mode=2)
        # the rows of the distance array that getDistances fills: {distance, M00 .. M33} in float
        rows = np.array([(r.distance,) + tuple(r.matrix) for r in res], np.float32)
        return {"rows": rows, "angles": np.array([r.so3_angles[0][:] for r in res], np.float32),
                "overlap": np.array([r.overlap for r in res], np.float32),
                "candidates": np.array([r.n_cand for r in res], np.int32)}
    refs = x["refs"].clone()  # the iteration replaces its references by the class averages
    torch.cuda.current_stream().synchronize()
    cls, sel, dist, mats = s.plan.mra_iteration(refs, x["vols"], s.descs, type=3, form=2, top_percentage=0.8)
    return {"class": cls, "selected": sel, "distance": dist, "matrix": mats, "averages": refs}


def work(case):
    op = case["op"]
    if op == "so3":
        n = 2 * case["B"]
        # degree sums of the synthesis over the three orders, and a 2-D transform per slice
        flops = case["pairs"] * (8.0 * n * sum((2 * l + 1) ** 2 for l in range(case["B"])) + n * 10.0 * n * n * math.log2(n))
        return {"bytes": case["pairs"] * 8.0 * (n ** 3 + 2 * n * n), "flops": flops}
    if op == "extract":
        vox = case["n"] * float(case["N"]) ** 3
        return {"bytes": 4.0 * (vox + min(vox, case["nx"] * case["ny"] * case["nz"])), "flops": 170.0 * vox}
    N, n = case["N"], case["n"]
    v = float(N) ** 3
    fft = 2.5 * v * 3 * math.log2(N)  # one real 3-D transform
    ccc = 170.0 * v + 5 * fft + 40.0 * v
    if op == "ccc":
        return {"bytes": 4.0 * v * (n + 1) + 260.0 * case["evals"], "flops": case["evals"] * ccc}
    if op == "score":
        return {"bytes": 4.0 * v * (n + 1) + 450.0 * n, "flops": n * (3 * fft + 110.0 * v)}
    if op == "average":
        return {"bytes": 4.0 * v * (n + 1), "flops": n * (170.0 * v + fft + 6.0 * v) + fft}
    if op == "project":
        return {"bytes": 4.0 * (v * n + n * 4 * case["B"] ** 2), "flops": n * (170.0 * v + 2.5 * 8 * v * 3 * math.log2(2 * N))}
    B = 2.0 * case["B"]
    search = 170.0 * v + 20.0 * v * 3 * math.log2(2 * N) + 3 * 10.0 * B ** 3 * (B / 4 + 2 * math.log2(B))
    if op == "align":
        return {"bytes": 4.0 * v * (n + 1), "flops": n * (search + 11 * ccc + 20 * (3 * fft + 110.0 * v))}
    K = case["K"]
    return {"bytes": 4.0 * v * (n + 2 * K), "flops": n * K * (search + 10 * ccc + K * ccc)}


# ---------------------------------------------------------------------------------------------------- in 64 bits
def _rot(deg, ax):
    a = math.radians(float(deg))
    M, (i, j) = np.eye(4), {0: (1, 2), 2: (0, 1)}[ax]
    M[i, i] = M[j, j] = math.cos(a)
    M[i, j], M[j, i] = -math.sin(a), math.sin(a)
    return M


def _tricubic(vol, A, b, N):
    """Keys (a = -1/2) samples of vol [z, y, x] at A (i, j, k) + b for the output voxel (i, j, k), taps clamped to the
    border, and whether a sample lies within half a voxel of the volume."""
    dev = vol.device
    ar = torch.arange(N, dtype=torch.float64, device=dev)
    p = [A[r, 0] * ar[:, None, None] + A[r, 1] * ar[None, :, None] + A[r, 2] * ar[None, None, :] + b[r] for r in range(3)]
    size = vol.shape[::-1]
    ok = torch.ones((N, N, N), dtype=torch.bool, device=dev)
    at, w = [], []
    for r in range(3):
        ok &= (p[r] >= -0.5) & (p[r] <= size[r] - 0.5)
        q = p[r] + TOL
        fl = torch.floor(q)
        f = q - fl
        i = fl.long()
        at.append([(i - 1 + k).clamp(0, size[r] - 1) for k in range(4)])
        w.append([-0.5 * f * (f - 1) ** 2, ((1.5 * f - 1) * f - 1) * (f - 1), -((3 * f - 4) * f - 1) * 0.5 * f,
                  0.5 * f * f * (f - 1)])
    flat, out = vol.double().reshape(-1), torch.zeros((N, N, N), dtype=torch.float64, device=dev)
    for c in range(4):
        for d in range(4):
            row = (at[2][c] * size[1] + at[1][d]) * size[0]
            line = sum(w[0][k] * flat[row + at[0][k]] for k in range(4))
            out += w[2][c] * w[1][d] * line
    return out, ok


def _resliced(vol, fin, N, cut=0.0):
    """The particle at the pose fin, A(i, j, k) with i = x: valid voxels minus their mean, 0 elsewhere."""
    b = fin[:3, :3] @ np.array([-N / 2, -N / 2, -N / 2 - cut]) + fin[:3, 3] + N / 2
    v, ok = _tricubic(vol, fin[:3, :3], b, N)
    return torch.where(ok, v - v[ok].mean(), torch.zeros((), dtype=torch.float64, device=v.device))


def _smooth(A, sd, radius):
    """Separable Gaussian with clipped, renormalised taps."""
    taps = [math.exp(-x * x / (2 * sd * sd)) for x in range(-radius, radius + 1)]
    for ax in (2, 1, 0):
        out, norm = torch.zeros_like(A), torch.zeros(A.shape[ax], dtype=A.dtype, device=A.device)
        n = A.shape[ax]
        for q, t in zip(range(-radius, radius + 1), taps):
            lo, hi = max(0, -q), min(n, n - q)
            out.narrow(ax, lo, hi - lo).add_(A.narrow(ax, lo + q, hi - lo), alpha=t)
            norm[lo:hi] += t
        A = out / norm.reshape([-1 if a == ax else 1 for a in range(3)])
    return A


class _Tables:
    def __init__(self, p):
        N, dev = p.N, "cuda"
        self.N, self.H, self.p = N, N // 2 + 1, p
        c = torch.arange(N, dtype=torch.float64, device=dev) - N / 2
        self.c, self.ck = c, c[: self.H]
        r = torch.sqrt(c[:, None, None] ** 2 + c[None, :, None] ** 2 + c[None, None, :] ** 2)
        r1, r2 = p.mask_radius - p.mask_sigma / 2, min(N - 1, p.mask_radius + p.mask_sigma / 2)
        self.m1 = torch.where(r <= r1, 1.0, torch.where(r >= r2, 0.0, (1 + torch.cos(math.pi / (r2 - r1) * (r - r1))) / 2))
        box = torch.zeros((N, N, N), dtype=torch.float64, device=dev)
        q = p.square_mask
        box[q : N - q, q : N - q, q : N - q] = 1.0
        self.window = _smooth(box, 2.5, int(2.5 * (2.5 * 0.75)))
        par = torch.arange(N, device=dev)
        self.shift = 1.0 - 2.0 * ((par[:, None, None] + par[None, :, None] + par[None, None, :]) % 2).double()
        rad = r[:, :, : self.H] / (N // 2)
        f = torch.ones_like(rad)
        lo, hi, dl, dh = p.bp_lo, p.bp_hi, p.bp_lo_decay, p.bp_hi_decay
        f = torch.where(rad < lo, torch.exp(-((lo - rad) ** 2) / 2 / dl ** 2), f)
        f = torch.where(rad > hi, torch.exp(-((rad - hi) ** 2) / 2 / dh ** 2), f)
        f[N // 2, N // 2, self.H - 1] = 0.0
        self.filter = f

    def plane(self, v):
        """v . d over the centred half grid."""
        return v[0] * self.c[:, None, None] + v[1] * self.c[None, :, None] + v[2] * self.ck[None, None, :]

    def wedge(self, limits, fin):
        ns = _normals(*limits)
        if ns is None or not self.p.missing_wedge:
            return None
        R = np.linalg.inv(fin)[:3, :3]
        W = (self.plane(R @ ns[0]) * self.plane(R @ ns[1]) <= 0).double()
        return _smooth(W, 2.0, 1)


def _c2r(F, N):
    G = torch.fft.ifftn(F, dim=(0, 1), norm="forward")
    G[:, :, 0] = G[:, :, 0].real.to(G.dtype)
    G[:, :, N // 2] = G[:, :, N // 2].real.to(G.dtype)
    return torch.fft.irfft(G, n=N, dim=2, norm="forward")


def _exact_ccc(case, x):
    p = _params(case)
    T = _Tables(p)
    N, H = T.N, T.H
    hw = torch.full((H,), 2.0, dtype=torch.float64, device="cuda")
    hw[H - 1] = 1.0
    E = 2 * int(math.floor(max(2.0 * p.trans_restrict, 1.0))) + 1
    u = torch.arange(E, dtype=torch.float64, device="cuda") - E // 2
    sg = 1.0 - 2.0 * (T.c.long() % 2).double()
    A = torch.polar(torch.ones((E, N), dtype=torch.float64, device="cuda"), math.pi / N * u[:, None] * T.c[None, :]) * sg
    Kt = A[:, :H] * hw
    far = u[:, None, None] ** 2 + u[None, :, None] ** 2 + u[None, None, :] ** 2 >= max(2 * p.trans_restrict, 1.0) ** 2

    def weigh(F, fw):
        if p.mcf:
            m = F.abs()
            F = torch.where(m > 0, F / torch.sqrt(torch.where(m > 0, m, torch.ones_like(m))), F)
        F = F * fw
        F[N // 2, N // 2, H - 1] = 0
        return F / torch.sqrt((F.abs() ** 2 * hw).sum() / N ** 3)

    F1 = torch.fft.rfftn(x["refs"][0].double().permute(2, 1, 0) * T.window * T.shift)
    Mf = torch.fft.rfftn(T.m1 * T.shift)
    dist, mats = [], []
    for e in range(case["evals"]):
        q = int(x["idx"][e])
        W = T.wedge(x["limits"][q], x["t"][e])
        fw = T.filter if W is None else T.filter * W
        r1 = _c2r(weigh(F1, fw), N)
        k1 = (r1 * r1 * T.m1).sum()
        F1m = torch.fft.rfftn(r1 * T.m1)
        X2 = weigh(torch.fft.rfftn(_resliced(x["vols"][q], x["t"][e], N) * T.window * T.shift), fw)
        Q = torch.fft.rfftn(_c2r(X2, N) ** 2 * T.shift)
        C = (-Mf * Q.conj() + 2.0 * N ** 3 * F1m * X2.conj()) * T.shift[:, :, :H]
        G = torch.einsum("xi,ijk->xjk", A, C)
        G = torch.einsum("yj,xjk->xyk", A, G)
        V = torch.einsum("zk,xyk->xyz", Kt, G).real * (8.0 / (2.0 * N) ** 3)
        V = torch.where(far, torch.full_like(V, -1e300), V)
        best, at = V.reshape(-1).max(0)
        peak = max(0.0, float(k1 - best))
        if p.overlap_norm and p.missing_wedge:
            peak *= float(T.filter.sum() / fw.sum())
        dist.append(peak / (2.0 * N) ** 6)
        at = int(at)
        sh = (np.array([at // (E * E), at // E % E, at % E]) - (E - 1) / 2) / 2
        M = x["t"][e].copy()
        M[:3, 3] -= M[:3, :3] @ sh
        mats.append(M)
    return {"distance": np.array(dist), "transform": np.array(mats)}


def _exact_score(case, x):
    p = _params(case)
    T = _Tables(p)
    N, H = T.N, T.H
    ar = torch.arange(N, dtype=torch.float64, device="cuda") - N / 2
    ref = x["refs"][0].double()
    flat = (ref - ref.mean()).reshape(-1)
    ch = torch.full((H,), 2.0, dtype=torch.float64, device="cuda")
    ch[0] = ch[H - 1] = 1.0
    win = T.window * T.shift
    val, grad = [], []
    for q in range(case["n"]):
        th = torch.from_numpy(x["x"][q].astype(np.float64)).cuda().requires_grad_(True)
        a = th[:3] * (math.pi / 180)
        c, s, o, z = torch.cos(a), torch.sin(a), torch.ones_like(a[0]), torch.zeros_like(a[0])
        Rx = torch.stack([o, z, z, z, c[0], -s[0], z, s[0], c[0]]).reshape(3, 3)
        Ry = torch.stack([c[1], z, s[1], z, o, z, -s[1], z, c[1]]).reshape(3, 3)
        Rz = torch.stack([c[2], -s[2], z, s[2], c[2], z, z, z, o]).reshape(3, 3)
        seed = torch.from_numpy(x["seeds"][q]).cuda()
        R = seed[:3, :3] @ Rx @ Ry @ Rz
        Ri = torch.linalg.inv(R)
        off = -Ri @ (seed[:3, 3] + th[3:])
        pos = [Ri[r, 0] * ar[None, None, :] + Ri[r, 1] * ar[None, :, None] + Ri[r, 2] * ar[:, None, None] + off[r] + N / 2
               for r in range(3)]
        lo = [torch.floor(v.detach()) for v in pos]
        f = [v - l for v, l in zip(pos, lo)]
        i0 = [l.long().clamp(0, N - 1) for l in lo]
        i1 = [(l.long() + 1).clamp(0, N - 1) for l in lo]
        img = 0.0
        for b in range(8):
            i = [(i1 if b >> r & 1 else i0)[r] for r in range(3)]
            w = [f[r] if b >> r & 1 else 1 - f[r] for r in range(3)]
            img = img + w[0] * w[1] * w[2] * flat[(i[2] * N + i[1]) * N + i[0]]
        Hw = T.filter
        ns = _normals(*x["limits"][q])
        if ns is not None:  # the half axis is x, the slow axis z
            side = [n[0] * T.ck[None, None, :] + n[1] * T.c[None, :, None] + n[2] * T.c[:, None, None] for n in ns]
            Hw = torch.where(side[0] * side[1] > 0, torch.zeros_like(Hw), Hw)
        v = x["vols"][q].double()
        X1, X2 = torch.fft.rfftn(img * win) * Hw, torch.fft.rfftn((v - v.mean()) * win) * Hw

        def dot(A, B):
            return ((A.real * B.real + A.imag * B.imag) * ch).sum()

        S = dot(X1, X2) / torch.sqrt(dot(X1, X1) * dot(X2, X2))
        S.backward()
        val.append(float(S.detach()))
        grad.append((th.grad * float(x["up"][q])).cpu().numpy())
    return {"score": np.array(val), "gradient": np.array(grad)}


def _exact_project(case, x):
    p = _params(case)
    T = _Tables(p)
    N, B = T.N, case["B"]
    M, n = 2 * N, 2 * B
    bandL, bandU = max(4, math.ceil(np.float32(p.bp_lo) * np.float32(M - 1))), math.ceil(min(0.5, p.bp_hi) * (M - 1))
    phi = math.pi / 4 / B + torch.arange(n, dtype=torch.float64, device="cuda") * (math.pi / 2 / B)
    th = torch.arange(n, dtype=torch.float64, device="cuda") * (math.pi / B)
    r = torch.arange(bandL, bandU + 1, dtype=torch.float64, device="cuda")
    sp = torch.sin(phi)[:, None, None]
    p3 = torch.stack([sp * torch.cos(th)[None, :, None] * r, sp * torch.sin(th)[None, :, None] * r,
                      (torch.cos(phi)[:, None, None] * r).expand(n, n, len(r))]) + M / 2 + TOL
    fl = torch.floor(p3)
    f, i0 = p3 - fl, fl.long() - 1
    w = [-0.5 * f * (f - 1) ** 2, ((1.5 * f - 1) * f - 1) * (f - 1), -((3 * f - 4) * f - 1) * 0.5 * f, 0.5 * f * f * (f - 1)]
    par = torch.arange(M, device="cuda")
    sg = 1.0 - 2.0 * ((par[:, None, None] + par[None, :, None] + par[None, None, :]) % 2).double()
    out = []
    for q in range(case["n"]):
        img = _resliced(x["vols"][q], np.eye(4), N)
        img = (img - img.mean()) * T.m1 + img.mean()
        A = img[0, 0, 0].expand(M, M, M).clone()
        A[:N, :N, :N] = img
        F = torch.fft.rfftn(A * sg).abs()
        A[:, :, : N + 1] = torch.sqrt(F) if p.mcf else F
        A[0] = 0.0
        A[1:, 1:, N + 1 :] = torch.flip(A[1:, 1:, 1:N], (0, 1, 2))  # the mirrored half as the metric fills it
        flat, s = A.reshape(-1), 0.0
        for a in range(4):
            for b in range(4):
                for c in range(4):
                    at = (((i0[0] + a) % M) * M + (i0[1] + b) % M) * M + (i0[2] + c) % M
                    s = s + w[a][0] * w[b][1] * w[c][2] * flat[at]
        out.append(s.sum(-1).cpu().numpy())
    return np.array(out)


def _exact_so3(case, x):
    B = case["B"]
    n, W = 2 * B, 2 * B - 1
    th = (2 * np.arange(n) + 1) * np.pi / (4 * B)
    k = np.arange(B)
    dh = 2.0 / B * np.sin(th) * (np.sin(np.outer(th, 2 * k + 1)) / (2 * k + 1)).sum(1)
    P = np.zeros((n, B, B))  # orthonormal Legendre functions, Condon-Shortley phase
    for m in range(B):
        P[:, m, m] = math.sqrt(1 / (4 * math.pi)) if m == 0 else -math.sqrt((2 * m + 1) / (2 * m)) * np.sin(th) * P[:, m - 1, m - 1]
        for l in range(m + 1, B):
            a = math.sqrt((4 * l * l - 1) / (l * l - m * m))
            b = math.sqrt(((l - 1) ** 2 - m * m) / (4 * (l - 1) ** 2 - 1)) if l > m + 1 else 0.0
            P[:, l, m] = a * (np.cos(th) * P[:, l - 1, m] - (b * P[:, l - 2, m] if l > m + 1 else 0.0))

    def coef(f):
        F = np.fft.fft(f, axis=1) * (dh * 2 * np.pi / n)[:, None]
        c = np.zeros((B, W), complex)
        for l in range(B):
            for m in range(l + 1):
                c[l, m + B - 1] = (F[:, m] * P[:, l, m]).sum()
                c[l, -m + B - 1] = (F[:, -m % n] * P[:, l, m]).sum() * (-1) ** m
        return c

    d = np.zeros((B, n, W, W))  # Wigner d at the n angles, from the spectrum of J_y
    for l in range(B):
        m = np.arange(-l, l)
        up = 0.5 * np.sqrt(l * (l + 1) - m * (m + 1))
        J = np.zeros((2 * l + 1, 2 * l + 1), complex)
        J[np.arange(1, 2 * l + 1), np.arange(2 * l)] = -1j * up
        J[np.arange(2 * l), np.arange(1, 2 * l + 1)] = 1j * up
        ev, V = np.linalg.eigh(J)
        ev = np.round(ev)
        s = slice(B - 1 - l, B + l)
        d[l][:, s, s] = np.einsum("ab,tb,cb->tac", V, np.exp(-1j * np.outer(th, ev)), V.conj(), optimize=True).real
    sgn = (-1.0) ** np.abs(np.add.outer(np.arange(W), np.arange(W)))
    at = np.arange(-(B - 1), B) % n
    out = np.zeros((case["pairs"], n, n, n))
    for q in range(case["pairs"]):
        cs, cp = coef(x["sig"][q])[:, ::-1], coef(x["pat"][q])[:, ::-1].conj()
        lw = np.sqrt((2 * np.arange(B) + 1) / (8 * np.pi ** 2))
        S = np.einsum("la,lb,ltab->tab", cs * lw[:, None], cp, d, optimize=True) * sgn
        G = np.zeros((n, n, n), complex)
        G[np.ix_(np.arange(n), at, at)] = S
        out[q] = np.fft.fft2(G, axes=(1, 2)).real.transpose(1, 0, 2)
    return out


def _exact_average(case, x):
    N = case["N"]
    par = torch.arange(N, device="cuda")
    sg = 1.0 - 2.0 * ((par[:, None, None] + par[None, :, None] + par[None, None, :]) % 2).double()
    num, den = 0.0, 0.0
    for q in range(case["n"]):
        if x["w"][q] == 0:
            continue
        F = torch.fft.rfftn(_resliced(x["vols"][q], x["mats"][q], N) * sg)
        num = num + float(x["w"][q]) * F.abs() * F
        den = den + abs(float(x["w"][q])) * F.abs()
    F = torch.where(den > 0, num / den, torch.zeros_like(num))
    F[N // 2, N // 2, N // 2] = 0
    A = _c2r(F, N) / N ** 3 * sg
    return (A / torch.sqrt((A * A).mean())).permute(2, 1, 0).contiguous()


def _exact_extract(case, x):
    N, out = case["N"], []
    for q in range(case["n"]):
        nrm = x["normal"][q]
        fin = _rot(-nrm[2], 2) @ _rot(-nrm[0], 0) @ _rot(-nrm[1], 2)
        b = fin[:3, :3] @ np.array([-N / 2, -N / 2, -N / 2 - float(x["cut"][q])]) + x["pos"][q]
        v, ok = _tricubic(x["tomo"], fin[:3, :3], b, N)
        v = torch.where(ok, v - v[ok].mean(), torch.zeros((), dtype=torch.float64, device=v.device))
        out.append(v.permute(2, 1, 0))
    return torch.stack(out)


def exact(case, seed):
    f = {"ccc": _exact_ccc, "score": _exact_score, "project": _exact_project, "so3": _exact_so3,
         "average": _exact_average, "extract": _exact_extract}.get(case["op"])
    # a whole alignment or classification has no value of its own in 64 bits: it searches, and its answers turn on choices
    return None if f is None else f(case, _inputs(case, seed))
