"""The staged box of the tricubic tiles (tile_box, tricubic.hpp) holds every sample's stencil, replayed in FP32.

Per input axis the kernels stage the voxels floor(mn - margin) - 1 .. floor(mn + ext + margin) + 2 of a tile and index the
box without a clamp: the 4 taps of a sample at p start at floor(p + 2^-17) - 1.  Positions and bounds are rounded to FP32
here as there, each sum both with every product rounded by itself and fused in either order.  Only a tile's extreme corners
can leave the box, so those are drawn, within 1.5 units in the last place of a whole coordinate, where the rounding
decides.  The margins are read from the header, so the rule under test is the compiled one.
"""
import re
from pathlib import Path

import numpy as np
import pytest

f32 = np.float32
HEADER = (Path(__file__).resolve().parents[1] / "ettk_amd" / "csrc" / "tricubic.hpp").read_text()


def constant(name, default):
    m = re.search(rf"\b{name} = ([0-9.e+-]+)f[,;]", HEADER)
    return f32(m.group(1)) if m else f32(default)


def margin(n, N):
    """tile_margin(n, N); without a relative part, as k_reslice for N <= 128, where N is None."""
    least = constant("kMarginMin", 1e-3)
    if N is None:
        return least
    return max(least, constant("kMarginUlp", 0) * (f32(n) + f32(4) * f32(N)) + constant("kMarginSmall", 0))


def fma(a, b, c):
    return (np.float64(a) * np.float64(b) + np.float64(c)).astype(f32)


def position(m, x, y, z, order):
    if order == "rounded":
        return ((m[0] * x + m[1] * y) + m[2] * z) + m[3]
    if order == "fused":
        return fma(m[2], z, fma(m[1], y, m[0] * x)) + m[3]
    return fma(m[2], z, fma(m[0], x, m[1] * y)) + m[3]


def escapes(first, last, N, mg, order, scale=1.0, count=1_000_000, seed=0):
    """Samples whose taps leave the staged box, and the widest box, over rigid rows (times `scale`)."""
    g = np.random.default_rng(seed)
    v = g.standard_normal((3, count))
    v *= scale / np.linalg.norm(v, axis=0)
    m = [c.astype(f32) for c in v]
    tile = [(8 * g.integers(0, max(N // 8, 1), count)).astype(f32) for _ in range(3)]
    near = np.spacing(f32(last)) * g.uniform(-1.5, 1.5, count)
    whole = np.floor(g.uniform(first, last, count))
    ext = f32(7) * ((np.abs(m[0]) + np.abs(m[1])) + np.abs(m[2]))
    low = (np.minimum(m[0], f32(0)) + np.minimum(m[1], f32(0))) + np.minimum(m[2], f32(0))
    out, width = 0, 0
    for top in (True, False):
        corner = [tile[a] + np.where((m[a] > 0) == top, f32(7), f32(0)) for a in range(3)]
        at = sum(m[a].astype(np.float64) * corner[a] for a in range(3))
        row = m + [(whole + near - at).astype(f32)]
        c0 = position(row, *tile, order)
        mn = c0 + f32(7) * low if order == "rounded" else fma(f32(7), low, c0)
        lo, hi = np.floor(mn - mg) - 1, np.floor((mn + ext) + mg) + 2
        tap = np.floor(position(row, *corner, order) + f32(2.0 ** -17)) - 1
        out += int(np.count_nonzero((tap < lo) | (tap + 3 > hi)))
        width = max(width, int((hi - lo).max()) + 1)
    return out, width


@pytest.mark.parametrize("order", ["rounded", "fused", "fused the other way"])
@pytest.mark.parametrize("first,last,N", [(0, 120, 16), (900, 1020, 64), (2050, 4090, 256), (4100, 8180, 1024),
                                          (8200, 9990, 128), (8200, 9990, 1024), (60000, 99990, 512)])
def test_extraction_boxes_hold_every_stencil(first, last, N, order):
    out, width = escapes(first, last, N, margin(last + 10, N), order)
    assert out == 0
    assert width <= 17


@pytest.mark.parametrize("order", ["rounded", "fused", "fused the other way"])
@pytest.mark.parametrize("N", [16, 48, 64, 96, 128])
def test_reslice_boxes_hold_every_stencil(N, order):
    out, width = escapes(0, N, N, margin(N, None), order)
    assert out == 0
    assert width <= 17


@pytest.mark.parametrize("N", [128, 1024])
def test_steep_rows_stay_covered(N):
    """Rows of absolute sum up to 2, the steepest whose box can fit (their corners are 14 voxels apart)."""
    out, _ = escapes(0, N, N, margin(N, None if N == 128 else N), "rounded", scale=2.0 / np.sqrt(3.0))
    assert out == 0
