"""CPU check of the LDS footprint boxes of every kernel that uses one: the
backprojector's z-runs (fdk_backproject.hip) and the adjoint's 32-bit and 64-bit sums
(fdk_adjoint.hip), whose LDS accesses have no other bounds than these boxes.

The rule of fdk_box.hpp is evaluated in float32 for blocks of `edge` x `edge` columns x
`zr` slices and boxes of W columns and H rows, and for every active column and slice
both taps must lie inside the box; where a box is flagged as inside the detector, the
skipped range tests must hold.
"""
import os
import re

import numpy as np
import pytest

import oracle as O
from test_footprint import CASES, f32, fma

# (edge, zr, W, H)
KERNELS = {
    "bp_zr8": (16, 8, 64, 64), "bp_zr16": (16, 16, 64, 64), "bp_zr24": (16, 24, 64, 80),
    "bp_zr32": (16, 32, 64, 96), "bp_low_box": (16, 8, 64, 16),
    "adjoint_tile": (32, 64, 108, 160), "adjoint_both_boxes": (32, 64, 136, 254),
    "adjoint_block": (16, 64, 108, 160), "adjoint_64_bit": (16, 64, 68, 252),
}
ALIGN = 4


def test_the_boxes_are_the_kernels():
    src = open(os.path.join(os.path.dirname(O.__file__), "..", "tomokvas_amd", "csrc",
                            "fdk_adjoint.hip")).read()
    tiles = re.findall(r"constexpr int T = (\d+), W = (\d+), H = (\d+);", src)
    words = eval(re.search(r"constexpr int FP_WORDS = ([0-9 *]+);", src).group(1))
    W2 = int(re.search(r"constexpr int FP_W2 = (\d+)", src).group(1))
    t32, t64 = (tuple(map(int, t)) for t in tiles)
    assert KERNELS["adjoint_tile"] == (t32[0], 64) + t32[1:]
    assert KERNELS["adjoint_block"] == (16, 64) + t32[1:]
    assert KERNELS["adjoint_64_bit"] == (t64[0], 64) + t64[1:]
    assert KERNELS["adjoint_both_boxes"] == (t32[0], 64, W2, words // (W2 + 1))
    # cells of a box, pitch W + 1: 4 bytes twice, 8 bytes once, 4 bytes once
    assert 2 * t32[2] * (t32[1] + 1) <= words and 2 * t64[2] * (t64[1] + 1) <= words


def footprint(c, s, xs, ys, azlo, azhi, g, W, H):
    """(bu0, bv0, bw, bh, inner_v, inner_u); bw as the kernel's, without its flags."""
    cX, cZ, D = f32(g.cX), f32(g.cZ), f32(g.D)
    us, Us = [], []
    for aX in xs:
        for aY in ys:
            S, T = fma(aX, c, f32(aY * s)), fma(aY, c, f32(-(aX * s)))
            den = f32(D - S)
            if not den > f32(0.01) * D:
                return 0, 0, -1, 0, False, False
            Us.append(f32(D / den))
            us.append(fma(T, Us[-1], cX))
    p = [f32(a * U) for a in (azlo, azhi) for U in (min(Us), max(Us))]
    vlo, vhi = f32(min(p) + cZ), f32(max(p) + cZ)
    cl = lambda x, n: int(np.floor(min(max(x, -8.0), n + 8.0)))   # noqa: E731
    bu0, bu1 = max(cl(min(us), g.Nu) - 2, 0) & ~(ALIGN - 1), min(cl(max(us), g.Nu) + 3, g.Nu - 1)
    bv0, bv1 = max(cl(vlo, g.Nv) - 2, 0), min(cl(vhi, g.Nv) + 3, g.Nv - 1)
    bw, bh = bu1 - bu0 + 1, bv1 - bv0 + 1
    if bw <= 0 or bh <= 0:
        return 0, 0, 0, 0, False, False
    if bw >= W or bh >= H:
        return 0, 0, -1, 0, False, False
    m = f32(0.02)
    return (bu0, bv0, bw, bh, bool(vlo >= m and vhi <= f32(g.Nv - 1) - m),
            bool(min(us) >= m and max(us) <= f32(g.Nu - 1) - m))


@pytest.mark.parametrize("kernel", list(KERNELS))
@pytest.mark.parametrize("name", list(CASES))
def test_taps_lie_inside_the_box(name, kernel):
    make, tile_stride, ang_stride = CASES[name]
    edge, zr, W, H = KERNELS[kernel]
    tile_stride = max(1, tile_stride * 16 // edge)
    g = make()
    ax, ay, az = [a.astype(f32) for a in O.axis_tables(g)]
    step = az[1] - az[0]
    n = (len(az) + 63) // 64 * 64 + 64        # the host's table, padded past Nz
    az = np.concatenate([az, (az[-1] + step * np.arange(1, n - len(az) + 1)).astype(f32)])
    s64, c64 = O.sincos(g)
    cX, cZ, D = f32(g.cX), f32(g.cZ), f32(g.D)
    kinds = dict(staged=0, empty=0, beyond=0, inner_u=0)
    for z0 in range(0, g.Nz, zr):
        azr = az[z0:z0 + zr]
        for y0 in range(0, g.Ny, edge * tile_stride):
            for x0 in range(0, g.Nx, edge * tile_stride):
                xs, ys = ax[x0:x0 + edge], ay[y0:y0 + edge]
                X, Y = (a.ravel() for a in np.meshgrid(xs, ys))
                inside = X.astype(np.float64) ** 2 + Y.astype(np.float64) ** 2 < 0.25 * g.Nu ** 2
                if not inside.any():
                    continue
                for b in range(0, g.Nang, ang_stride):
                    c, s = f32(c64[b]), f32(s64[b])
                    bu0, bv0, bw, bh, inner_v, inner_u = footprint(
                        c, s, (xs[0], xs[-1]), (ys[0], ys[-1]), min(azr[0], azr[-1]),
                        max(azr[0], azr[-1]), g, W, H)
                    if bw < 0:
                        kinds["beyond"] += 1
                        continue
                    S, T = fma(X, c, (Y * s).astype(f32)), fma(Y, c, (-(X * s)).astype(f32))
                    U = (D / (D - S)).astype(f32)
                    u = fma(T, U, cX)
                    act = inside & (u >= 0) & (u <= f32(g.Nu - 1))
                    v = fma(azr[None, :], U[act, None], cZ)
                    ok = (v >= 0) & (v <= f32(g.Nv - 1))
                    where = (name, kernel, z0, y0, x0, b)
                    if bw == 0:
                        kinds["empty"] += 1
                        assert not ok.any(), where
                        continue
                    kinds["staged"] += 1
                    if inner_u:
                        # the backprojector then takes every column of the cylinder
                        kinds["inner_u"] += 1
                        assert act[inside].all(), where
                    if not act.any():
                        continue
                    col = u[act].astype(np.int64) - bu0
                    assert col.min() >= 0 and col.max() + 1 <= bw <= W - 1, where
                    # columns past the lanes that load the box read as zeros: only taps
                    # past the detector may
                    loaded = (bw + 3) // 4 * 4
                    assert ((col + 1 < loaded) | (bu0 + col + 1 >= g.Nu)).all(), where
                    if inner_v:
                        assert ok.all(), where
                    row = (np.floor(v).astype(np.int64) - bv0)[ok]
                    if row.size:
                        assert row.min() >= 0 and row.max() + 1 <= bh <= H - 1, where
    assert kinds["staged"] + kinds["beyond"] > 0
    if kernel not in ("bp_low_box",) and name in ("small", "cfg1"):
        assert kinds["staged"] > 0 and kinds["beyond"] == 0, kinds
    if name == "wide" and kernel.startswith("bp"):
        # voxels of four samples: boxes beyond the LDS tile beside staged ones (the
        # adjoint's hold this detector's 96 rows)
        assert kinds["beyond"] > 0, kinds


def may_be_wide(g):
    """may_be_wide() of fdk_adjoint.hip."""
    across = 21.3 * g.scale
    r = 0.5 * g.Nu + across
    if g.D <= r:
        return True
    U = g.D / (g.D - r)
    az_max = g.scale * (0.5 * g.Nz + abs(g.cz) + 64.)
    return (63 * g.scale * U + az_max * across * U * U / g.D + 8. >= 128 or
            across * (U + r * U * U / g.D) + 11. >= 64)


@pytest.mark.parametrize("seed", range(40))
def test_blocks_of_a_narrow_scan_are_narrow(seed):
    """Where may_be_wide says no, no block with a column in the cylinder has a footprint
    of 64 columns or 128 rows; the scans are drawn about the line between the two."""
    from gpu_util import ogeom, scan

    rng = np.random.default_rng(seed)
    scale = float(rng.uniform(0.8, 2.1))
    n = int(rng.integers(20, 120))
    Nu = int(n * scale * rng.uniform(0.9, 1.5)) + 8
    g = ogeom(scan(Nu, int(rng.integers(100, 400)), 13, n, n, int(rng.integers(30, 200)),
                   D=float(Nu * np.exp(rng.uniform(np.log(0.7), np.log(20.)))), tau=0.1, scale=scale,
                   cz=float(rng.uniform(-20, 20)), rot=float(rng.uniform(0, 1))))
    ax, ay, az = [a.astype(f32) for a in O.axis_tables(g)]
    az = np.concatenate([az, (az[-1] + (az[1] - az[0]) * np.arange(1, 129)).astype(f32)])
    s64, c64 = O.sincos(g)
    wide = False
    for z0 in range(0, g.Nz, 64):
        zs = az[z0], az[z0 + 63]
        for y0 in range(0, g.Ny, 16):
            for x0 in range(0, g.Nx, 16):
                xs, ys = ax[x0:x0 + 16], ay[y0:y0 + 16]
                if np.min(np.abs(xs)) ** 2 + np.min(np.abs(ys)) ** 2 >= 0.25 * g.Nu ** 2:
                    continue
                for b in range(g.Nang):
                    wide = wide or footprint(f32(c64[b]), f32(s64[b]), (xs[0], xs[-1]),
                                             (ys[0], ys[-1]), min(zs), max(zs), g, 64, 128)[2] < 0
    assert may_be_wide(g) or not wide
