"""The FP32 adjoint on volumes whose voxels differ widely in size, and on voxels
that are not finite, against the same splats summed in double."""
import numpy as np
import pytest

import oracle as O
from gpu_util import ogeom, say, scan, stages

pytestmark = pytest.mark.gpu

f32, f64 = np.float32, np.float64


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


def splats(g, x):
    """The adjoint of x [Nz][Ny][Nx] with the FP32 sample positions, its weights and
    sums in double."""
    og = ogeom(g)
    ax, ay, az = (a.astype(f32) for a in O.axis_tables(og))
    s64, c64 = O.sincos(og)
    cX, cZ, D = f32(g.cX), f32(g.cZ), f32(g.D)
    fma = lambda a, b, c: (f64(a) * f64(b) + f64(c)).astype(f32)   # noqa: E731
    fscale = f64(f32(g.dbeta) * (f32(1) / f32(og.p)))
    Y, X = np.meshgrid(ay, ax, indexing="ij")
    inside = X.astype(f64) ** 2 + Y.astype(f64) ** 2 < 0.25 * g.Nu * g.Nu
    out = np.zeros((g.Nv + 1, g.Nang, g.Nu + 1))
    for b in range(g.Nang):
        c, s = f32(c64[b]), f32(s64[b])
        S, T = fma(X, c, Y * s), fma(Y, c, -(X * s))
        U = (D / (D - S)).astype(f32)
        u = fma(T, U, cX)
        act = inside & (u >= 0) & (u <= f32(g.Nu - 1))
        v = fma(az[:, None], U[act][None], cZ)
        ok = (v >= 0) & (v <= f32(g.Nv - 1))
        iu = np.broadcast_to(np.floor(u[act]).astype(int), v.shape)[ok]
        fu = np.broadcast_to(u[act].astype(f64) - np.floor(u[act]), v.shape)[ok]
        w = np.broadcast_to(U[act].astype(f64) ** 2, v.shape)[ok] * x[:, act].astype(f64)[ok] * fscale
        v = v[ok].astype(f64)
        iv, fv = np.floor(v).astype(int), v - np.floor(v)
        flat = np.zeros((g.Nv + 1) * (g.Nu + 1))
        for dv, wv in ((0, 1 - fv), (1, fv)):
            for du, wu in ((0, 1 - fu), (1, fu)):
                flat += np.bincount((iv + dv) * (g.Nu + 1) + iu + du, w * wv * wu, flat.size)
        out[:, b] = flat.reshape(g.Nv + 1, g.Nu + 1)
    return out[:g.Nv, :, :g.Nu]


def project(torch, g, x):
    return stages(g).forward_project(torch.from_numpy(x).cuda()).double().cpu().numpy()


# Footprints of 16 x 16 columns x 64 slices beyond 64 x 128 samples at every angle
# (two samples per voxel, and with the source near), or at some angles only, where the
# others are summed in 32 bits per block
WIDE = {
    "two": (dict(Nu=140, Nv=150, Nang=8, Nx=64, Ny=61, Nz=66, D=900.0, scale=2.0), "voxel", 5e-7),
    "some": (dict(Nu=130, Nv=170, Nang=9, Nx=64, Ny=64, Nz=64, D=330.0, scale=1.75), "block", 1e-6),
    "near": (dict(Nu=150, Nv=230, Nang=9, Nx=60, Ny=64, Nz=70, D=230.0, scale=2.0), "block", 1e-6),
}


# A splat takes at most 7 FP32 roundings, about 1e-7 of it together, and a sample is
# the FP32 sum of some 64 of them in any order, again 1e-7: 5e-7 is three times that.
# Sums in 32 bits: see below.
@pytest.mark.parametrize("ratio", [1.0, 1e2, 1e4, 1e6, 1e9, 1e20])
@pytest.mark.parametrize("case", list(WIDE))
def test_wide_footprints_keep_relative_errors(torch, case, ratio):
    """Samples that one large voxel, or its block, does not reach are as accurate as
    without it."""
    kw, reach, tol = WIDE[case]
    g = scan(**kw, tau=0.1)
    x = np.random.default_rng(7).standard_normal((g.Nz, g.Ny, g.Nx)).astype(f32)
    x[20, 25, 23] += ratio
    near = np.zeros_like(x)
    if reach == "voxel":
        near[20, 25, 23] = 1
    else:
        near[:64, 16:32, 16:32] = 1
    say(f"wide footprints {case}, ratio {ratio:g}")
    got, ref = project(torch, g, x), splats(g, x)
    far = splats(g, near) == 0
    err = O.rel_rmse(got[far], ref[far])
    say(f"  error of the samples out of its reach {err:.2e}, of all {O.rel_rmse(got, ref):.2e}")
    assert far.any() and err <= tol


NARROW = {
    "one": dict(Nu=72, Nv=80, Nang=9, Nx=64, Ny=64, Nz=64, D=900.0),
    "fine": dict(Nu=90, Nv=120, Nang=7, Nx=70, Ny=50, Nz=70, D=700.0, scale=1.25),
}


# the step of the fixed-point sums is at most 2^-23 of a block's largest voxel (its
# bound is below 2^7 of it), 0.3 steps a splat whose weight is 1/4 on average: 4e-7
# of the largest voxel at most for normal voxels of up to 4.5; a third of that beside
# the FP32 roundings in practice.  1e-6 bounds both.
@pytest.mark.parametrize("ratio", [1.0, 1e1, 1e2, 1e4, 1e6])
@pytest.mark.parametrize("at", [(3, 5), (25, 19), (40, 33)])
@pytest.mark.parametrize("case", list(NARROW))
def test_a_large_voxel_sets_the_step_of_its_own_columns(torch, case, at, ratio):
    """Samples that the 16 x 16 columns x 64 slices around a large voxel do not reach
    are as accurate as without it."""
    g = scan(**NARROW[case], tau=0.1)
    x = np.random.default_rng(8).standard_normal((g.Nz, g.Ny, g.Nx)).astype(f32)
    x[30, at[0], at[1]] = 5 * ratio
    block = np.zeros_like(x)
    y0, x0 = at[0] // 16 * 16, at[1] // 16 * 16
    block[:64, y0:y0 + 16, x0:x0 + 16] = 1
    say(f"large voxel {case} at {at}, ratio {ratio:g}")
    got, ref = project(torch, g, x), splats(g, x)
    far = splats(g, block) == 0
    err = O.rel_rmse(got[far], ref[far])
    say(f"  error of the samples out of its block's reach {err:.2e}")
    assert far.any() and err <= 1e-6


# 32-bit sums at every angle, and 64-bit ones at every angle
ODD = {"narrow": NARROW["one"], "wide": WIDE["two"][0]}


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 3e38])
@pytest.mark.parametrize("case", list(ODD))
def test_voxels_that_are_not_finite_reach_their_samples(torch, case, value):
    """Such a voxel, or one whose sums overflow fixed point, makes the samples that it
    reaches not finite (or large) and changes no others."""
    g = scan(**ODD[case], tau=0.1)
    x = np.random.default_rng(9).standard_normal((g.Nz, g.Ny, g.Nx)).astype(f32)
    x[20, 25, 23] = x[33, 40, 12] = 0
    say(f"voxels that are not finite {case}, {value}")
    odd = np.zeros_like(x)
    odd[20, 25, 23] = odd[33, 40, 12] = 1
    ref, hit = splats(g, x), splats(g, odd)
    x[odd == 1] = value
    got = project(torch, g, x)
    assert np.count_nonzero(hit) >= 2 * 4 * g.Nang - 8
    # a weight of a few FP32 roundings of zero may be zero there
    reached = hit > 1e-5 * hit.max()
    if np.isfinite(value):
        assert O.rel_rmse(got[reached], (hit * value)[reached]) <= 5e-7
    else:
        assert not np.isfinite(got[reached]).any()
    assert O.rel_rmse(got[hit == 0], ref[hit == 0]) <= 1e-6
