"""Kernels and dispatch rules at the sizes where they can go wrong, each
against the oracle or the general path."""
import ctypes as C
import math
import threading

import numpy as np
import pytest

import oracle as O
from tomokvas_amd import _lib
from tomokvas_amd._hip import DeviceBuffer

from gpu_util import ogeom, say, scan, stages

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


# every shape of the filter's plan: more transforms than threads / 2 (p < 16),
# several transforms per wave, one to sixteen waves per transform, 512- and
# 1024-thread workgroups; odd projection counts, so a workgroup's last row and
# its rows' projections wrap
@pytest.mark.parametrize("Nu", [1, 3, 9, 37, 300, 700, 1024, 2048, 3000, 5000])
@pytest.mark.parametrize("Nang", [1, 7])
def test_filter_maxima_are_the_rows_maxima(torch, Nu, Nang):
    g = scan(Nu, 5, Nang, 8, 8, 8, D=max(2500.0, Nu))
    st = stages(g)
    gen = torch.Generator(device="cuda").manual_seed(Nu)
    d = torch.randn(st.sino_shape(), device="cuda", generator=gen)
    m = torch.zeros(Nang, dtype=torch.int32, device="cuda")
    st.filter(d, weight=True, maxabs=m)
    assert torch.equal(m.view(torch.float32), d.abs().amax(dim=(0, 2)))


def test_volume_range_from_many_threads():
    """More calls at once than the range has scratch slots."""
    L = _lib.load()
    n, errs = 100003, []
    bufs = []
    for k in range(12):
        v = np.random.default_rng(k).standard_normal(n).astype(np.float32)
        b = DeviceBuffer(v.nbytes)
        b.upload(v)
        bufs.append((v, b))

    def work(v, b):
        mm = (C.c_double * 2)()
        for _ in range(20):
            if L.fdk_volume_minmax(b.ptr, n, mm, None) or \
                    (mm[0], mm[1]) != (float(v.min()), float(v.max())):
                errs.append((mm[0], mm[1]))

    say("volume range from 12 threads")
    ts = [threading.Thread(target=work, args=a) for a in bufs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for _, b in bufs:
        b.close()
    assert not errs


# tiles and z-runs with remainders, boxes wider than 64 columns (two samples per
# voxel at 45 degrees), boxes beyond the LDS tile (four), one angle, more angles
# than a footprint group, columns that are zero or outside the cylinder
FP_CASES = {
    "one": dict(Nu=9, Nv=7, Nang=1, Nx=1, Ny=1, Nz=1, D=60.0),
    "edge32": dict(Nu=72, Nv=80, Nang=70, Nx=33, Ny=31, Nz=65, D=400.0),
    "two": dict(Nu=140, Nv=140, Nang=8, Nx=64, Ny=64, Nz=64, D=900.0, scale=2.0),
    "half": dict(Nu=48, Nv=40, Nang=9, Nx=70, Ny=40, Nz=67, D=300.0, scale=0.5),
    "four": dict(Nu=160, Nv=160, Nang=6, Nx=40, Ny=40, Nz=40, D=900.0, scale=4.0),
    # footprints of both boxes' memory at every angle or at some, with the others
    # in one box or in HBM
    "large": dict(Nu=170, Nv=190, Nang=9, Nx=64, Ny=64, Nz=70, D=420.0, scale=2.0),
    "larger": dict(Nu=180, Nv=240, Nang=9, Nx=64, Ny=60, Nz=64, D=260.0, scale=2.2),
    "mixed": dict(Nu=150, Nv=170, Nang=30, Nx=66, Ny=66, Nz=64, D=700.0, scale=1.9),
}


@pytest.mark.parametrize("case", list(FP_CASES))
@pytest.mark.parametrize("crop", [False, True])
def test_adjoint_tiles_and_splits(torch, case, crop):
    """The FP32 adjoint against the oracle's FP32 transcription: the sample
    positions are the same bits, so what differs is the rounding of the sums
    (bar of the FP32 path, 1e-5)."""
    g = scan(**FP_CASES[case], tau=0.1)
    st = stages(g)
    x = np.random.default_rng(5).standard_normal((g.Nz, g.Ny, g.Nx)).astype(np.float32)
    if crop:
        m = np.zeros_like(x)
        m[g.Nz // 3:g.Nz // 3 + 5, :2, :] = 1
        x = x * m
    say(f"adjoint {case}, crop {crop}")
    got = st.forward_project(torch.from_numpy(x).cuda()).cpu().numpy()
    ref = O.forward_project(ogeom(g), x)
    if not np.abs(ref).max():
        assert not np.abs(got).max()
        return
    assert O.rel_rmse(got, ref) <= 1e-5


def test_adjoint_at_tiny_and_huge_values(torch):
    """The box's fixed-point scale follows the tile's values."""
    g = scan(72, 60, 12, 48, 48, 40, D=400.0, tau=0.1)
    st = stages(g)
    x = np.random.default_rng(6).standard_normal((g.Nz, g.Ny, g.Nx)).astype(np.float32)
    one = st.forward_project(torch.from_numpy(x).cuda()).double().cpu().numpy()
    for s in (2.0 ** -90, 2.0 ** 90):
        y = st.forward_project(torch.from_numpy(x * np.float32(s)).cuda()).double().cpu().numpy()
        assert O.rel_rmse(y / s, one) <= 1e-6


# box heights from 16 rows to the limit and beyond it (gathered from HBM): small
# and large voxels, a source close to the object (U up to 2.5), a tall volume
# whose top and bottom runs leave the detector
BP_CASES = {
    "fine": dict(Nu=40, Nv=36, Nang=9, Nx=60, Ny=44, Nz=70, D=300.0, scale=0.4),
    "coarse": dict(Nu=90, Nv=100, Nang=9, Nx=40, Ny=37, Nz=40, D=500.0, scale=2.3),
    "near": dict(Nu=64, Nv=64, Nang=70, Nx=50, Ny=50, Nz=50, D=54.0, scale=1.1),
    "tall": dict(Nu=64, Nv=24, Nang=130, Nx=48, Ny=48, Nz=99, D=200.0, scale=1.25, cX=29.5),
    # blocks of 16^3 voxels either side of each change of shape (128, 256, 1024,
    # 8192), with fewer angles than groups, and with more than one batch of 64
    "one": dict(Nu=24, Nv=20, Nang=1, Nx=9, Ny=7, Nz=5, D=90.0, scale=1.5),
    "128": dict(Nu=130, Nv=60, Nang=66, Nx=128, Ny=127, Nz=30, D=400.0),
    "136": dict(Nu=130, Nv=60, Nang=3, Nx=129, Ny=70, Nz=42, D=400.0),
    "256": dict(Nu=200, Nv=40, Nang=70, Nx=250, Ny=256, Nz=16, D=500.0, scale=0.8),
    "272": dict(Nu=260, Nv=40, Nang=5, Nx=257, Ny=250, Nz=15, D=700.0),
    "1024": dict(Nu=260, Nv=20, Nang=67, Nx=511, Ny=512, Nz=15, D=900.0, scale=0.5),
    "1056": dict(Nu=260, Nv=20, Nang=4, Nx=513, Ny=505, Nz=14, D=900.0, scale=0.5),
    "8192": dict(Nu=1100, Nv=40, Nang=5, Nx=1024, Ny=1020, Nz=20, D=2000.0),
    "8320": dict(Nu=1100, Nv=40, Nang=5, Nx=1025, Ny=1010, Nz=20, D=2000.0),
    "8450, high boxes": dict(Nu=2140, Nv=60, Nang=4, Nx=1040, Ny=1030, Nz=20, D=7400.0, scale=2.05),
    "8450": dict(Nu=2300, Nv=70, Nang=3, Nx=1040, Ny=1040, Nz=17, D=3800.0, scale=2.2),
}


@pytest.mark.parametrize("case", list(BP_CASES))
@pytest.mark.parametrize("store", [_lib.F32, _lib.F16, _lib.BF16])
def test_backprojection_boxes(torch, case, store):
    """Against the FP32 mirror's backprojection of the decoded samples: positions
    and weights are the same bits, the sums are rounded in another order."""
    g = scan(**BP_CASES[case], tau=0.1)
    st = stages(g)
    gen = torch.Generator(device="cuda").manual_seed(3)
    d = torch.randn(st.sino_shape(), device="cuda", generator=gen)
    m = d.abs().amax(dim=(0, 2)).view(torch.int32)
    say(f"backprojection {case}, storage {store}")
    stack, scales = st.pack(d, store, m)
    got = st.backproject(stack, store, scales).cpu().numpy()
    # the stored samples [Nang][Nv][pitch], decoded
    dt = {_lib.F32: torch.float32, _lib.F16: torch.float16, _lib.BF16: torch.bfloat16}[store]
    per = st.stack_bytes(store, 1) - st.stack_bytes(store, 0)
    q = stack[:per * g.Nang].view(dt).view(g.Nang, g.Nv, -1)[:, :, :g.Nu].float()
    dec = (q * scales[:, None, None]).transpose(0, 1).contiguous()
    ref = O.backproject(ogeom(g), dec.cpu().numpy())
    assert O.rel_rmse(got, ref) <= 1e-6


# (sin_x, sin_y, n, axis): one column, one row, an odd sinogram left over, one to
# several waves side by side, rows that end inside a wave's
RSQ_SIZES = [(1, 1, 1, 0), (2, 3, 3, 0), (64, 37, 2, 0), (65, 361, 5, 1), (130, 100, 3, 2),
             (300, 203, 1, 40), (513, 90, 4, 0)]


@pytest.mark.parametrize("size", RSQ_SIZES)
@pytest.mark.parametrize("step", [1.0, 0.93, 1.21])
def test_rsq_full_fan(torch, size, step):
    """The one-pass rebinning against the reference's formula over whole rows, for
    angle steps of a full turn and others (whose pairs wrap around the scan), with
    columns without flat field and counts at and below dark."""
    from oracle import rsq as R
    from rsq_util import synthetic_raw

    sx, sy, n, axis = size
    raw = synthetic_raw(n, sy, sx, seed=sx)
    raw[:, 1, ::29] = raw[:, 0, ::29]                # flat = dark
    raw[:, 1, 7::31] = 50                            # flat < dark
    raw[:, 2::11, 3::13] = raw[:, :1, 3::13]         # count = dark
    raw[:, 5::17, 1::19] = 3                         # count < dark
    L = _lib.load()
    p = _lib.RsqParams()
    _lib.check(L.fdk_rsq_default_params(C.byref(p)), "rsq params")
    p.sin_x, p.sin_y, p.axis_move, p.complete, p.flip = sx, sy, axis, 1, sx % 2
    p.distance, p.delta_fi = 4.0 * sx, step * 2 * math.pi / sy
    w = 2 * sx - 1 - 2 * axis
    d_raw = torch.from_numpy(raw.view(np.int16)).cuda()
    got = {}
    for dt, store in ((torch.float64, _lib.F64), (torch.float32, _lib.F32)):
        out = torch.zeros((n, sy, w), device="cuda", dtype=dt)
        say(f"rsq {size} step {step} dtype {store}")
        _lib.check(L.fdk_rsq_process(C.byref(p), 1.1, 0.1, C.c_void_p(d_raw.data_ptr()), n, store,
                                     C.c_void_p(out.data_ptr()), None), "rsq")
        got[store] = out.cpu().numpy()
    f = np.arange(sy)[:, None]
    c0 = sx - 1 - axis
    t = np.arange(-c0, 0)
    base = f * p.delta_fi - 2 * np.arctan(t / p.distance)
    nf = (base - math.pi) / p.delta_fi
    nf = np.where((nf > sy - 1) | (nf < 0), (base + math.pi) / p.delta_fi, nf)
    ca, fl = np.ceil(nf), np.floor(nf)
    want = np.empty((n, sy, w))
    with np.errstate(invalid="ignore"):
        for k in range(n):
            ff = R.flat_field(raw[k], 1.1, 0.1, False)
            A, B = (ff[(v.astype(np.int64) % sy), axis - t] for v in (ca, fl))
            want[k, :, :c0] = np.where(ca != fl, A + (B - A) * (ca - nf), A)
            want[k, :, c0:] = ff[:, axis:]
    if p.flip:
        want = want[:, ::-1]
    fin = np.isfinite(want)
    assert np.array_equal(got[_lib.F64][~fin], want[~fin], equal_nan=True)
    err = np.abs(got[_lib.F64] - want)[fin]
    assert err.size == 0 or err.max() <= 1e-12 * max(np.abs(want[fin]).max(), 1.0)
    np.testing.assert_array_equal(got[_lib.F32], got[_lib.F64].astype(np.float32))


def test_prepare_again_equals_a_new_context(torch):
    """One context prepared for one geometry and filter after another -- larger
    tables, smaller ones, other taps -- filters and backprojects as a context
    prepared once does."""
    from tomokvas_amd import diff
    from tomokvas_amd.stages import Stages

    sizes = [dict(Nu=40, Nv=12, Nang=9, Nx=24, Ny=20, Nz=16, D=200.0),
             dict(Nu=140, Nv=30, Nang=37, Nx=50, Ny=48, Nz=90, D=500.0),
             dict(Nu=40, Nv=12, Nang=9, Nx=24, Ny=20, Nz=16, D=300.0)]
    one = None
    for i, kw in enumerate(sizes):
        g = scan(**kw)
        fresh = stages(g)
        if one is None:
            one = stages(g)
        else:
            fbp = one.fbp
            g.apply(fbp, None, None)
            _lib.check(fbp.SetFilter(_lib.FILTER_RAMLAK), "SetFilter")
            one = Stages(fbp)
        for taps in (None, np.random.default_rng(i).standard_normal(fresh.p)):
            say(f"prepare again {i} taps {taps is not None}")
            got = []
            for st in (fresh, one):
                if taps is not None:
                    diff.set_taps(st, taps)
                gen = torch.Generator(device="cuda").manual_seed(i)
                d = torch.randn(st.sino_shape(), device="cuda", generator=gen)
                st.filter(d, weight=True)
                stack, scales = st.pack(d, _lib.F32)
                got.append(st.backproject(stack, _lib.F32, scales).cpu())
            assert torch.equal(got[0], got[1])


# one row, rows that end inside a pair and a workgroup, several launches of the
# capped grid (2048 workgroups x 4 pairs of a transform); NT = 1 to 256
@pytest.mark.parametrize("Nu,Nv,Nang", [(1, 1, 1), (5, 3, 7), (64, 11, 29), (300, 70, 31),
                                        (1024, 40, 601), (1500, 130, 141)])
def test_weighted_tap_gradient(torch, Nu, Nv, Nang):
    """The cosine weight applied as the rows are loaded gives the products of the
    weighted rows."""
    g = scan(Nu, Nv, Nang, 8, 8, 8, D=max(900.0, 2.0 * Nu), cX=0.4 * Nu)
    st = stages(g)
    gen = torch.Generator(device="cuda").manual_seed(Nu)
    # (FP64 transforms of 4096 don't fit: refused)
    for dt in (torch.float32, torch.float64)[:2 if st.p <= 2048 else 1]:
        p, G = (torch.randn(st.sino_shape(), device="cuda", generator=gen, dtype=dt)
                for _ in range(2))
        say(f"weighted tap gradient {Nu}x{Nv}x{Nang} {dt}")
        got = st.tap_gradient(p, G, weight=True)
        want = st.tap_gradient(st.weight(p.clone()), G)
        # the same products in the same order: FMA contraction of the weight into
        # the first pass is all that may differ
        tol = 2e-6 if dt == torch.float32 else 1e-14
        assert np.abs(got - want).max() <= tol * max(np.abs(want).max(), 1e-30) * math.sqrt(Nu)
        if Nu <= 64:
            ref = O.tap_gradient(ogeom(g), st.weight(p.clone()).double().cpu().numpy(),
                                 G.double().cpu().numpy())
            assert np.abs(got - ref).max() <= (1e-5 if dt == torch.float32 else 1e-12) * np.abs(ref).max()


@pytest.mark.parametrize("Nu", [1, 3, 37, 300, 700, 1024, 2048, 3000])
@pytest.mark.parametrize("store", [_lib.F32, _lib.BF16, _lib.F64])
def test_filter_into_the_stored_stack(torch, Nu, store):
    """Slices of a stack filtered straight into a stored stack, into rows, and with
    the weight after the filter, against the filter, pack and weight in turn."""
    Nv, Nang, cut = 5, 7, 3
    g = scan(Nu, Nv, Nang, 8, 8, 8, D=max(2500.0, Nu))
    st = stages(g)
    dt = torch.float64 if store == _lib.F64 else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(Nu)
    d = torch.randn(st.sino_shape(), device="cuda", generator=gen, dtype=dt)
    say(f"filter into, Nu {Nu} storage {store}")
    # a slice's rows are transformed in pairs of its own, so the slices are filtered
    # one by one on both sides
    ya, yb = (st.filter(x.contiguous(), weight=True) for x in (d[:, :cut], d[:, cut:]))
    want, wscales = st.pack(d, store)
    st.pack_into(ya, store, want, wscales, 0)
    st.pack_into(yb, store, want, wscales, cut)
    got = torch.full_like(want, 0x55)
    scales = torch.zeros_like(wscales)
    st.filter_store(d, store, got, scales, 0, 0, cut)
    st.filter_store(d, store, got, scales, cut, cut)
    n = (st.stack_bytes(store, 1) - st.stack_bytes(store, 0)) * Nang
    assert torch.equal(got[:n], want[:n]) and torch.equal(scales, wscales)
    rows = torch.empty(st.sino_shape(Nang - cut), device="cuda", dtype=dt)
    m = torch.zeros(Nang - cut, dtype=torch.int32, device="cuda")
    st.filter_into(d, rows, weight=1, ang0=cut, maxabs=m)
    assert torch.equal(rows, yb)
    if dt == torch.float32:
        assert torch.equal(m.view(torch.float32), rows.abs().amax(dim=(0, 2)))
    z = st.weight(st.filter(d.clone(), adjoint=True))
    st.filter_into(d, d, weight=2, adjoint=True)
    assert torch.equal(d, z)
    with pytest.raises(ValueError):
        st.filter_into(d, rows, ang0=cut + 1)
    with pytest.raises(_lib.FDKError):
        st.filter_store(d, _lib.F16, got, scales)
