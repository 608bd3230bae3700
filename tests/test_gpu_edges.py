"""Calls at the edges of what the entry points accept, each against the oracle or the
general path."""
import numpy as np
import pytest

import oracle as O
from tomokvas_amd import _lib

from gpu_util import ogeom, say, scan, stages
from test_gpu_dispatch import BP_CASES

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


def decoded(torch, st, g, stack, scales, store):
    """The stored samples as float [Nv][Nang][Nu] on the host."""
    dt = {_lib.F32: torch.float32, _lib.F16: torch.float16, _lib.F16_PACKED: torch.float16,
          _lib.BF16: torch.bfloat16}[store]
    per = st.stack_bytes(store, 1) - st.stack_bytes(store, 0)
    q = stack[:per * g.Nang].view(dt).view(g.Nang, g.Nv, -1)[:, :, :g.Nu].float()
    return (q * scales[:, None, None]).transpose(0, 1).contiguous().cpu().numpy()


# the reciprocal of D - S leaves the normal numbers beyond 2^126
@pytest.mark.parametrize("D", [1e30, 8.6e37, 3.4e38])
@pytest.mark.parametrize("store", [_lib.F32, _lib.F16, _lib.BF16, _lib.F16_PACKED])
def test_backprojection_of_a_parallel_beam(torch, D, store):
    """A source so far away that U = 1 for every voxel."""
    g = scan(60, 40, 9, 40, 37, 33, D=D, tau=0.1)
    st = stages(g)
    gen = torch.Generator(device="cuda").manual_seed(4)
    d = torch.randn(st.sino_shape(), device="cuda", generator=gen)
    say(f"parallel beam D {D:g}, storage {store}")
    stack, scales = st.pack(d, store, d.abs().amax(dim=(0, 2)).view(torch.int32))
    got = st.backproject(stack, store, scales).cpu().numpy()
    ref = O.backproject(ogeom(g), decoded(torch, st, g, stack, scales, store))
    assert np.abs(ref).max() > 0
    # FP32 sums in another order; packed FP16 also rounds weights and lerps to FP16
    assert O.rel_rmse(got, ref) <= (1e-3 if store == _lib.F16_PACKED else 1e-6)


def test_stored_stacks_that_do_not_fit_are_refused(torch):
    """A stack or scales that are strided, on the host, too small or of another type."""
    g = scan(40, 12, 9, 16, 16, 16, D=200.0, tau=0.1)
    st = stages(g)
    d = torch.randn(st.sino_shape(), device="cuda")
    for store in (_lib.F32, _lib.BF16):
        stack, scales = st.pack(d, store)
        n = stack.numel()
        bad = [(stack.cpu(), scales), (stack, scales.cpu()), (stack[:n - 1], scales),
               (torch.zeros(2 * n, dtype=torch.uint8, device="cuda")[::2], scales),
               (stack, scales[:-1]), (stack, scales.double()), (stack, scales.half()),
               (stack, torch.zeros(2 * g.Nang, device="cuda")[::2])]
        for a, b in bad:
            with pytest.raises(ValueError):
                st.filter_store(d, store, a, b)
            with pytest.raises(ValueError):
                st.pack_into(d, store, a, b, 0)
        st.filter_store(d, store, stack, scales)
        st.pack_into(d, store, stack, scales, 0)
        torch.cuda.synchronize()


@pytest.mark.parametrize("chunk", [None, 4])
@pytest.mark.parametrize("store", [_lib.F32, _lib.F16, _lib.F64])
def test_projections_that_are_not_contiguous(torch, store, chunk):
    """An angle-major stack, passed as a transposed view, gives what its copy gives."""
    from tomokvas_amd import diff

    g = scan(40, 12, 9, 24, 20, 16, D=200.0, tau=0.1)
    st = stages(g)
    dt = torch.float64 if store == _lib.F64 else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(6)
    p = torch.randn((g.Nang, g.Nv, g.Nu), device="cuda", generator=gen, dtype=dt).transpose(0, 1)
    gvol = torch.randn(st.vol_shape, device="cuda", generator=gen, dtype=dt)
    assert not p.is_contiguous() and tuple(p.shape) == st.sino_shape()
    say(f"not contiguous, storage {store}, chunk {chunk}")
    keep = p.clone()
    got = diff.forward(st, p, storage=store, chunk=chunk)
    assert torch.equal(got, diff.forward(st, p.contiguous(), storage=store, chunk=chunk))
    gp, dh = diff.backward(st, p, gvol, chunk=chunk)
    wp, wh = diff.backward(st, p.contiguous(), gvol, chunk=chunk)
    assert torch.equal(p, keep)
    # the splats are atomics, and a slice's rows are transformed in pairs of its own
    tol = 1e-12 if dt == torch.float64 else 1e-5
    assert O.rel_rmse(gp.cpu().numpy(), wp.cpu().numpy()) <= tol
    assert O.rel_rmse(dh, wh) <= tol


@pytest.mark.parametrize("contiguous", [True, False])
def test_tap_gradient_of_the_first_angles(torch, contiguous):
    """Projections of the first angles only, in chunks, with a volume gradient of the
    whole scan: dL/dh takes those angles' rows of the adjoint."""
    from tomokvas_amd import diff

    g = scan(40, 12, 9, 24, 20, 16, D=200.0, tau=0.1)
    st = stages(g)
    n = 7
    gen = torch.Generator(device="cuda").manual_seed(6)
    p = torch.randn(st.sino_shape(n), device="cuda", generator=gen, dtype=torch.float64)
    if not contiguous:
        p = p.transpose(0, 1).contiguous().transpose(0, 1)
    gvol = torch.randn(st.vol_shape, device="cuda", generator=gen, dtype=torch.float64)
    say("tap gradient of the first angles")
    _, dh = diff.backward(st, p, gvol, chunk=3, need_proj=False)
    q = st.weight(p.contiguous().clone())
    G = st.forward_project(gvol)[:, :n].contiguous()
    ref = O.tap_gradient(ogeom(scan(40, 12, n, 24, 20, 16, D=200.0, tau=0.1)),
                         q.cpu().numpy(), G.cpu().numpy())
    assert O.rel_rmse(dh, ref) <= 1e-12
    with pytest.raises(ValueError):
        diff.backward(st, p, gvol, need_proj=False)


# zeros of both signs in one thread, in two lanes, waves and workgroups
@pytest.mark.parametrize("at", [1, 4, 300, 2000, 5000, 40000, 99999])
@pytest.mark.parametrize("first", [0.0, -0.0])
def test_volume_range_keeps_the_sign_of_zero(torch, first, at):
    """-0 is below +0, wherever either lies."""
    import ctypes as C
    L = _lib.load()
    n = 100000
    v = torch.full((n,), first, device="cuda")
    v[at] = -first
    mm = (C.c_double * 2)()
    say(f"range of zeros, {-first} at {at}")
    _lib.check(L.fdk_volume_minmax(C.c_void_p(v.data_ptr()), n, mm, None), "minmax")
    assert (mm[0], mm[1]) == (0.0, 0.0)
    assert np.signbit(mm[0]) and not np.signbit(mm[1])


@pytest.mark.parametrize("chunk", [None, 3])
@pytest.mark.parametrize("store", [_lib.F32, _lib.F16])
def test_forward_of_the_first_angles(torch, store, chunk):
    """Projections of the first angles only give those angles' share of the volume."""
    from tomokvas_amd import diff

    g = scan(40, 12, 9, 24, 20, 16, D=200.0, tau=0.1)
    st = stages(g)
    n = 7
    gen = torch.Generator(device="cuda").manual_seed(6)
    p = torch.randn(st.sino_shape(n), device="cuda", generator=gen)
    say(f"forward of the first angles, storage {store}, chunk {chunk}")
    got = diff.forward(st, p, storage=store, chunk=chunk)
    q = torch.zeros(st.sino_shape(), device="cuda")
    q[:, :n] = p
    want = diff.forward(st, q, storage=store, chunk=chunk)
    # the rows are transformed in other pairs
    assert O.rel_rmse(got.cpu().numpy(), want.cpu().numpy()) <= (1e-3 if store == _lib.F16 else 1e-5)


@pytest.mark.parametrize("case", list(BP_CASES))
def test_packed_backprojection_boxes(torch, case):
    """Packed FP16 in every shape and box, against the FP32 mirror on the decoded
    samples.  Fraction, weights, difference and lerp each round to FP16 (2^-11 at most,
    a third of it in the mean): about 3.5e-4 of a sample together, half as much again
    measured (weights and fractions are common to many samples)."""
    g = scan(**BP_CASES[case], tau=0.1)
    st = stages(g)
    gen = torch.Generator(device="cuda").manual_seed(3)
    d = torch.randn(st.sino_shape(), device="cuda", generator=gen)
    say(f"packed backprojection {case}")
    stack, scales = st.pack(d, _lib.F16_PACKED, d.abs().amax(dim=(0, 2)).view(torch.int32))
    got = st.backproject(stack, _lib.F16_PACKED, scales).cpu().numpy()
    ref = O.backproject(ogeom(g), decoded(torch, st, g, stack, scales, _lib.F16_PACKED))
    err = O.rel_rmse(got, ref)
    say(f"  {err:.2e}")
    assert err <= 1e-3
