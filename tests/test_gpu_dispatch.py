"""Kernels and dispatch rules at the sizes where they can go wrong, each
against the oracle or the general path."""
import ctypes as C
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
