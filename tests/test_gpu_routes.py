"""Calls that can take more than one route through the library, on the device: each route's
results against the others' and the oracle's."""
import ctypes

import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def q():
    import qcu_cg_inverter_amd as q

    q.init(0)
    return q


def test_full_dslash_in_place_on_changed_links(q):
    """fullDslashQcu with output = input on a gauge that was changed in place is M of the
    new links applied once; without a change, and into another buffer, likewise."""
    L = (4, 6, 2, 10)
    vh = q.half_volume(L)
    prm = q.param(L)
    u = orc.gauge_random(L, 47, 0.3)
    v = orc.source_gauss(L, 14)
    gd = q.DeviceBuffer.from_numpy(u)
    out = q.DeviceBuffer(2 * vh * 192)
    for step in range(3):
        if step == 1:
            u[1, 0, 3] = orc.gauge_random(L, 48, 0.3)[1, 0, 3]
            gd.upload(u)
        A = orc.clover_fields(u, L, 1.0, 1.0, recon=12)[0]
        ref = orc.full_op(v, u, L, 1.0, A=A, s=1, tbc=1.0, recon=12)
        a = q.DeviceBuffer.from_numpy(v)
        q.lib().fullDslashQcu(a.ptr, a.ptr, gd.ptr, ctypes.byref(prm), 0)
        assert q.lib().qcuGetLastError() == 0
        got = a.to_numpy((2, vh, 4, 3))
        assert np.linalg.norm(got - ref) <= 1e-14 * np.linalg.norm(ref), step
        a.upload(v)
        q.lib().fullDslashQcu(out.ptr, a.ptr, gd.ptr, ctypes.byref(prm), 0)
        assert np.array_equal(out.to_numpy((2, vh, 4, 3)), got), step
