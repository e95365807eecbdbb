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
        q.lib().qcuClearLastError()
        q.lib().fullDslashQcu(a.ptr, a.ptr, gd.ptr, ctypes.byref(prm), 0)
        assert q.lib().qcuGetLastError() == 0
        got = a.to_numpy((2, vh, 4, 3))
        assert np.linalg.norm(got - ref) <= 1e-14 * np.linalg.norm(ref), step
        a.upload(v)
        q.lib().fullDslashQcu(out.ptr, a.ptr, gd.ptr, ctypes.byref(prm), 0)
        assert np.array_equal(out.to_numpy((2, vh, 4, 3)), got), step


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_hop_shapes_keep_bits_on_internal_fields(q, prec):
    """Every launch shape of a 12-RHS hop gives the bits of single launches from and to the
    caller's buffers.  A batch whose outputs are its inputs goes through internal fields,
    where the pinned shape is the one that runs."""
    L = (16, 16, 16, 16)  # 128-site planes: whole-plane and 8-row (y, z, t) walk tiles apply
    g = q.Gauge.random(L, seed=34, eps=0.3)
    vh = q.half_volume(L)
    vs = [orc.source_gauss(L, 80 + r)[1] for r in range(12)]
    singles = [q.hop(g, v, 0, dagger=0, t_boundary=-1, recon=12, precision=prec) for v in vs]
    bufs = [q.DeviceBuffer(vh * 192) for _ in vs]
    ptrs = (ctypes.c_void_p * 12)(*[b.ptr for b in bufs])
    # (block, rb, rpt, xcd, tile_z, tile_t, group_major, tile_y, rpw, spt, cached, lds)
    shapes = [None,  # the default
              (256, 4, 1, 1, 4, 4, 1, 0, 1, 1, 0, 0), (128, 2, 3, 1, 4, 4, 1, 8, 1, 2, 1, 0),
              (64, 1, 2, 0, 0, 0, 1, 0, 1, 1, 0, 0), (256, 2, 1, 1, 8, 8, 0, 8, 1, 4, 1, 0),
              (128, 1, 4, 0, 4, 4, 0, 0, 1, 1, 0, 0), (192, 3, 1, 1, 4, 4, 0, 0, 4, 1, 1, 0),
              (64, 1, 1, 1, 0, 0, 1, 0, 4, 2, 0, 0), (128, 2, 1, 0, 4, 4, 1, 8, 2, 4, 1, 0),
              (256, 2, 1, 1, 8, 8, 1, 0, 2, 2, 1, 0), (256, 1, 1, 1, 4, 4, 0, 8, 1, 1, 0, 1),
              (128, 1, 1, 0, 0, 0, 0, 0, 1, 2, 1, 1), (64, 1, 1, 1, 8, 8, 0, 0, 1, 3, 0, 1),
              (256, 1, 1, 0, 2, 4, 0, 8, 1, 1, 1, 1), (256, 1, 1, 2, 8, 16, 0, 0, 1, 1, 1, 1),
              (128, 1, 1, 2, 0, 0, 0, 0, 1, 1, 0, 1), (256, 1, 1, 4, 8, 8, 0, 0, 1, 1, 1, 2)]
    for sh in shapes:
        if sh:
            shape = dict(zip(q.SHAPE_KEYS, sh))
            if prec == 0:
                shape["rpt"] = 1
            q.set_hop_shape(g, prec, 12, 12, shape)
        for b, v in zip(bufs, vs):
            b.upload(v)
        q.check(q.lib().qcuHopBatch(g.handle, 12, ptrs, ptrs, 0, 0, -1, 12, prec))
        for r in range(12):
            assert np.array_equal(bufs[r].to_numpy((vh, 4, 3)), singles[r]), (sh, r)


# half volumes that no other test pins a shape for: off the 64-site chunk and of whole chunks
@pytest.mark.parametrize("L", [(10, 2, 2, 6), (6, 6, 6, 10), (12, 8, 6, 14), (8, 8, 6, 10)])
def test_split_kernel_bits_equal_pinned_shape_every_epilogue(q, L):
    """The leg-split kernel (the default here) against hop_kernel under a pinned shape, on
    internal fields: Mhat, Wilson and clover, in each precision and link storage, and a
    solve's iterations, solution and true residual.  A pin holds for the process, so every
    default result comes before the first of them."""
    b = orc.source_gauss(L, 5)
    cases = [(p, r, csw) for p in (0, 1, 2) for r in (12, 18) for csw in (0.0, 1.0)]

    def results():
        out = {}
        for prec, recon, csw in cases:
            g = q.Gauge.random(L, seed=43, eps=0.2)
            op = q.Operator(0.12, csw, -1, recon)
            sp = q.default_solve_params(tol=1e-9, precision=prec, chunk=4, max_iter=200)
            x, st = q.solve(g, op, b, sp, raise_on_error=False)
            assert st.true_residual <= 1e-9
            out[prec, recon, csw] = [q.apply_mhat(g, op, b[0], dagger=d, precision=prec) for d in (0, 1)] + [
                x, np.array([st.iterations, st.true_residual])]
            g.destroy()
        return out

    want = results()
    g = q.Gauge.random(L, seed=43, eps=0.2)
    for prec in (0, 1, 2):
        for recon in (12, 18):
            q.set_hop_shape(g, prec, recon, 1, {"block": 128, "rb": 1, "rpt": 1})
    got = results()
    for k in cases:
        for i, (a, c) in enumerate(zip(want[k], got[k])):
            assert np.array_equal(a, c), (k, i)


def test_scalar_steps_hand_over_mid_solve(q):
    """Eight right-hand sides of 16^3x64, checked after every iteration: with 2,048 partials
    seven and more take their scalar steps in one-block kernels, six and fewer in the vector
    kernels.  Source r is M^r of a Gaussian one, its low modes the weaker the higher r, so
    the sources converge apart and the solve goes from one to the other.  Each right-hand
    side keeps the bits and iterations of its solve alone."""
    L = (16, 16, 16, 64)
    chains = q.lib()["_ZN3qcu14cg_step_chainsEli"]
    chains.argtypes, chains.restype = [ctypes.c_long, ctypes.c_int], ctypes.c_int
    nw = q.half_volume(L) // 64
    g = q.Gauge.random(L, seed=45, eps=0.2)
    op = q.Operator(0.115, 0.0, -1, 12)
    sp = q.default_solve_params(tol=1e-8, precision=1, chunk=1)
    bs = [q.source_gaussian_device(L, 60)]
    for r in range(7):
        bs.append(q.DeviceBuffer(bs[0].nbytes))
        q.check(q.lib().qcuApplyM(g.handle, ctypes.byref(op), bs[-1].ptr, bs[-2].ptr, 0))
    vh = q.half_volume(L)
    xs = [q.DeviceBuffer(2 * vh * 192) for _ in bs]
    sts = q.solve_batch_device(g, op, xs, bs, sp)
    its = [s.iterations for s in sts]
    assert all(s.converged for s in sts)
    left = {sum(i > t for i in its) for t in its} - {0}  # right-hand sides still active after a harvest
    assert chains(nw, 8) == 0 and any(chains(nw, n) != 0 for n in left), (its, left)
    xa = q.DeviceBuffer(2 * vh * 192)
    for r in range(8):
        sa = q.solve_batch_device(g, op, [xa], [bs[r]], sp)[0]
        assert sa.converged and sa.iterations == its[r], (r, its)
        assert np.array_equal(xa.to_numpy((2, vh, 4, 3)), xs[r].to_numpy((2, vh, 4, 3))), r


@pytest.mark.parametrize("L", [(24, 24, 24, 36), (22, 22, 26, 38)])
def test_dslash_past_the_cache(q, L):
    """dslashQcu on data well beyond the 256 MB Infinity Cache takes its chunks in storage
    order; half volumes on and off the 64-site chunk, the bits of the hop on packed links."""
    g = q.Gauge.random(L, seed=49, eps=0.25)
    vh = q.half_volume(L)
    assert vh * (8 * 144 + 2 * 192) > 340 << 20
    prm = q.param(L)
    gd, a = q.DeviceBuffer(8 * vh * 144), q.source_gaussian_device(L, 15)
    q.check(q.lib().qcuGaugeExport(g.handle, gd.ptr))
    b, c = q.DeviceBuffer(vh * 192), q.DeviceBuffer(vh * 192)
    q.lib().qcuClearLastError()
    for parity in (0, 1):
        src = a.ptr + (1 - parity) * vh * 192
        q.lib().dslashQcu(b.ptr, src, gd.ptr, ctypes.byref(prm), parity)
        assert q.lib().qcuGetLastError() == 0
        q.check(q.lib().qcuHop(g.handle, c.ptr, src, parity, 0, 1, 12, 0))
        assert np.array_equal(b.to_numpy((vh, 4, 3)), c.to_numpy((vh, 4, 3))), parity


@pytest.mark.parametrize("L,field,n", [((24, 24, 24, 32), 0, 12), ((16, 16, 16, 32), 1, 36), ((24, 24, 24, 64), 0, 12)])
def test_layout_round_trip_at_each_cache_policy(q, L, field, n):
    """A spinor of 85 MB, whose lexicographic output alone is streamed, and a gauge of 75 MB and
    a spinor of 170 MB, streamed on both sides: there and back gives the same words, and the even-odd field is the
    one numpy makes."""
    vol = 2 * q.half_volume(L)
    a, b, c = (q.DeviceBuffer(vol * n * 16) for _ in range(3))
    src = np.random.default_rng(7).standard_normal((n // (12 if field == 0 else 9), vol, 12 if field == 0 else 9, 2))
    a.upload(src)
    I = (ctypes.c_int * 4)(*L)
    q.check(q.lib().qcuLexToEvenOdd(b.ptr, a.ptr, I, field))
    q.check(q.lib().qcuEvenOddToLex(c.ptr, b.ptr, I, field))
    assert np.array_equal(c.to_numpy((vol * n * 2,), np.float64), src.ravel())
    t, z, y, x = np.indices(L[::-1]).reshape(4, -1)
    par = (t + z + y + x) & 1
    eo = b.to_numpy(src.shape, np.float64)
    for p in (0, 1):
        assert np.array_equal(eo[:, p * vol // 2:(p + 1) * vol // 2], src[:, par == p]), p
